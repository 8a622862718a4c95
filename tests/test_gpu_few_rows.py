"""GPU parity of the exact product for a few rows (few_rows.hip), through
holo_matmul_batch and its forms.

Truth and elementwise bar are those of test_gpu_batch_exact: the float64
product of the fp32 activations and the bit-exact dequantised weights, within
(K/32 + 70) 2^-24 sum_k |x w| (doubled for Q4_K).  The waves' eight partial
sums, up to 32 over four parts of K, replace as many roundings of the
block-order sum, so the bar holds unchanged.
"""
import ctypes as C

import numpy as np
import pytest

from test_gpu_batch_exact import F16, NAMES, Q4_0, Q4_K, Q6_K, Q8_0, check_rows, down, up, weights

pytestmark = pytest.mark.gpu

# rows at the edges of 16- and 64-row tiles; columns at the edges of 16- and
# 32-column tiles; K of one block, odd block counts (windows straight from
# memory), one unit of 256, more units than waves, and K split over several
# workgroups (every tile that can run: test_gpu_few_rows_plans)
CASES = [(Q4_0, 3, 1, 32), (Q4_0, 16, 15, 256), (Q4_0, 17, 16, 288), (Q4_0, 33, 301, 1056), (Q4_0, 64, 4096, 4096),
         (Q4_0, 20, 1000, 11008), (Q4_0, 130, 100, 2304), (Q4_0, 192, 333, 1024), (Q8_0, 3, 17, 32),
         (Q8_0, 15, 49, 2080), (Q8_0, 32, 130, 4096), (Q8_0, 63, 64, 544), (Q8_0, 50, 700, 8192), (Q4_K, 4, 3, 256),
         (Q4_K, 16, 1024, 4096), (Q4_K, 31, 65, 2304), (Q4_K, 65, 500, 14336), (Q6_K, 3, 33, 256),
         (Q6_K, 16, 47, 768), (Q6_K, 23, 1001, 4096), (Q6_K, 64, 200, 11008), (Q6_K, 100, 129, 2304), (F16, 5, 31, 96),
         (F16, 16, 129, 4096), (F16, 48, 77, 1056)]


@pytest.mark.parametrize("t,M,N,K", CASES, ids=[f"{NAMES[t]}-{m}x{n}x{k}" for t, m, n, k in CASES])
def test_few_rows(holo, synth, oracle, t, M, N, K):
    """The product, the add in its store and the SwiGLU in its split: within
    the bound, the fused forms bit-identical to the unfused sequence, two
    calls bit-identical, nothing written past the output."""
    print(f"case few rows {NAMES[t]} {M}x{N}x{K}", flush=True)
    lib = holo.lib()
    src, w = weights(synth, oracle, t, N, K, seed=M + 3 * N + K)
    X = synth.normal(M * K, seed=K + 5).reshape(M, K)
    U = synth.normal(M * K, seed=K + 6).reshape(M, K)
    R = synth.normal(M * N, seed=K + 7).reshape(M, N)
    X[0] *= 1e5  # rows of very different size share a tile
    X[-1] *= 1e-6
    dW, dX, dU, dR = up(holo, src), up(holo, X), up(holo, U), up(holo, R)
    outs = []
    for _ in range(2):
        dY = up(holo, np.full(M * N + 64, 7.0, np.float32))
        lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
        lib.cuda_sync()
        holo.check("few rows")
        outs.append(down(dY, M * N + 64))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert np.all(outs[0][M * N:] == 7.0)
    y = outs[0][:M * N].reshape(M, N)
    for r in (np.arange(1), np.arange(1, M - 1), np.arange(M - 1, M)):  # each scale by itself
        if len(r):
            check_rows(y, X, w, r, t, K)
    dS, dZ, dG, dH, dT = up(holo, R), up(holo, R), up(holo, X), holo.DeviceBuffer(4 * M * K), holo.DeviceBuffer(4 * M * N)
    lib.holo_matmul_batch_add(dS.ptr, dW.ptr, dX.ptr, dS.ptr, M, N, K, t)
    lib.cuda_silu_mul(dH.ptr, dG.ptr, dU.ptr, M * K)
    lib.holo_matmul_batch(dT.ptr, dW.ptr, dH.ptr, M, N, K, t)
    lib.holo_matmul_batch_swiglu_add(dZ.ptr, dW.ptr, dG.ptr, dU.ptr, dR.ptr, M, N, K, t)
    lib.cuda_sync()
    holo.check("few rows add")
    assert np.array_equal(down(dS, M * N).reshape(M, N), R + y)
    assert np.array_equal(down(dZ, M * N).reshape(M, N), R + down(dT, M * N).reshape(M, N))


def test_few_rows_multi(holo, synth, oracle):
    """q, k, v of mixed types and gate, up of one: each output within the bound."""
    lib = holo.lib()
    M, K = 23, 2304
    for types, Ns in (((Q4_K, Q4_K, Q6_K), (256, 128, 128)), ((Q4_0, Q4_0), (384, 384))):
        srcs, ws = zip(*[weights(synth, oracle, t, n, K, seed=90 + i) for i, (t, n) in enumerate(zip(types, Ns))])
        X = synth.normal(M * K, seed=91).reshape(M, K)
        dWs, dX, dYs = [up(holo, s) for s in srcs], up(holo, X), [holo.DeviceBuffer(4 * M * n) for n in Ns]
        k = len(Ns)
        lib.holo_matmul_batch_multi_types((C.c_void_p * k)(*[d.ptr for d in dYs]),
                                          (C.c_void_p * k)(*[d.ptr for d in dWs]), (C.c_int * k)(*types),
                                          (C.c_int * k)(*Ns), k, dX.ptr, M, K)
        lib.cuda_sync()
        holo.check("few rows multi")
        for i, n in enumerate(Ns):
            check_rows(down(dYs[i], M * n).reshape(M, n), X, ws[i], np.arange(M), types[i], K)


@pytest.mark.parametrize("M,N,K", [(16, 512, 2048), (40, 2000, 11008)], ids=["whole", "parts"])
def test_few_rows_streams_and_graph(holo, synth, oracle, M, N, K):
    """Calls issued on two streams at once, and a captured graph replayed
    between eager calls: the bits of the call on its own."""
    lib = holo.lib()
    src, _ = weights(synth, oracle, Q4_0, N, K, seed=N)
    Xs = [synth.normal(M * K, seed=s).reshape(M, K) for s in (1, 2)]
    dW, dXs = up(holo, src), [up(holo, x) for x in Xs]

    def call(x):
        d = holo.DeviceBuffer(4 * M * N)
        lib.holo_matmul_batch(d.ptr, dW.ptr, x.ptr, M, N, K, Q4_0)
        return d

    want = [call(x) for x in dXs]
    lib.cuda_sync()
    want = [down(d, M * N).view(np.uint32) for d in want]
    streams = [lib.holo_stream_create() for _ in range(2)]
    try:
        got = []
        for _ in range(6):
            for s, x in zip(streams, dXs):
                lib.holo_set_stream(s)
                got.append(call(x))
        lib.cuda_sync()
        for i, d in enumerate(got):
            assert np.array_equal(down(d, M * N).view(np.uint32), want[i % 2]), i
        dG = holo.DeviceBuffer(4 * M * N)
        lib.holo_set_stream(streams[0])
        assert lib.holo_graph_begin() == 0
        lib.holo_matmul_batch(dG.ptr, dW.ptr, dXs[0].ptr, M, N, K, Q4_0)
        g = lib.holo_graph_end()
        holo.check("capture")
        for rep in range(3):
            lib.holo_graph_launch(g)
            other = call(dXs[1])
            lib.cuda_sync()
            assert np.array_equal(down(dG, M * N).view(np.uint32), want[0]), rep
            assert np.array_equal(down(other, M * N).view(np.uint32), want[1]), rep
        lib.holo_graph_destroy(g)
    finally:
        lib.holo_set_stream(None)
        for s in streams:
            lib.holo_stream_destroy(s)
    holo.check("streams")


def test_few_rows_keeps_gemv_cases(holo, synth, oracle):
    """Rows that the product does not take still run one GEMV each: no matrix
    (zeros), another activation mode, activations off 16-byte alignment."""
    lib = holo.lib()
    M, N, K = 5, 70, 512
    src, _ = weights(synth, oracle, Q4_0, N, K, seed=4)
    X = synth.normal(M * K + 1, seed=5)
    dW, dX, dY = up(holo, src), up(holo, X), up(holo, np.ones(M * N, np.float32))
    lib.holo_matmul_rows(dY.ptr, None, dX.ptr, M, N, K, Q4_0, 0)
    lib.cuda_sync()
    holo.check("no matrix")
    assert np.all(down(dY, M * N) == 0)
    ref = np.stack([oracle.matmul(Q4_0, src, X[1 + m * K:1 + (m + 1) * K], N, K) for m in range(M)])
    lib.holo_matmul_rows(dY.ptr, dW.ptr, dX.ptr + 4, M, N, K, Q4_0, 0)
    lib.cuda_sync()
    holo.check("misaligned rows")
    assert np.max(np.abs(down(dY, M * N).reshape(M, N) - ref)) <= 1e-3 * np.max(np.abs(ref))
    single = holo.DeviceBuffer(4 * N)
    lib.holo_gemv_set_xmode(0)
    try:
        lib.holo_matmul_rows(dY.ptr, dW.ptr, dX.ptr, M, N, K, Q4_0, 0)
        lib.holo_matmul(single.ptr, dW.ptr, dX.ptr + 4 * K, N, K, Q4_0)
        lib.cuda_sync()
    finally:
        lib.holo_gemv_set_xmode(2)
    holo.check("fp32 mode")
    assert np.array_equal(down(dY, M * N).reshape(M, N)[1], down(single, N))


def test_few_rows_infinities(holo, synth, oracle):
    """A row with an infinity gives infinities and NaNs, as fp32 does; the
    other rows keep their bits."""
    lib = holo.lib()
    M, N, K = 7, 40, 512
    src, w = weights(synth, oracle, Q8_0, N, K, seed=14)
    X = synth.normal(M * K, seed=15).reshape(M, K)
    dW, outs = up(holo, src), []
    for k in range(2):
        if k:
            X[3, 100] = np.inf
        dX, dY = up(holo, X), holo.DeviceBuffer(4 * M * N)
        lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, Q8_0)
        lib.cuda_sync()
        outs.append(down(dY, M * N).reshape(M, N))
    holo.check("infinities")
    rest = np.r_[0:3, 4:7]
    assert np.array_equal(outs[0][rest], outs[1][rest])
    want = np.where(w[:, 100] > 0, np.inf, np.where(w[:, 100] < 0, -np.inf, np.nan))
    assert np.array_equal(outs[1][3], want, equal_nan=True)


@pytest.mark.parametrize("t,M,N,K", [(Q4_0, 5, 40, 288), (Q4_0, 20, 100, 4096), (Q8_0, 3, 33, 32), (Q8_0, 63, 50, 1056),
                                     (Q4_K, 7, 70, 256), (Q4_K, 40, 4096, 2304), (Q6_K, 16, 47, 768), (Q6_K, 33, 129, 4096),
                                     (F16, 5, 31, 288), (F16, 40, 2000, 2080), (F16, 16, 129, 11008)],
                         ids=lambda v: NAMES[v] if v in NAMES and v != 16 and v != 32 else str(v))
def test_few_rows_rows_with_infinities(holo, synth, oracle, t, M, N, K):
    """Rows with infinities anywhere (the last block of a K that is no multiple
    of 256 among the places), beside finite values past f16's range, give the
    infinities and NaNs of the dequantised weights' products; the other rows
    keep their bits, and the add in the store and the SwiGLU in the split give
    what the unfused sequence gives."""
    print(f"case infinities {NAMES[t]} {M}x{N}x{K}", flush=True)
    lib = holo.lib()
    src, w = weights(synth, oracle, t, N, K, seed=M + N + K)
    X = synth.normal(M * K, seed=K + 15).reshape(M, K)
    U = synth.normal(M * K, seed=K + 16).reshape(M, K)
    R = synth.normal(M * N, seed=K + 17).reshape(M, N)
    dW, dU, dR = up(holo, src), up(holo, U), up(holo, R)
    dX, dY = up(holo, X), holo.DeviceBuffer(4 * M * N)
    lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
    lib.cuda_sync()
    y0 = down(dY, M * N).reshape(M, N)
    X[0, K - 1] = np.inf
    X[0, K // 2] = 7e4
    X[M // 2, K - 20] = -np.inf
    X[M - 1, 3], X[M - 1, K - 2] = np.inf, -np.inf
    X[M - 1, K // 2] = 1e36  # its products with weights up to 1e2 stay in fp32 range
    bad = sorted({0, M // 2, M - 1})
    dX, dS, dZ, dT, dH = up(holo, X), up(holo, R), *(holo.DeviceBuffer(4 * n) for n in (M * N, M * N, M * K))
    lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
    lib.holo_matmul_batch_add(dS.ptr, dW.ptr, dX.ptr, dS.ptr, M, N, K, t)
    lib.cuda_silu_mul(dH.ptr, dX.ptr, dU.ptr, M * K)
    lib.holo_matmul_batch(dT.ptr, dW.ptr, dH.ptr, M, N, K, t)
    lib.holo_matmul_batch_swiglu_add(dZ.ptr, dW.ptr, dX.ptr, dU.ptr, dR.ptr, M, N, K, t)
    lib.cuda_sync()
    holo.check("rows with infinities")
    y = down(dY, M * N).reshape(M, N)
    rest = np.setdiff1d(np.arange(M), bad)
    assert np.array_equal(y[rest].view(np.uint32), y0[rest].view(np.uint32))
    with np.errstate(invalid="ignore"):
        for r in bad:
            want = (X[r].astype(np.float64) * w).sum(1)  # infinite or NaN each
            assert np.array_equal(y[r], want.astype(np.float32), equal_nan=True), r
        assert np.array_equal(down(dS, M * N).reshape(M, N), R + y, equal_nan=True)
        assert np.array_equal(down(dZ, M * N).reshape(M, N), R + down(dT, M * N).reshape(M, N), equal_nan=True)


def without_first_unit(src, w, t, N, K):
    """The matrix with its first 256 weights of every row (32 for the types of
    32-weight blocks) zero: their scales and minima cleared."""
    raw, w, n = np.array(src).view(np.uint8).reshape(N, -1).copy(), w.copy(), 256 if t in (Q4_K, Q6_K) else 32
    for at, size in {Q4_0: [(0, 2)], Q8_0: [(0, 2)], Q4_K: [(0, 4)], Q6_K: [(208, 2)], F16: [(0, 64)]}[t]:
        raw[:, at:at + size] = 0
    w[:, :n] = 0
    return raw.reshape(-1), w


@pytest.mark.parametrize("big", [3e7, 1e12, 1e30])
@pytest.mark.parametrize("t,M,N,K", [(Q4_0, 3, 40, 1056), (Q4_0, 20, 1000, 11008), (Q8_0, 17, 65, 4096), (Q4_K, 40, 100, 2304),
                                     (Q6_K, 23, 129, 4096), (Q6_K, 63, 50, 16384), (F16, 16, 77, 1056)],
                         ids=lambda v: str(v))
def test_few_rows_range(holo, synth, oracle, t, M, N, K, big):
    """Rows whose largest value lies far above their other blocks, and meets
    zero weights: the other blocks keep the bits that a GEMV, which scales
    them by themselves, gives them."""
    print(f"case range {NAMES[t]} {M}x{N}x{K} {big}", flush=True)
    lib = holo.lib()
    src, w = without_first_unit(*weights(synth, oracle, t, N, K, seed=N + K), t, N, K)
    X = synth.normal(M * K, seed=K + 25).reshape(M, K)
    U = synth.normal(M * K, seed=K + 26).reshape(M, K)
    Y0, H = holo.DeviceBuffer(4 * M * N), holo.DeviceBuffer(4 * M * K)
    rows = sorted({0, M // 2, M - 1})
    dW, dU = up(holo, src), up(holo, U)
    lib.holo_matmul_batch(Y0.ptr, dW.ptr, up(holo, X).ptr, M, N, K, t)
    lib.cuda_sync()
    y0 = down(Y0, M * N).reshape(M, N)
    X[rows, 7] = big
    dX, dT, dZ = up(holo, X), holo.DeviceBuffer(4 * M * N), up(holo, np.zeros(M * N, np.float32))
    lib.holo_matmul_batch(Y0.ptr, dW.ptr, dX.ptr, M, N, K, t)
    lib.cuda_silu_mul(H.ptr, dX.ptr, dU.ptr, M * K)
    lib.holo_matmul_batch(dT.ptr, dW.ptr, H.ptr, M, N, K, t)
    lib.holo_matmul_batch_swiglu_add(dZ.ptr, dW.ptr, dX.ptr, dU.ptr, dZ.ptr, M, N, K, t)
    lib.cuda_sync()
    holo.check("range")
    y = down(Y0, M * N).reshape(M, N)
    rest = np.setdiff1d(np.arange(M), rows)
    assert np.array_equal(y[rest].view(np.uint32), y0[rest].view(np.uint32))
    check_rows(y, X, w, np.array(rows), t, K)
    check_rows(down(dT, M * N).reshape(M, N), down(H, M * K).reshape(M, K), w, np.array(rows), t, K)
    assert np.array_equal(down(dZ, M * N), 0.0 + down(dT, M * N))


@pytest.mark.parametrize("t", [Q4_0, Q8_0, Q4_K, Q6_K, F16], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("M,N,K", [(16, 500, 256), (16, 500, 1024), (3, 500, 2048), (16, 1000, 4096), (23, 500, 11008),
                                   (40, 300, 14336), (63, 4096, 4096)])
def test_few_rows_no_less_precise_than_gemvs(holo, synth, oracle, t, M, N, K):
    """The error against 64 bits (2-norm) is no larger than that of the GEMVs,
    one per row, that these products replace."""
    print(f"case precision {NAMES[t]} {M}x{N}x{K}", flush=True)
    lib = holo.lib()
    src, w = weights(synth, oracle, t, N, K, seed=M + N + K)
    X = synth.normal(M * K, seed=K + 35).reshape(M, K)
    dW, dX, dY, dG = up(holo, src), up(holo, X), holo.DeviceBuffer(4 * M * N), holo.DeviceBuffer(4 * M * N)
    lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
    for m in range(M):
        lib.holo_matmul(dG.ptr + 4 * m * N, dW.ptr, dX.ptr + 4 * m * K, N, K, t)
    lib.cuda_sync()
    holo.check("precision")
    truth = X.astype(np.float64) @ w.astype(np.float64).T
    here, gemv = (np.linalg.norm(down(d, M * N).reshape(M, N) - truth) / np.linalg.norm(truth) for d in (dY, dG))
    print(f"  {here:.2e}, one GEMV a row {gemv:.2e}", flush=True)
    assert here <= gemv


@pytest.mark.parametrize("M,N,K", [(3, 40, 1056), (17, 500, 4096), (48, 100, 2080), (100, 64, 512)])
def test_few_rows_infinite_f16_weights(holo, synth, oracle, M, N, K):
    """Infinite F16 weights: an infinity of the products' sign (NaN against a
    zero activation, infinities of both signs and a NaN weight) in their
    outputs, the other outputs' bits unchanged."""
    print(f"case infinite f16 weights {M}x{N}x{K}", flush=True)
    lib = holo.lib()
    src, w = weights(synth, oracle, F16, N, K, seed=M + N)
    X = synth.normal(M * K, seed=K + 45).reshape(M, K)
    X[1, K // 2] = 0.0
    X[2, K // 2] = 0.5  # its low half is zero
    dX, outs = up(holo, X), []
    h = np.array(src).view(np.float16).reshape(N, K).copy()
    for k in range(2):
        if k:
            h[5, K // 2], h[9, K - 1], h[20, 3], h[20, 40], h[31, 7] = np.inf, -np.inf, np.inf, -np.inf, np.nan
        dW, dY = up(holo, h.view(np.uint16)), holo.DeviceBuffer(4 * M * N)
        lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, F16)
        lib.cuda_sync()
        outs.append(down(dY, M * N).reshape(M, N))
    holo.check("infinite f16 weights")
    rest = np.setdiff1d(np.arange(N), [5, 9, 20, 31])
    assert np.array_equal(outs[0][:, rest].view(np.uint32), outs[1][:, rest].view(np.uint32))
    with np.errstate(invalid="ignore"):
        for n in (5, 9, 20, 31):
            want = (X.astype(np.float64) * h[n].astype(np.float64)).sum(1)
            assert np.array_equal(outs[1][:, n], want.astype(np.float32), equal_nan=True), n
