"""GPU parity of the exact product's 64 x 256 tiles at ragged shapes.  Up to
1024 rows most small shapes run the tiles for few rows (test_gpu_few_rows);
every shape here runs the large ones, which each test asserts: more than 1024
rows, or shapes that fill the chip.  Rows that are no multiple of 64 or 32,
columns ragged against 32, 64 and 256, odd block counts (the first tiling)
and even ones (the second), K in parts, the fused and multi forms, rows far
from unit scale, and a prepared Q6_K copy.

Bars: test_gpu_batch_exact's.
"""
import ctypes as C

import numpy as np
import pytest

from test_gpu_batch_exact import F16, NAMES, Q4_0, Q4_K, Q6_K, Q8_0, check_rows, down, up, weights

pytestmark = pytest.mark.gpu


def on_large_tiles(holo, t, M, N, K, prepared=0):
    return holo.lib().holo_few_rows_plan(t, M, N, K, prepared, (C.c_int * 4)()) == 0


def _shapes():
    rng = np.random.default_rng(77)
    out = []
    for t in (Q4_0, Q8_0, Q4_K, Q6_K, F16):
        step = 256 if t in (Q4_K, Q6_K) else 32
        for N in (1, 8, 31, 64, 100, 257, 330):
            M = int(rng.choice([1025, 1030, 1055, 1057, 1088, 1100]))
            out.append((t, M, N, step * int(rng.integers(1, 5 if step == 256 else 25))))
        if step == 32:  # odd and even block counts, long rows
            out += [(t, 1029, 200, 1056), (t, 1029, 200, 1088), (t, 1031, 130, 4128)]
    # fewer rows that fill the chip
    return out + [(Q4_0, 300, 5000, 2336), (Q4_0, 512, 11000, 2080), (Q8_0, 300, 5000, 2336), (F16, 256, 11000, 2080),
                  (F16, 192, 4090, 2080), (F16, 300, 4090, 4096), (Q4_K, 512, 11000, 2304), (Q6_K, 512, 11000, 2304)]


SHAPES = _shapes()


@pytest.mark.parametrize("t,M,N,K", SHAPES, ids=[f"{NAMES[t]}-{m}x{n}x{k}" for t, m, n, k in SHAPES])
def test_exact_tiles(holo, synth, oracle, t, M, N, K):
    print(f"case exact tiles {NAMES[t]} {M}x{N}x{K}", flush=True)
    assert on_large_tiles(holo, t, M, N, K)
    lib = holo.lib()
    src, w = weights(synth, oracle, t, N, K, seed=7 * M + 3 * N + K)
    X = synth.normal(M * K, seed=M + K).reshape(M, K)
    dW, dX, outs = up(holo, src), up(holo, X), []
    for _ in range(2):
        dY = up(holo, np.full(M * N + 64, 7.0, np.float32))
        lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
        lib.cuda_sync()
        holo.check("exact tiles")
        outs.append(down(dY, M * N + 64))
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert np.all(outs[0][M * N:] == 7.0)
    rows = np.arange(M) if M * N * K <= 2 * 10**9 else np.unique(np.r_[0:M:32, 31:M:32, M - 1])
    check_rows(outs[0][:M * N].reshape(M, N), X, w, rows, t, K)


@pytest.mark.parametrize("t,K", [(Q4_0, 512), (Q4_0, 544), (Q8_0, 512), (Q8_0, 544), (Q4_K, 512), (Q6_K, 512), (F16, 512),
                                 (F16, 544)], ids=lambda v: str(v))
def test_exact_tiles_forms(holo, synth, oracle, t, K):
    """Three matrices in one launch, mixed types, the add in the store and the
    SwiGLU in the split: the bits of single calls and of the unfused sequence."""
    print(f"case exact tiles forms {NAMES[t]} K {K}", flush=True)
    lib = holo.lib()
    M, Ns = 1030, (256, 128, 128)
    assert all(on_large_tiles(holo, t, M, n, K) for n in Ns)
    T = (t, t, Q8_0 if t != Q8_0 else Q4_0)
    srcs, ws = zip(*[weights(synth, oracle, tt, n, K, seed=60 + i) for i, (tt, n) in enumerate(zip(T, Ns))])
    X = synth.normal(M * K, seed=61).reshape(M, K)
    dWs, dX = [up(holo, s) for s in srcs], up(holo, X)
    dYm, singles = ([holo.DeviceBuffer(4 * M * n) for n in Ns] for _ in range(2))
    lib.holo_matmul_batch_multi_types((C.c_void_p * 3)(*[d.ptr for d in dYm]), (C.c_void_p * 3)(*[d.ptr for d in dWs]),
                                      (C.c_int * 3)(*T), (C.c_int * 3)(*Ns), 3, dX.ptr, M, K)
    for i, n in enumerate(Ns):
        lib.holo_matmul_batch(singles[i].ptr, dWs[i].ptr, dX.ptr, M, n, K, T[i])
    two = [holo.DeviceBuffer(4 * M * n) for n in Ns[:2]]
    lib.holo_matmul_batch_multi((C.c_void_p * 2)(*[d.ptr for d in two]), (C.c_void_p * 2)(*[d.ptr for d in dWs[:2]]),
                                (C.c_int * 2)(*Ns[:2]), 2, dX.ptr, M, K, t)
    N = Ns[0]
    U, R = synth.normal(M * K, seed=63).reshape(M, K), synth.normal(M * N, seed=64).reshape(M, N) * 5.0
    dG, dU, dH, dT = up(holo, X), up(holo, U), holo.DeviceBuffer(4 * M * K), holo.DeviceBuffer(4 * M * N)
    lib.cuda_silu_mul(dH.ptr, dG.ptr, dU.ptr, M * K)
    lib.holo_matmul_batch(dT.ptr, dWs[0].ptr, dH.ptr, M, N, K, t)
    dS, dZ = up(holo, R), up(holo, R)
    lib.holo_matmul_batch_add(dS.ptr, dWs[0].ptr, dX.ptr, dS.ptr, M, N, K, t)
    lib.holo_matmul_batch_swiglu_add(dZ.ptr, dWs[0].ptr, dG.ptr, dU.ptr, dZ.ptr, M, N, K, t)
    lib.cuda_sync()
    holo.check("exact tiles forms")
    for i, n in enumerate(Ns):
        got = down(dYm[i], M * n)
        assert np.array_equal(got.view(np.uint32), down(singles[i], M * n).view(np.uint32)), i
        check_rows(got.reshape(M, n), X, ws[i], np.unique(np.r_[0:M:32, 31:M:32, M - 1]), T[i], K)
    for i, n in enumerate(Ns[:2]):
        assert np.array_equal(down(two[i], M * n).view(np.uint32), down(singles[i], M * n).view(np.uint32)), i
    assert np.array_equal(down(dS, M * N).reshape(M, N), (R + down(singles[0], M * N).reshape(M, N)).astype(np.float32))
    assert np.array_equal(down(dZ, M * N).reshape(M, N), (R + down(dT, M * N).reshape(M, N)).astype(np.float32))


@pytest.mark.parametrize("t", [Q4_0, Q8_0, Q4_K, Q6_K, F16], ids=lambda t: NAMES[t])
def test_exact_tiles_row_range(holo, synth, oracle, t):
    """Rows near 1e5, 1e30, 1e-6 and 1e-30, and a zero row, beside unit ones."""
    print(f"case exact tiles row range {NAMES[t]}", flush=True)
    M, N, K = 1026, 100, 512
    assert on_large_tiles(holo, t, M, N, K)
    src, w = weights(synth, oracle, t, N, K, seed=90 + t)
    X = synth.normal(M * K, seed=91).reshape(M, K)
    scales = {0: 1e5, 1: 7e4, 65: 1e30, 66: 1e-6, M - 1: 1e-30, M - 2: 0.0}
    for r, f in scales.items():
        X[r] *= np.float32(f)
    dW, dX, dY = up(holo, src), up(holo, X), holo.DeviceBuffer(4 * M * N)
    holo.lib().holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
    holo.lib().cuda_sync()
    holo.check("exact tiles row range")
    got = down(dY, M * N).reshape(M, N)
    assert np.all(np.isfinite(got)) and np.all(got[M - 2] == 0.0)
    for r in [*range(8), 64, 65, 66, M - 3, M - 1]:
        check_rows(got, X, w, np.array([r]), t, K)


@pytest.mark.parametrize("M,N,K", [(1030, 384, 1024), (100, 14336, 4096)])
def test_exact_tiles_prepared_q6_k(holo, synth, oracle, M, N, K):
    """A prepared copy on the large tiles: within the bound, and where the call
    without a copy runs them too, its bits."""
    print(f"case exact tiles prepared {M}x{N}x{K}", flush=True)
    assert on_large_tiles(holo, Q6_K, M, N, K, prepared=1)
    lib = holo.lib()
    src, w = weights(synth, oracle, Q6_K, N, K, seed=M + N)
    X = synth.normal(M * K, seed=K + 23).reshape(M, K)
    dW, dX, dY = up(holo, src), up(holo, X), holo.DeviceBuffer(4 * M * N)
    lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, Q6_K)
    lib.cuda_sync()
    y0 = down(dY, M * N).reshape(M, N)
    assert lib.holo_prefill_prepare(dW.ptr, N, K, Q6_K) == 0
    try:
        lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, Q6_K)
        lib.cuda_sync()
    finally:
        lib.holo_prefill_release(dW.ptr)
    holo.check("exact tiles prepared")
    y1 = down(dY, M * N).reshape(M, N)
    check_rows(y1, X, w, np.unique(np.r_[0:M:32, 31:M:32, M - 1]), Q6_K, K)
    if on_large_tiles(holo, Q6_K, M, N, K):
        assert np.array_equal(y1.view(np.uint32), y0.view(np.uint32))
