"""cuda_matmul_q6_k with enough rows for the staged kernel: an odd row count,
one and two passes of 16 superblocks a row (whole and partial), long rows, the
longest staged one (27392: 160 KiB of LDS) and the first past it, matrices off
4- and 16-byte alignment, and activations that are tiny, zero in places, not
finite (NaN, as from the straight kernel, whose 32 sum(x) meets sum(q x)) or
with outliers.

Bar, from the number formats: a group of 16 activations is within 2^-24 of its
largest magnitude a each, its sum, scale and product round five times, a lane
adds 4 groups a pass and the wave's tree 6 more: (4 passes + 16) 2^-24 sum over
groups a_g sum |w|.
"""
import os
import pathlib
import subprocess
import sys

import numpy as np
import pytest

from test_gpu_batch_exact import Q6_K, down, up, weights

pytestmark = pytest.mark.gpu

CASES = [(16385, 256, 0), (16384, 4096, 2), (17001, 4352, 14), (16390, 768, 6), (8193, 24576, 0), (8193, 26624, 2),
         (8193, 27392, 0), (8193, 27392, 6), (8193, 27648, 2)]


@pytest.mark.parametrize("rows,K,off", CASES)
def test_q6_many_rows(holo, synth, oracle, rows, K, off):
    print(f"case q6 rows {rows}x{K} offset {off}", flush=True)
    lib = holo.lib()
    n = 67  # distinct rows, repeated down the matrix
    src, w = weights(synth, oracle, Q6_K, n, K, seed=K + off)
    raw = np.frombuffer(np.ascontiguousarray(src).tobytes(), np.uint8).reshape(n, -1)
    raw = np.concatenate([raw] * (rows // n + 1))[:rows].reshape(-1)
    buf = up(holo, np.concatenate([np.zeros(off, np.uint8), raw]))
    w = np.asarray(w, np.float64).reshape(n, K)
    for case in ("plain", "zeros", "tiny", "inf"):
        x = synth.normal(K, seed=K + 9)
        if case == "zeros":
            x[: K // 2 - 3] = 0.0
            x[K - 5] = 3e4
        elif case == "tiny":
            x *= np.float32(1e-32)
        elif case == "inf":
            x[K // 3] = -np.inf
        d = up(holo, np.full(rows + 4, 7.0, np.float32))
        lib.cuda_matmul_q6_k(d.ptr, buf.ptr + off, up(holo, x).ptr, rows, K)
        lib.cuda_sync()
        holo.check("q6 rows")
        got = down(d, rows + 4)
        assert np.all(got[rows:] == 7.0)
        if case == "inf":
            assert np.all(np.isnan(got[:rows]))
            continue
        x = x.astype(np.float64)
        a = np.abs(x).reshape(-1, 16).max(1)
        bound = (4 * ((K // 256 + 15) // 16) + 16) * 2.0**-24 * (np.abs(w).reshape(n, -1, 16).sum(2) @ a) + 2.0**-140
        err = np.abs(got[:n] - w @ x)
        print(f"  {case}: max err / bound {np.max(err / bound):.3f}", flush=True)
        assert np.all(err <= bound), case
        assert np.array_equal(got[:rows], np.concatenate([got[:n]] * (rows // n + 1))[:rows])


@pytest.mark.parametrize("ratio", [1.0, 30.0, 1e3, 1e6])
def test_q6_outliers(holo, synth, oracle, ratio):
    """An outlier in every group of 16, facing weights of zero (q = 32): the
    outliers' rounding is all that shows, in the staged kernel (a group's fixed
    point) as in the straight one (sum(q x) - 32 sum(x)).  The staged kernel's
    error against 64 bits (2-norm) stays within 1.2 of the straight one's, and
    below it without outliers."""
    print(f"case q6 outliers {ratio}", flush=True)
    lib = holo.lib()
    n, rows, K = 500, 16400, 4096
    src, _ = weights(synth, oracle, Q6_K, n, K, seed=77)
    raw = np.frombuffer(np.ascontiguousarray(src).tobytes(), np.uint8).reshape(n, K // 256, 210).copy()
    x = synth.normal(K, seed=78)
    if ratio > 1:
        for i in range(0, K, 16):
            i += (7 * i // 16) % 16
            x[i] *= np.float32(ratio)
            b, r = divmod(i, 256)
            h, r = divmod(r, 128)
            j, l = divmod(r, 32)
            low, high = 64 * h + 32 * (j & 1) + l, 128 + 32 * h + l
            raw[:, b, low] &= 0x0F if j >> 1 else 0xF0
            raw[:, b, high] = raw[:, b, high] & ~np.uint8(3 << 2 * j) | np.uint8(2 << 2 * j)
    w = np.asarray(oracle.dequant(Q6_K, raw.reshape(-1), n * K), np.float64).reshape(n, K)
    many = np.concatenate([raw.reshape(n, -1)] * (rows // n + 1))[:rows].reshape(-1)
    dM, dx = up(holo, many), up(holo, x)
    ds, dm = holo.DeviceBuffer(4 * n), holo.DeviceBuffer(4 * rows)
    lib.cuda_matmul_q6_k(ds.ptr, dM.ptr, dx.ptr, n, K)
    lib.cuda_matmul_q6_k(dm.ptr, dM.ptr, dx.ptr, rows, K)
    lib.cuda_sync()
    holo.check("q6 outliers")
    truth = w @ x.astype(np.float64)
    straight, staged = (np.linalg.norm(down(d, n) - truth) / np.linalg.norm(truth) for d in (ds, dm))
    print(f"  straight {straight:.2e}, staged {staged:.2e}", flush=True)
    assert staged <= (1.2 if ratio > 1 else 1.0) * straight


def test_q6_forced_rows(holo, synth, oracle):
    """HOLO_Q6K_ROWS keeps straight loads at any row count: the bits of a call
    of few rows.  (It is read once a process, so in one of its own.)"""
    code = """
import sys
sys.path[:0] = ["google-classic_amd", "tests", "."]
import numpy as np, holo_mi355x as holo
from holo_mi355x import synth
holo.load(); holo.init()
lib = holo.lib()
raw = np.frombuffer(np.ascontiguousarray(synth.blocks(14, 100, 4096, 5)).tobytes(), np.uint8)
w = holo.DeviceBuffer.from_array(np.tile(raw, 165))
x = holo.DeviceBuffer.from_array(synth.normal(4096, seed=6))
a, b = holo.DeviceBuffer(400), holo.DeviceBuffer(4 * 16500)
lib.cuda_matmul_q6_k(a.ptr, w.ptr, x.ptr, 100, 4096)
lib.cuda_matmul_q6_k(b.ptr, w.ptr, x.ptr, 16500, 4096)
lib.cuda_sync()
holo.check("forced rows")
assert np.array_equal(np.tile(a.download(np.float32, 100), 165), b.download(np.float32, 16500))
"""
    root = pathlib.Path(__file__).resolve().parent.parent
    r = subprocess.run([sys.executable, "-c", code], cwd=root, env={**os.environ, "HOLO_Q6K_ROWS": "2"}, timeout=60,
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
