"""cuda_matmul_q6_k with enough rows for the staged kernel: an odd row count,
one and two passes of 16 superblocks a row (whole and partial), the largest
staged row and the first past it, matrices off 4- and 16-byte alignment, and
activations that are tiny, zero in places or not finite.

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

CASES = [(16385, 256, 0), (16384, 4096, 2), (17001, 4352, 14), (16390, 768, 6), (8193, 24576, 0), (8193, 26624, 2)]


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
