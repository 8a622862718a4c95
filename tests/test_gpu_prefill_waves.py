"""Prompt attention where few workgroups take eight waves each, and at the
edges of its 32-key tiles (keys staged through LDS in whole rows): the last
tile of 1, 31 and 32 keys, fewer tiles than waves, head sizes of one and two
staged halves, grouped heads, a KV stride that is no power of two.

Bar: float64 numpy, 2e-6 normwise (the split products keep 22 bits; a score is
a 128-term sum, see test_gpu_decode_ranges).
"""
import numpy as np
import pytest

from oracle.oracle import normwise_err
from test_gpu_attention import down, up, want_attention

pytestmark = pytest.mark.gpu

CASES = [(128, 4, 2, 5, 123), (128, 4, 2, 5, 124), (128, 4, 4, 32, 96), (128, 8, 2, 33, 128), (128, 3, 3, 70, 250),
         (64, 4, 1, 17, 239), (64, 8, 8, 40, 500), (32, 6, 2, 64, 193), (128, 32, 8, 256, 33), (128, 32, 8, 257, 33)]


@pytest.mark.parametrize("hd,nh,nkv,rows,pos0", CASES)
def test_prefill_waves(holo, synth, hd, nh, nkv, rows, pos0):
    print(f"case prefill waves hd {hd} heads {nh}/{nkv} rows {rows} pos0 {pos0}", flush=True)
    lib = holo.lib()
    kv_dim, kv_len = nkv * hd, pos0 + rows
    q, kc, vc = (synth.normal(n, seed=80 + i) for i, n in enumerate((rows * nh * hd, (kv_len + 40) * kv_dim,
                                                                     (kv_len + 40) * kv_dim)))
    kc[kv_len * kv_dim:] = np.nan  # positions after the prompt do not count, whatever they hold
    vc[kv_len * kv_dim:] = np.nan
    dq, dk, dv = up(holo, q), up(holo, kc), up(holo, vc)
    d = up(holo, np.full(rows * nh * hd + 8, 7.0, np.float32))
    lib.holo_attention_prefill(d.ptr, dq.ptr, dk.ptr, dv.ptr, rows, pos0, hd, nh, nkv)
    lib.cuda_sync()
    holo.check("prefill waves")
    got = down(d, rows * nh * hd + 8)
    assert np.all(got[rows * nh * hd:] == 7.0)
    got = got[:rows * nh * hd].reshape(rows, nh * hd)
    K, V = (a.reshape(-1, nkv, hd).astype(np.float64) for a in (kc, vc))
    for m in sorted({0, 1, rows // 2, rows - 2, rows - 1}):
        want = want_attention(q[m * nh * hd:(m + 1) * nh * hd], K, V, nh, nkv, hd, pos0 + m + 1)
        assert normwise_err(got[m], want) <= 2e-6, m
