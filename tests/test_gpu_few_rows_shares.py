"""The activation split of the few-row product with a row shared by several
workgroups: the forms and row counts at the edges of the share rule (whole
rows from 129 up; shares without a float4 of their own at K = 32), and SwiGLU
rows whose largest value sits on a power of two, where silu underflows, and
where it is not finite.

Bar: test_gpu_few_rows' for the plain product; the SwiGLU form is the bits of
cuda_silu_mul followed by the plain product.
"""
import numpy as np
import pytest

from test_gpu_batch_exact import Q4_0, Q8_0, check_rows, down, up, weights

pytestmark = pytest.mark.gpu

CASES = [(Q4_0, 5, 32), (Q8_0, 16, 16384), (Q4_0, 23, 11008), (Q4_0, 64, 4096), (Q8_0, 85, 2304), (Q4_0, 128, 1056),
         (Q4_0, 129, 1024)]


@pytest.mark.parametrize("t,M,K", CASES)
def test_few_rows_shares(holo, synth, oracle, t, M, K):
    print(f"case shared rows type {t} {M}x{K}", flush=True)
    lib = holo.lib()
    N = 40
    src, w = weights(synth, oracle, t, N, K, seed=M + K)
    X = synth.normal(M * K, seed=K + 1).reshape(M, K)
    G = synth.normal(M * K, seed=K + 2).reshape(M, K)
    U = synth.normal(M * K, seed=K + 3).reshape(M, K)
    G[:4], U[:4] = 0.5, 0.25
    G[0, K - 1], U[0, K - 1] = 64.0, 2.0                              # 128
    G[1, K // 2], U[1, K // 2] = 64.0, np.nextafter(np.float32(2), np.float32(0))
    G[2, :], U[2, :] = -90.0, 1e30                                    # 1 / (1 + e^90) underflows
    G[3, 0] = np.inf
    dW, dX, dG, dU = up(holo, src), up(holo, X), up(holo, G), up(holo, U)
    dY, dT, dZ, dH = (holo.DeviceBuffer(4 * n) for n in (M * N, M * N, M * N, M * K))
    lib.holo_matmul_batch(dY.ptr, dW.ptr, dX.ptr, M, N, K, t)
    lib.cuda_silu_mul(dH.ptr, dG.ptr, dU.ptr, M * K)
    lib.holo_matmul_batch(dT.ptr, dW.ptr, dH.ptr, M, N, K, t)
    dR = up(holo, np.zeros(M * N, np.float32))
    lib.holo_matmul_batch_swiglu_add(dZ.ptr, dW.ptr, dG.ptr, dU.ptr, dR.ptr, M, N, K, t)
    lib.cuda_sync()
    holo.check("shared rows")
    check_rows(down(dY, M * N).reshape(M, N), X, w, np.arange(M), t, K)
    assert np.array_equal(down(dZ, M * N), 0.0 + down(dT, M * N), equal_nan=True)


@pytest.mark.parametrize("M,K", [(3, 1056), (23, 11008), (85, 4096)])
def test_few_rows_shares_end_of_silu(holo, synth, oracle, M, K):
    """Ordinary rows whose largest silu(g) u is at a g where 1 / (1 + e^-g) is
    subnormal, as u is huge there: the row's scale has to come from it."""
    print(f"case end of silu {M}x{K}", flush=True)
    lib = holo.lib()
    N = 40
    src, w = weights(synth, oracle, Q8_0, N, K, seed=M + K)
    G = synth.normal(M * K, seed=K + 2).reshape(M, K)
    U = synth.normal(M * K, seed=K + 3).reshape(M, K)
    for r, (g, u) in enumerate([(-88.0, 1e38), (-87.4, -3e38), (-88.6, 2e38)]):
        G[r, K // 3 + r], U[r, K // 3 + r] = g, u
    dW, dG, dU, dR = up(holo, src), up(holo, G), up(holo, U), up(holo, np.zeros(M * N, np.float32))
    dT, dZ, dH = (holo.DeviceBuffer(4 * n) for n in (M * N, M * N, M * K))
    lib.cuda_silu_mul(dH.ptr, dG.ptr, dU.ptr, M * K)
    lib.holo_matmul_batch(dT.ptr, dW.ptr, dH.ptr, M, N, K, Q8_0)
    lib.holo_matmul_batch_swiglu_add(dZ.ptr, dW.ptr, dG.ptr, dU.ptr, dR.ptr, M, N, K, Q8_0)
    lib.cuda_sync()
    holo.check("end of silu")
    H = down(dH, M * K).reshape(M, K)
    assert all(np.max(np.abs(H[r])) > 20 for r in range(3))
    check_rows(down(dZ, M * N).reshape(M, N), H, w, np.arange(M), Q8_0, K)
    assert np.array_equal(down(dZ, M * N), 0.0 + down(dT, M * N))
