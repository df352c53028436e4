"""Scheme II shapes that take the four-slot ring (deep_ring, ozablas_amd/csrc/k_igemm.hip: large operand planes,
few products per byte) and neighbours that do not, at edges of tiles and parts, against the oracle; alpha,
beta and transposes through the BLAS-style call."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu

CASES = [(1, 40, 9000, 20), (33, 257, 12001, 20), (300, 129, 8803, 20), (513, 70, 6000, 20), (2, 513, 100000, 1),
         (700, 3, 30000, 3), (40, 260, 5900, 20), (64, 64, 8700, 20), (64, 64, 8900, 20), (257, 255, 5889, 20)]


@pytest.mark.parametrize("M,N,K,S", CASES)
def test_matches_the_oracle(ex, orc, M, N, K, S):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 17)
    want = orc.s2_gemm(A, B, S)
    ws = oz.WorkspaceScheme2(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    oz.ozaki_scheme2_gemm(ws, dA, dB, dC)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
    At, Bt = ex.to_device(np.ascontiguousarray(A.T)), ex.to_device(np.ascontiguousarray(B.T))
    dC.upload(np.zeros((M, N)))
    oz.gemm(ex, M, N, K, 1.0, At, M, Bt, K, 0.0, dC, N, transA=oz.OP_T, transB=oz.OP_T, scheme=2, slices=S)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
