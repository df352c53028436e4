"""Steps 1 and 2 in one launch for 2048 < K <= 4096 (blocks of 8 rows; one_pass, ozablas_amd/csrc/k_slice.hip)
and the neighbouring shapes that stay on two: shifts and planes against the separate kernels of the stage
entry points and the oracle, and row-contiguous and K-contiguous storage of both operands."""
import pytest

import test_gpu_one_pass as short

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 2049, 20), (7, 9, 2050, 1), (33, 64, 4096, 3), (31, 65, 4095, 8), (8, 1000, 3000, 17),
         (1000, 990, 2200, 5), (1024, 1024, 2177, 4), (1030, 1010, 2500, 4), (1500, 1350, 2300, 3),
         (2040, 2050, 2050, 3), (2080, 2060, 2050, 3), (60, 50, 4097, 6)]


@pytest.mark.parametrize("scheme", [1, 2])
@pytest.mark.parametrize("M,N,K,S", CASES)
def test_planes_match_separate_steps(ex, orc, rng, scheme, M, N, K, S):
    short.test_planes_match_separate_steps(ex, orc, rng, scheme, M, N, K, S)


@pytest.mark.parametrize("scheme,S", [(2, 15), (1, 6)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_orientations(ex, orc, scheme, S, ta, tb):
    import numpy as np

    import ozablas_amd as oz
    from test_gpu_parity import gen_pair

    M, N, K = 70, 45, 2601
    A, B = gen_pair(orc, M, N, K, 1.0, 5)
    sA, sB = (np.pad(X.T if t else X, ((0, 0), (0, 3))) for X, t in ((A, ta), (B, tb)))
    dA, dB, dC = ex.to_device(sA), ex.to_device(sB), ex.alloc(8 * M * N)
    oz.gemm(ex, M, N, K, 1.0, dA, sA.shape[1], dB, sB.shape[1], 0.0, dC, N, transA=ta, transB=tb, scheme=scheme, slices=S)
    ex.synchronize()
    want = (orc.s2_gemm if scheme == 2 else orc.s1_gemm)(A, B, S)
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
