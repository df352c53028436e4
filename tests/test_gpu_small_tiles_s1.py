"""Scheme I calls with 64 x 64 and 128 x 128 tiles (small_edge_s1, ozablas_amd/csrc/plan_host.cpp) at the edges of
those tiles, of the ring's four stages and of the rule's lines, and neighbours on the other side; the group
products left in the workspace feed a second call; alpha and beta; a workspace of exactly the S planes."""
import numpy as np
import pytest

from test_gpu_item_split import sizes
from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 1, 1), (63, 64, 128, 20), (65, 129, 129, 7), (64, 128, 384, 3), (127, 63, 512, 11), (257, 255, 640, 9),
         (512, 512, 300, 8), (512, 513, 300, 8), (100, 90, 2100, 5), (100, 90, 2700, 5), (760, 1030, 257, 3),
         (1000, 1000, 130, 4), (1024, 1024, 385, 5), (1100, 900, 1025, 6), (1290, 1300, 140, 6), (600, 620, 600, 8)]


@pytest.mark.parametrize("M,N,K,S", CASES)
def test_matches_the_oracle(ex, orc, M, N, K, S):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 29)
    want = orc.s1_gemm(A, B, S)
    ws = oz.WorkspaceScheme1(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    for _ in range(2):
        oz.ozaki_scheme1_gemm(ws, dA, dB, dC)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
    w = ex.alloc(sizes(1, M, N, K, S)[0])
    dC.upload(np.ones((M, N)))  # -0.5 * X + 2 * 1 rounded once
    oz.gemm(ex, M, N, K, -0.5, dA, K, dB, N, 2.0, dC, N, scheme=1, slices=S, workspace=w)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), (want * -0.5 + 2.0).view(np.uint64))
