"""Scheme II calls with 64 x 64 and 128 x 128 tiles (small_edge, ozablas_amd/csrc/plan_host.cpp) at the edges of
those tiles, of the ring's four stages and of the rule's lines, and neighbours on the other side of the lines
(256 x 256 tiles, also on the four-slot ring); digits left in the workspace; alpha and beta."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 1, 1), (63, 64, 128, 20), (65, 129, 129, 7), (64, 128, 384, 3), (127, 63, 512, 11), (128, 65, 513, 4),
         (257, 255, 640, 16), (512, 512, 300, 8), (512, 513, 300, 8), (513, 511, 1025, 9), (1024, 1000, 130, 8),
         (900, 897, 200, 8), (700, 1030, 257, 10), (40, 70, 16384, 5), (40, 70, 16385, 5), (500, 390, 4096, 8),
         (450, 520, 4097, 10), (640, 700, 2049, 9), (896, 1024, 2200, 8), (300, 290, 20000, 9), (513, 70, 17000, 9),
         (600, 600, 5000, 13)]


@pytest.mark.parametrize("M,N,K,S", CASES)
def test_matches_the_oracle(ex, orc, M, N, K, S):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 23)
    want = orc.s2_gemm(A, B, S)
    ws = oz.WorkspaceScheme2(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    for _ in range(2):
        oz.ozaki_scheme2_gemm(ws, dA, dB, dC)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
    if M * N * K * S < 3e8:
        L = oz._lib
        ap, bp = ws.planar_slices()
        pl = ex.alloc(S * M * N)
        L.check(L.lib.oza_unpack_digits(ex.ctx, M, N, S, ws.C_tc.ptr, pl.ptr))
        np.testing.assert_array_equal(pl.download((S, M, N), np.uint8), orc.crt_digits(orc.s2_products(ap, bp)))
    C0 = np.ones((M, N))
    dC.upload(C0)  # -0.5 * X + 2 * 1 rounded once
    oz.gemm(ex, M, N, K, -0.5, dA, K, dB, N, 2.0, dC, N, scheme=2, slices=S)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), (want * -0.5 + 2.0).view(np.uint64))
