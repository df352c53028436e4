"""Edge tiles of the GEMMs: waves that compute all, half or a quarter of their part of a tile, or nothing
(for_part, ozablas_amd/csrc/igemm_core.hpp), at every 32-row edge of a 256 x 256 tile and beside it."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu

EDGES = [1, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 191, 192, 193, 224, 225, 255, 256, 257, 320, 385]


@pytest.mark.parametrize("scheme,S,K", [(2, 3, 129), (2, 5, 640), (1, 3, 129), (1, 4, 515)])
@pytest.mark.parametrize("M", EDGES)
def test_edges_match_the_oracle(ex, orc, scheme, S, K, M):
    import ozablas_amd as oz

    for N in EDGES[(M * 7) % 3::3]:
        A, B = gen_pair(orc, M, N, K, 1.0, M + N)
        ws = (oz.WorkspaceScheme2 if scheme == 2 else oz.WorkspaceScheme1)(ex, M, N, K, S)
        dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
        (oz.ozaki_scheme2_gemm if scheme == 2 else oz.ozaki_scheme1_gemm)(ws, dA, dB, dC)
        ex.synchronize()
        want = (orc.s2_gemm if scheme == 2 else orc.s1_gemm)(A, B, S)
        np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64), str(N))
        ws.free()


@pytest.mark.parametrize("tile", [0, 64, 128, 256])
def test_grouped_edges_match_the_oracle(ex, orc, tile):
    import ozablas_amd as oz
    from test_gpu_group import inputs, run_group, same_bits

    shapes = [(M, EDGES[(5 * i + tile // 64) % len(EDGES)], 200 + 64 * (i % 3), 4) for i, M in enumerate(EDGES)]
    data = inputs(orc, shapes, 3)
    g = oz.GroupScheme2(ex, shapes, tile=tile)
    for (A, B), (M, N, K, S), C in zip(data, shapes, run_group(ex, g, shapes, data, False)):
        assert same_bits(C, orc.s2_gemm(A, B, S)), (M, N, K, S)
    g.free()
