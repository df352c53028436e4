"""Steps 1 and 2 of grouped problems with K <= 2048 in one pass (k_group_pass): K at the edges of its row
counts per block (64, 32, 16, 8), of a unit and of the path; rows at the edges of a block and of a fragment
block; one, two and three words per value; problems on both sides of the path in one group; non-finite
values; rows that start off a 16-byte boundary."""
import numpy as np
import pytest

from test_gpu_group import inputs, run_group, same_bits, single
from test_gpu_parity import special_matrix

pytestmark = pytest.mark.gpu

KS = [1, 15, 17, 128, 129, 256, 257, 384, 512, 513, 1000, 1024, 1025, 2047, 2048, 2049]
ROWS = [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130]


def cases(seed):
    r = np.random.default_rng(seed)
    return [(int(r.choice(ROWS)), int(r.choice(ROWS)), K, int(s)) for K in KS for s in (3, r.integers(8, 14), r.integers(17, 21))]


@pytest.mark.parametrize("seed", [1, 2])
def test_group_pass_matches_the_oracle(ex, orc, seed):
    import ozablas_amd as oz

    shapes = cases(seed)
    data = inputs(orc, shapes, 40 * seed)
    g = oz.GroupScheme2(ex, shapes)
    for graph in (False, True):
        for (A, B), (M, N, K, S), C in zip(data, shapes, run_group(ex, g, shapes, data, graph)):
            assert same_bits(C, orc.s2_gemm(A, B, S)), (M, N, K, S)
    g.free()


def test_group_pass_non_finite(ex, orc, rng):
    import ozablas_amd as oz

    shapes = [(M, N, K, S) for M, N, K, S in cases(3) if K >= 15]
    data = []
    for A, B in inputs(orc, shapes, 7):
        A[:8, :16], B[:16, :8] = special_matrix(rng, *A[:8, :16].shape), special_matrix(rng, *B[:16, :8].shape)
        A[0, :], B[-1, -1] = np.inf, np.nan
        data.append((A, B))
    g = oz.GroupScheme2(ex, shapes)
    for (A, B), (M, N, K, S), C in zip(data, shapes, run_group(ex, g, shapes, data, False)):
        assert same_bits(C, single(ex, A, B, S)), (M, N, K, S)
    g.free()
