"""Scheme II on the four-slot ring with several items per workgroup (the hand-over of the ring from one item to the
next), unsplit, with the last round in parts and with every item in parts, and neighbours on the other side of the rule's
lines; each case is held to its route on the host.  All of C against the grouped GEMM's 128 wide tiles, which have
two slots, and rows and columns of it, with the full K, against the oracle."""
import numpy as np
import pytest

import plan_lib
from test_gpu_parity import gen_pair

# (M, N, K, S), four slots, parts, whole items: 480 items of 8, 9 and 6 K steps of 128; 768 whole items; tails in five,
# three and two unequal parts; every item in parts; both sides of the bytes' and of the width's line
CASES = [((20, 6000, 1000, 20), True, 1, 480), ((5900, 33, 1100, 20), True, 1, 480), ((20, 6000, 641, 20), True, 1, 480),
         ((20, 6000, 640, 20), False, 1, 480), ((300, 8000, 2048, 12), True, 1, 768), ((3000, 1000, 2050, 16), True, 1, 768),
         ((20, 3800, 4200, 20), True, 5, 256), ((300, 4600, 6000, 9), True, 3, 256), ((1024, 1000, 9000, 10), True, 3, 0),
         ((1600, 1600, 1200, 20), True, 1, 980), ((1601, 1601, 1200, 20), False, 1, 980)]


@pytest.mark.parametrize("case,deep,parts,whole", CASES)
def test_routes(case, deep, parts, whole):
    p = plan_lib.s2(*case)
    assert (p["edge"], p["deep"], p["parts"], p["whole"]) == (256, deep, parts, whole), p
    assert p["items"] > 256


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", [c[0] for c in CASES])
def test_matches_the_grouped_gemm_and_the_oracle(ex, orc, M, N, K, S):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 61)
    ws = oz.WorkspaceScheme2(ex, M, N, K, S)
    dA, dB, dC, dG = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N), ex.alloc(8 * M * N)
    oz.ozaki_scheme2_gemm(ws, dA, dB, dC)
    g = oz.GroupScheme2(ex, [(M, N, K, S)], tiles=[128], splits=[1])
    g.run([dA], [dB], [dG], use_graph=False)
    ex.synchronize()
    got = dC.download((M, N), np.float64)
    np.testing.assert_array_equal(got.view(np.uint64), dG.download((M, N), np.float64).view(np.uint64))
    rng = np.random.default_rng(K)
    rows = np.unique(np.r_[0, M - 1, rng.integers(0, M, 10)])
    cols = np.unique(np.r_[0, N - 1, rng.integers(0, N, 10)])
    want = orc.s2_gemm(np.ascontiguousarray(A[rows]), np.ascontiguousarray(B[:, cols]), S)
    np.testing.assert_array_equal(got[np.ix_(rows, cols)].view(np.uint64), want.view(np.uint64))
    At, Bt = ex.to_device(np.ascontiguousarray(A.T)), ex.to_device(np.ascontiguousarray(B.T))
    dC.upload(np.ones((M, N)))  # -0.5 * X + 2 * 1 rounded once
    oz.gemm(ex, M, N, K, -0.5, At, M, Bt, K, 2.0, dC, N, transA=oz.OP_T, transB=oz.OP_T, scheme=2, slices=S)
    ex.synchronize()
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), (got * -0.5 + 2.0).view(np.uint64))
    g.free()
    ws.free()
