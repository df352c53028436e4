"""Calls whose items run in parts along K, each held to its plan on the host: Scheme II with the last round's items or all
of them in parts, equal or with a shorter last one, on two and four slots; Scheme I with groups in parts.  The result
against the oracle, the planes that the call leaves in C_tc against the stage entry points, and workspaces with room
for the partial sums, for the planes only, and for less."""
import numpy as np
import pytest

import plan_lib
from test_gpu_digit_planes import block_index, planes, up
from test_gpu_item_split import sizes
from test_gpu_parity import gen_pair

# (M, N, K, S), parts, items that run whole, a shorter last part, four slots
S2 = [((1024, 1024, 1030, 18), 3, 256, False, False), ((777, 1501, 1003, 14), 2, 256, False, False),
      ((700, 1100, 1700, 19), 5, 256, True, False), ((1500, 900, 3000, 12), 6, 256, False, True),
      ((257, 513, 20000, 1), 32, 0, True, False), ((500, 300, 17000, 3), 19, 0, False, False),
      ((64, 40, 17000, 2), 27, 0, True, False), ((1, 1, 100000, 1), 32, 0, True, False),
      ((700, 600, 9000, 5), 5, 0, True, False), ((200, 130, 20000, 12), 20, 0, True, True),
      ((600, 600, 5000, 13), 2, 0, False, True)]
# (M, N, K, S), INT32 planes
S1 = [((300, 260, 1900, 10), 55), ((100, 90, 5000, 3), 41), ((1, 1, 11000, 2), 44), ((257, 300, 4000, 20), 60),
      ((1025, 1100, 2500, 4), 10), ((1499, 1200, 1801, 8), 12), ((31, 200, 6000, 9), 122)]
CASES = [(2, *c[0]) for c in S2] + [(1, *c[0]) for c in S1]


@pytest.mark.parametrize("case,parts,whole,short,deep", S2)
def test_plans_s2(case, parts, whole, short, deep):
    p = plan_lib.s2(*case)
    assert (p["edge"], p["parts"], p["whole"], p["short"], p["deep"]) == (256, parts, whole, short, deep), p


@pytest.mark.parametrize("case,planes_", S1)
def test_plans_s1(case, planes_):
    p = plan_lib.s1(*case)
    assert (p["edge"], p["planes"]) == (256, planes_), p
    assert planes_ > case[3]


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,M,N,K,S", CASES)
def test_split_calls(ex, orc, scheme, M, N, K, S):
    import ozablas_amd as oz

    L = oz._lib
    A, B = gen_pair(orc, M, N, K, 1.0, 67)
    ws = (oz.WorkspaceScheme2 if scheme == 2 else oz.WorkspaceScheme1)(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    for _ in range(2):  # the second call finds the first one's sums in the planes
        (oz.ozaki_scheme2_gemm if scheme == 2 else oz.ozaki_scheme1_gemm)(ws, dA, dB, dC)
    ex.synchronize()
    got = dC.download((M, N), np.float64)
    rng = np.random.default_rng(K)
    rows, cols = (np.unique(np.r_[0, n - 1, rng.integers(0, n, 6)]) for n in (M, N))
    want = (orc.s2_gemm if scheme == 2 else orc.s1_gemm)(np.ascontiguousarray(A[rows]), np.ascontiguousarray(B[:, cols]), S)
    np.testing.assert_array_equal(got[np.ix_(rows, cols)].view(np.uint64), want.view(np.uint64))
    n = S * up(M, 256) * up(N, 256)
    if scheme == 2:
        left = planes(ws.C_tc.download((n,), np.uint8), M, N, S)
        dg = ex.to_device(np.zeros(n, np.uint8))
        L.check(L.lib.oza_stage3_s2_digits(ex.ctx, M, N, K, S, ws.A_slices.ptr, ws.B_slices.ptr, dg.ptr))
        np.testing.assert_array_equal(left, planes(dg.download((n,), np.uint8), M, N, S))
    else:
        left = ws.C_tc.download((n,), np.int32).reshape(S, -1)[:, block_index(M, N)]
        T = ex.alloc(4 * S * M * N)
        L.check(L.lib.oza_stage3_s1_groups(ex.ctx, M, N, K, S, ws.A_slices.ptr, ws.B_slices.ptr, T.ptr))
        np.testing.assert_array_equal(left, T.download((S, M, N), np.int32))
    small, extra = sizes(scheme, M, N, K, S)
    assert extra > 0
    for nbytes in (small, small + 256, small + extra):
        w = ex.alloc(nbytes)
        dC.upload(np.full((M, N), np.nan))
        oz.gemm(ex, M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, scheme=scheme, slices=S, workspace=w)
        ex.synchronize()
        np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), got.view(np.uint64))
        w.free()
    w = ex.alloc(small - 256)
    with pytest.raises(ValueError):
        oz.gemm(ex, M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, scheme=scheme, slices=S, workspace=w)
    ws.free()
