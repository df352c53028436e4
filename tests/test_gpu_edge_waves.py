"""Edge tiles on every single-call GEMM that has waves with half, a quarter or none of their part to compute
(for_part, ozablas_amd/csrc/igemm_core.hpp): whole tiles and one more row and column of tiles of 1 to 256 rows and
columns.  Each case is held to its route on the host; the results beside the edges against the oracle."""
import numpy as np
import pytest

import plan_lib
from test_gpu_parity import gen_pair

E256 = [1, 31, 32, 33, 64, 65, 95, 97, 128, 129, 160, 191, 193, 224, 225, 256]
E128 = [1, 32, 33, 63, 64, 65, 96, 97, 127, 128]
# scheme, rows and columns of whole tiles, K, S, edge rows, what the plan has to be
ROUTES = {"s2_256": (2, 1024, 129, 20, E256, dict(edge=256, parts=1, deep=False)),
          "s2_256_parts": (2, 1024, 1100, 11, E256, dict(edge=256, parts=3, whole=256, deep=False)),
          "s2_256_deep": (2, 768, 2200, 20, E256[::3], dict(edge=256, parts=3, deep=True)),
          "s2_128": (2, 384, 200, 20, E128, dict(edge=128)),
          "s1_256_static": (1, 512, 2200, 6, E256[::2], dict(edge=256, planes=21, dynamic=False)),
          "s1_256_dynamic": (1, 1792, 520, 17, E256[::2], dict(edge=256, planes=17, dynamic=True)),
          "s1_128": (1, 1280, 200, 4, E128, dict(edge=128, planes=4))}
CASES = [(name, r[1] + e, r[1] + r[4][(7 * i + 3) % len(r[4])]) for name, r in ROUTES.items() for i, e in enumerate(r[4])]


@pytest.mark.parametrize("name,M,N", CASES)
def test_routes(name, M, N):
    scheme, _, K, S, _, want = ROUTES[name]
    plan = (plan_lib.s2 if scheme == 2 else plan_lib.s1)(M, N, K, S)
    assert {k: plan[k] for k in want} == want, plan


@pytest.mark.gpu
@pytest.mark.parametrize("name,M,N", CASES)
def test_edges_match_the_oracle(ex, orc, name, M, N):
    import ozablas_amd as oz

    scheme, base, K, S, _, _ = ROUTES[name]
    A, B = gen_pair(orc, M, N, K, 1.0, M + N)
    ws = (oz.WorkspaceScheme2 if scheme == 2 else oz.WorkspaceScheme1)(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    dC.upload(np.full((M, N), np.nan))
    (oz.ozaki_scheme2_gemm if scheme == 2 else oz.ozaki_scheme1_gemm)(ws, dA, dB, dC)
    ex.synchronize()
    got = dC.download((M, N), np.float64)
    gemm = orc.s2_gemm if scheme == 2 else orc.s1_gemm
    rng = np.random.default_rng(M)
    # the last row of tiles by some columns, and some rows by the last column of tiles
    for rows, cols in [(np.arange(base - 2, M), np.unique(np.r_[rng.integers(0, N, 6), base - 1, base, N - 1])),
                       (np.unique(np.r_[rng.integers(0, M, 6), base - 1, base, M - 1]), np.arange(base - 2, N))]:
        want = gemm(np.ascontiguousarray(A[rows]), np.ascontiguousarray(B[:, cols]), S)
        np.testing.assert_array_equal(got[np.ix_(rows, cols)].view(np.uint64), want.view(np.uint64))
    if scheme == 2:
        g = oz.GroupScheme2(ex, [(M, N, K, S)], tile=64)
        g.run([dA], [dB], [dC], use_graph=False)
        ex.synchronize()
        np.testing.assert_array_equal(got.view(np.uint64), dC.download((M, N), np.float64).view(np.uint64))
        g.free()
    assert np.isfinite(got).all()
    ws.free()
