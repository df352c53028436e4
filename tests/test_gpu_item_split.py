"""Tiles whose products run in several parts along K (ozablas_amd/csrc/plan_host.cpp): Scheme II with the
last items or all of them in parts, Scheme I with groups in parts; results and the planes left in the
workspace against the oracle and the reference-layout stage entry points, and workspaces that hold the
planes but not the partial sums."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

# fewer items than CUs; a round and a tail of it; K of one stage more or less than a part; S = 1 and 20
CASES = [(2, 256, 256, 640, 4), (2, 300, 70, 4097, 20), (2, 1024, 1024, 1030, 18), (2, 1300, 1290, 1100, 11),
         (2, 257, 513, 20000, 1), (2, 511, 255, 6400, 3), (1, 256, 256, 256, 4), (1, 257, 300, 1200, 20),
         (1, 100, 90, 5000, 1), (1, 512, 700, 640, 7), (1, 1025, 1100, 897, 6), (1, 31, 515, 9000, 9)]


def sizes(scheme, M, N, K, S):
    """Workspace bytes with every item whole, and what the library asks for."""
    import ozablas_amd as oz

    up = lambda x, r: -(-x // r) * r
    b = list(oz.workspace_bytes(scheme, M, N, K, S))
    asked = b[4]
    b[4] = S * up(M, 256) * up(N, 256) * (1 if scheme == 2 else 4)
    return sum(up(x, 256) for x in b), asked - b[4]


@pytest.mark.parametrize("scheme,M,N,K,S", CASES)
def test_workspace_sizes_grow_with_each_size(scheme, M, N, K, S):
    import ozablas_amd as oz

    big = oz.workspace_bytes(scheme, M, N, K, S)
    assert sizes(scheme, M, N, K, S)[1] >= 0
    for m, n, k, s in [(M - 1, N, K, S), (M, N // 2 + 1, K, S), (M, N, K // 3 + 1, S), (M, N, K, max(1, S - 1)),
                       (M // 2 + 1, N // 2 + 1, K, S)]:
        assert all(x <= y for x, y in zip(oz.workspace_bytes(scheme, m, n, k, s), big))


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,M,N,K,S", CASES)
def test_split_calls_match_the_oracle(ex, orc, scheme, M, N, K, S):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 31)
    want = (orc.s2_gemm if scheme == 2 else orc.s1_gemm)(A, B, S).view(np.uint64)
    ws = (oz.WorkspaceScheme2 if scheme == 2 else oz.WorkspaceScheme1)(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    run = oz.ozaki_scheme2_gemm if scheme == 2 else oz.ozaki_scheme1_gemm
    for _ in range(2):  # the second call finds the first one's sums in the planes
        run(ws, dA, dB, dC)
        ex.synchronize()
        np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want)
    if scheme == 2:  # the S digit planes hold the whole products afterwards
        L = oz._lib
        ap, bp = ws.planar_slices()
        pl = ex.alloc(S * M * N)
        L.check(L.lib.oza_unpack_digits(ex.ctx, M, N, S, ws.C_tc.ptr, pl.ptr))
        np.testing.assert_array_equal(pl.download((S, M, N), np.uint8), orc.crt_digits(orc.s2_products(ap, bp)))
    small, extra = sizes(scheme, M, N, K, S)
    for nbytes in {small, small + extra}:
        w = ex.alloc(nbytes)
        dC.upload(np.full((M, N), np.nan))
        oz.gemm(ex, M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, scheme=scheme, slices=S, workspace=w)
        ex.synchronize()
        np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want)
    w = ex.alloc(small - 256)
    with pytest.raises(ValueError):
        oz.gemm(ex, M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, scheme=scheme, slices=S, workspace=w)
