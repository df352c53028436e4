"""Steps 1 and 2 of single calls (one launch for Kp <= 2048, else partial maxima finished by the
slicing kernels) against the separate kernels of the
stage entry points and the oracle: shifts and planes byte for byte, at the edges of its unit, row-block,
word-count and part choices, with non-finite values, and for both orientations of each operand."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair, special_matrix, stage_shifts, stage_slices

pytestmark = pytest.mark.gpu

# K at the edges of the thread counts, of 1 and 2 units per thread and of the path; rows at the edges of 16, 32, 64; many
# and few row blocks (parts 1, 2, 4, 8); S at the edges of one, two and three words per value
CASES = [(1, 1, 1, 20), (15, 17, 128, 1), (16, 33, 129, 3), (31, 64, 256, 5), (65, 48, 257, 8), (100, 63, 384, 20),
         (63, 129, 512, 10), (64, 1, 513, 17), (250, 31, 1000, 16), (33, 260, 1024, 18), (1700, 2500, 700, 9),
         (40, 50, 1025, 12), (200, 8000, 900, 4), (1024, 33, 5001, 9), (1100, 1023, 2049, 6), (70, 1023, 1300, 6), (33, 40, 2048, 19), (130, 47, 1025, 2), (3, 70, 40000, 7)]


@pytest.mark.parametrize("scheme", [1, 2])
@pytest.mark.parametrize("M,N,K,S", CASES)
def test_planes_match_separate_steps(ex, orc, rng, scheme, M, N, K, S):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.5, 21)
    if M > 3 and N > 3 and K > 4:
        A[:8, :16], B[:16, :8] = special_matrix(rng, *A[:8, :16].shape), special_matrix(rng, *B[:16, :8].shape)
        A[2, 3], A[3, K - 1], B[K - 1, 2], B[4, 3], A[0, :] = np.inf, np.nan, -np.inf, np.nan, -np.inf
    ws = (oz.WorkspaceScheme1 if scheme == 1 else oz.WorkspaceScheme2)(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    (oz.ozaki_scheme1_gemm if scheme == 1 else oz.ozaki_scheme2_gemm)(ws, dA, dB, dC)
    ex.synchronize()
    shA, shB = stage_shifts(ex, scheme, A, B, S)
    for got, want in zip(ws.shifts(), (shA, shB)):
        np.testing.assert_array_equal(got, want)
    ap, bp, _, _ = stage_slices(ex, scheme, A, B, S, shA, shB)
    ga, gb = ws.planar_slices()
    np.testing.assert_array_equal(ga, ap)
    np.testing.assert_array_equal(gb, bp)
    off = orc.kparam(S, K) if scheme == 2 else 0
    np.testing.assert_array_equal(shA, orc.row_shifts(A, off))
    if scheme == 2 and np.isfinite(A).all():
        np.testing.assert_array_equal(ga, orc.slice_s2(A, shA, S, True))
        np.testing.assert_array_equal(gb, orc.slice_s2(B, shB, S, False))


@pytest.mark.parametrize("scheme,S", [(2, 15), (1, 6)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_orientations(ex, orc, scheme, S, ta, tb):
    """Row-contiguous and K-contiguous storage of either operand, odd leading dimensions."""
    import ozablas_amd as oz

    M, N, K = 70, 45, 601
    A, B = gen_pair(orc, M, N, K, 1.0, 5)

    def stored(X, t):
        Y = X.T if t else X
        out = np.zeros((Y.shape[0], Y.shape[1] + 3))
        out[:, :Y.shape[1]] = Y
        return out

    sA, sB = stored(A, ta), stored(B, tb)
    dA, dB, dC = ex.to_device(sA), ex.to_device(sB), ex.alloc(8 * M * N)
    oz.gemm(ex, M, N, K, 1.0, dA, sA.shape[1], dB, sB.shape[1], 0.0, dC, N, transA=ta, transB=tb, scheme=scheme, slices=S)
    ex.synchronize()
    want = orc.s2_gemm(A, B, S) if scheme == 2 else orc.s1_gemm(A, B, S)
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
