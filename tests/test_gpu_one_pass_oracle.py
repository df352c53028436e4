"""Shifts and planes that a single call leaves after steps 1 and 2 (one launch or two), against the oracle's own: finite
operands with zero rows and columns, subnormals and huge values, and Scheme II with infinities and NaNs, whose
residues are 0."""
import numpy as np
import pytest

from test_gpu_one_pass import CASES
from test_gpu_parity import gen_pair, special_matrix

pytestmark = pytest.mark.gpu

LONG = [(130, 70, 2049, 12), (65, 300, 3000, 20), (33, 18, 4096, 6), (2000, 40, 2100, 9), (1, 300, 3333, 1)]


def operands(orc, rng, M, N, K):
    A, B = gen_pair(orc, M, N, K, 1.5, 71)
    if M > 3 and N > 3 and K > 4:
        A[:8, :16], B[:16, :8] = special_matrix(rng, *A[:8, :16].shape), special_matrix(rng, *B[:16, :8].shape)
    return A, B


def planes_of_a_call(ex, scheme, A, B, S):
    import ozablas_amd as oz

    M, K = A.shape
    N = B.shape[1]
    ws = (oz.WorkspaceScheme1 if scheme == 1 else oz.WorkspaceScheme2)(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    (oz.ozaki_scheme1_gemm if scheme == 1 else oz.ozaki_scheme2_gemm)(ws, dA, dB, dC)
    ex.synchronize()
    out = (*ws.shifts(), *ws.planar_slices())
    ws.free()
    return out


@pytest.mark.parametrize("scheme", [1, 2])
@pytest.mark.parametrize("M,N,K,S", CASES + LONG)
def test_finite_operands(ex, orc, rng, scheme, M, N, K, S):
    A, B = operands(orc, rng, M, N, K)
    off = orc.kparam(S, K) if scheme == 2 else 0
    wa, wb = orc.row_shifts(A, off), orc.col_shifts(B, off)
    shA, shB, ga, gb = planes_of_a_call(ex, scheme, A, B, S)
    np.testing.assert_array_equal(shA, wa)
    np.testing.assert_array_equal(shB, wb)
    if scheme == 2:
        want = orc.slice_s2(A, wa, S, True), orc.slice_s2(B, wb, S, False)
    else:
        want = orc.slice_s1(A, wa, S, orc.beta(K), True), orc.slice_s1(B, wb, S, orc.beta(K), False)
    np.testing.assert_array_equal(ga, want[0])
    np.testing.assert_array_equal(gb, want[1])


@pytest.mark.parametrize("M,N,K,S", [c for c in CASES + LONG if min(c[:2]) > 3])
def test_non_finite_values_have_residue_zero(ex, orc, rng, M, N, K, S):
    A, B = operands(orc, rng, M, N, K)
    A[2, 3], A[3, K - 1], B[K - 1, 2], B[4, 3], A[0, :], B[:, 1] = np.inf, np.nan, -np.inf, np.nan, -np.inf, np.nan
    off = orc.kparam(S, K)
    wa, wb = orc.row_shifts(A, off), orc.col_shifts(B, off)
    shA, shB, ga, gb = planes_of_a_call(ex, 2, A, B, S)
    np.testing.assert_array_equal(shA, wa)
    np.testing.assert_array_equal(shB, wb)
    zero = [np.where(np.isfinite(X), X, 0.0) for X in (A, B)]
    np.testing.assert_array_equal(ga, orc.slice_s2(zero[0], wa, S, True))
    np.testing.assert_array_equal(gb, orc.slice_s2(zero[1], wb, S, False))
