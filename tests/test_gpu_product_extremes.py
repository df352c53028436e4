"""INT32 products at the ends of their range: the stage entry points take any int32 C_s, and any int8 slices whose
products fit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOP = 2 ** 31 - 1


@pytest.mark.parametrize("S", [1, 2, 5, 8, 13, 20])
def test_step4_takes_any_int32(ex, orc, rng, S):
    import ozablas_amd as oz

    L = oz._lib
    M, N = 40, 40
    Ct = rng.integers(-2 ** 31, 2 ** 31, size=(S, M, N)).astype(np.int32)
    ends = np.r_[np.arange(TOP - 300, TOP + 1), np.arange(-TOP - 1, -TOP + 299)]
    Ct[:, :ends.size // N] = ends[:ends.size // N * N].reshape(-1, N)
    sh = np.zeros(M, np.int32)
    dc, ds, dC = ex.to_device(Ct), ex.to_device(sh), ex.alloc(8 * M * N)
    L.check(L.lib.oza_stage4_s2_products(ex.ctx, M, N, 1, S, dc.ptr, ds.ptr, ds.ptr, dC.ptr))
    want = orc.recon_s2(Ct, sh, sh)
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))


def test_step3_digits_of_the_largest_product(ex, orc):
    """133145 products of slices of at most 127 that add up to 2^31 - 1, and to its negative."""
    import ozablas_amd as oz

    L = oz._lib
    M = N = 2
    K, S = 133145, 3
    a, b = np.full(K, 127, np.int8), np.full(K, 127, np.int8)
    a[-1], b[-1] = 59, 69
    A8 = np.broadcast_to(np.stack([a, -a]), (S, M, K))
    B8 = np.broadcast_to(np.stack([b, b], axis=1), (S, K, N))
    C = orc.s2_products(np.ascontiguousarray(A8), np.ascontiguousarray(B8))
    assert C.max() == TOP and C.min() == -TOP
    Kp = -(-K // 128) * 128

    def tiled(rows):  # [S][rows][K] -> the fragment-tiled planes of the first 32-row block
        X = np.zeros((S, 32, Kp), np.int8)
        X[:, :rows.shape[1], :K] = rows
        X = X.reshape(S, 32, Kp // 32, 2, 16).transpose(0, 2, 3, 1, 4)  # [S][k block][half][row][16]
        out = np.zeros((S, 256 * Kp), np.int8)
        out[:, :32 * Kp] = X.reshape(S, -1)
        return out

    dA, dB = ex.to_device(tiled(A8)), ex.to_device(tiled(B8.transpose(0, 2, 1)))
    dg, pl = ex.to_device(np.zeros(S * 65536, np.uint8)), ex.alloc(S * M * N)
    L.check(L.lib.oza_stage3_s2_digits(ex.ctx, M, N, K, S, dA.ptr, dB.ptr, dg.ptr))
    L.check(L.lib.oza_unpack_digits(ex.ctx, M, N, S, dg.ptr, pl.ptr))
    np.testing.assert_array_equal(pl.download((S, M, N), np.uint8), orc.crt_digits(C))
