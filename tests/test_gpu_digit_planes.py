"""The bytes of Scheme II's C_tc as the headers document them: S planes of C_s mod m_s, Mp x Np each, in
32 x 32 element blocks, whatever route the call took (tile sizes, parts along K, row bands, the stage entry
points), read and written here without the library's own unpacking."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu


def up(x, r):
    return -(-x // r) * r


def block_index(M, N):
    """Byte offset of element (row, col) in a plane: block (row / 32, col / 32), inside it 16 bytes per lane of the
    MFMA output layout."""
    row, col = np.meshgrid(np.arange(M), np.arange(N), indexing="ij")
    r = row % 32
    lane = 32 * ((r >> 2) & 1) + col % 32
    return ((row // 32) * (up(N, 256) // 32) + col // 32) * 1024 + lane * 16 + 4 * (r >> 3) + (r & 3)


def planes(raw, M, N, S):
    return raw[:S * up(M, 256) * up(N, 256)].reshape(S, -1)[:, block_index(M, N)]


def download(ex, buf, nbytes):
    return buf.download((nbytes,), np.uint8)


# 64, 128 and 256 wide tiles; all items in parts; the last round of them in parts; the four-slot ring; two row bands
@pytest.mark.parametrize("M,N,K,S,bands", [(70, 50, 300, 9, 0), (400, 390, 200, 14, 0), (300, 290, 20000, 9, 0),
                                           (1025, 1100, 300, 16, 0), (64, 3000, 6000, 13, 0), (600, 700, 500, 20, 2)])
def test_call_leaves_residues(ex, orc, M, N, K, S, bands):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 41)
    ws = oz.WorkspaceScheme2(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    ex.set_bands(bands)
    try:
        oz.ozaki_scheme2_gemm(ws, dA, dB, dC)
        ex.synchronize()
    finally:
        ex.set_bands(0)
    got = planes(download(ex, ws.C_tc, S * up(M, 256) * up(N, 256)), M, N, S)
    ap, bp = ws.planar_slices()
    rows, cols = np.unique(np.r_[0:M:17, M - 1]), np.unique(np.r_[0:N:13, N - 1])
    want = orc.crt_digits(orc.s2_products(np.ascontiguousarray(ap[:, rows]), np.ascontiguousarray(bp[:, :, cols])))
    np.testing.assert_array_equal(got[:, rows][:, :, cols], want)


def test_stage_entry_points_exchange_residues(ex, orc, rng):
    """Digits made by step 3 and by oza_pack_digits, and digits blocked here for step 4."""
    import ozablas_amd as oz

    L = oz._lib
    M, N, K, S = 75, 330, 190, 17
    nbytes = S * up(M, 256) * up(N, 256)
    A, B = gen_pair(orc, M, N, K, 1.0, 43)
    ws = oz.WorkspaceScheme2(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    oz.ozaki_scheme2_gemm(ws, dA, dB, dC)
    ap, bp = ws.planar_slices()
    digits = orc.crt_digits(orc.s2_products(ap, bp))
    dg = ex.to_device(np.zeros(nbytes, np.uint8))
    L.check(L.lib.oza_stage3_s2_digits(ex.ctx, M, N, K, S, ws.A_slices.ptr, ws.B_slices.ptr, dg.ptr))
    np.testing.assert_array_equal(planes(download(ex, dg, nbytes), M, N, S), digits)
    planar = ex.to_device(digits)
    L.check(L.lib.oza_pack_digits(ex.ctx, M, N, S, planar.ptr, dg.ptr))
    np.testing.assert_array_equal(planes(download(ex, dg, nbytes), M, N, S), digits)
    residues = np.stack([rng.integers(0, int(m), size=(M, N)) for m in orc.moduli()[:S]]).astype(np.uint8)
    raw = np.zeros((S, nbytes // S), np.uint8)
    raw[:, block_index(M, N)] = residues
    shA, shB = (rng.integers(-60, 60, size=n).astype(np.int32) for n in (M, N))
    dg, sa, sb = ex.to_device(raw), ex.to_device(shA), ex.to_device(shB)
    L.check(L.lib.oza_stage4_s2_digits(ex.ctx, M, N, K, S, dg.ptr, sa.ptr, sb.ptr, dC.ptr))
    want = orc.recon_s2(residues.astype(np.int32), shA, shB)
    np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want.view(np.uint64))
