"""oza_scheme1_gemm takes no buffer sizes, so it keeps to the S planes of C_tc that the layout names, also for shapes
that oza_scheme1_gemm_sized (the workspace classes) runs in parts along K: the bytes behind the planes stay as they
were.  oza_scheme1_gemm_sized for a buffer of every size."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

# in parts, one tile and four; 64 and 128 wide tiles, which run whole
CASES = [(31, 200, 6000, 9), (300, 260, 1900, 10), (100, 90, 2100, 5), (760, 1030, 257, 3)]


def up(x, r):
    return -(-x // r) * r


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,S", CASES)
def test_bytes_behind_the_planes(ex, orc, M, N, K, S):
    import ozablas_amd as oz

    L = oz._lib
    A, B = gen_pair(orc, M, N, K, 1.0, 47)
    want = orc.s1_gemm(A, B, S).view(np.uint64)
    ws = oz.WorkspaceScheme1(ex, M, N, K, S)
    planes, extra = 4 * S * up(M, 256) * up(N, 256), 64 << 20
    ctc = ex.alloc(planes + extra)  # more than any plan's partial sums
    assert ws.bytes[4] <= planes + extra
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    ptrs = [b.ptr for b in (ws.shift_A, ws.shift_B, ws.A_slices, ws.B_slices, ctc)]
    head = (ex.ctx, M, N, K, S, dA.ptr, dB.ptr, dC.ptr, *ptrs)
    guard = np.full(planes + extra, 0x5A, np.uint8)

    def check(call, behind):
        ctc.upload(guard)
        dC.upload(np.full((M, N), np.nan))
        L.check(call())
        ex.synchronize()
        np.testing.assert_array_equal(dC.download((M, N), np.float64).view(np.uint64), want)
        assert (ctc.download((planes + extra,), np.uint8)[behind:] == 0x5A).all()

    check(lambda: L.lib.oza_scheme1_gemm(*head, None), planes)
    for size in (planes, planes + 4, ws.bytes[4]):
        check(lambda: L.lib.oza_scheme1_gemm_sized(*head, size, None), max(planes, size))
    assert L.lib.oza_scheme1_gemm_sized(*head, planes - 1, None) == oz._lib.INVALID_ARGUMENT


def test_arguments_are_checked_before_anything_else():
    import ozablas_amd as oz

    L = oz._lib
    assert L.lib.oza_scheme1_gemm_sized(None, 8, 8, 8, 4, *[None] * 8, 1 << 20, None) == L.INVALID_ARGUMENT
