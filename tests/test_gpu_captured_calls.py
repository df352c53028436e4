"""Single calls captured into a HIP graph and replayed between eager calls on other inputs, one per route:
small tiles, one launch or two for steps 1 and 2, items in parts, the four-slot ring, both schemes."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu

CASES = [(2, 100, 90, 200, 6), (2, 700, 600, 300, 9), (2, 1300, 1290, 300, 11), (2, 60, 50, 5000, 7),
         (2, 300, 290, 20000, 9), (1, 100, 90, 200, 6), (1, 1000, 900, 200, 5), (1, 100, 90, 4200, 6),
         (1, 2100, 2050, 130, 3)]


@pytest.mark.parametrize("scheme,M,N,K,S", CASES)
def test_replays_match_the_oracle(ex, orc, scheme, M, N, K, S):
    import ozablas_amd as oz

    hip = C.CDLL("libamdhip64.so")
    run = oz.ozaki_scheme2_gemm if scheme == 2 else oz.ozaki_scheme1_gemm
    gemm = orc.s2_gemm if scheme == 2 else orc.s1_gemm
    (A1, B1), (A2, B2) = gen_pair(orc, M, N, K, 1.0, 51), gen_pair(orc, M, N, K, 2.0, 52)
    want1, want2 = gemm(A1, B1, S).view(np.uint64), gemm(A2, B2, S).view(np.uint64)
    ws = (oz.WorkspaceScheme2 if scheme == 2 else oz.WorkspaceScheme1)(ex, M, N, K, S)
    d = [ex.to_device(X) for X in (A1, B1, A2, B2)]
    out = ex.alloc(8 * M * N)
    st = C.c_void_p(ex.stream())
    graph, gexec = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(st, 1) == 0  # thread-local capture mode
    run(ws, d[0], d[1], out)
    assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)) == 0
    try:
        for _ in range(3):
            run(ws, d[2], d[3], out)
            ex.synchronize()
            np.testing.assert_array_equal(out.download((M, N), np.float64).view(np.uint64), want2)
            assert hip.hipGraphLaunch(gexec, st) == 0
            ex.synchronize()
            np.testing.assert_array_equal(out.download((M, N), np.float64).view(np.uint64), want1)
    finally:
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)
        ws.free()
