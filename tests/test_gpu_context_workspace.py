"""oza_gemm with the context's own workspace: once it holds a call's planes it stays where it is, so a call whose
partial sums do not fit behind them can still be captured, and graphs captured before stay valid."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu

# a first call, and one whose whole planes fit into its workspace but whose parts' sums do not
CASES = [((2, 167, 486, 2225, 7), (1, 137, 142, 4002, 5)), ((2, 1010, 654, 153, 12), (1, 448, 134, 1583, 8)),
         ((2, 86, 1369, 3173, 6), (2, 1927, 2274, 4227, 2))]


@pytest.mark.parametrize("first,second", CASES)
def test_second_call_is_captured(orc, first, second):
    import ozablas_amd as oz

    hip = C.CDLL("libamdhip64.so")
    with oz.HipExecutor(0) as ex:  # its workspace starts empty
        ops = {}
        for case in (first, second):
            scheme, M, N, K, S = case
            A, B = gen_pair(orc, M, N, K, 1.0, 53)
            dA, dB, dC, own = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N), ex.alloc(8 * M * N)
            w = ex.alloc(oz.gemm_workspace_bytes(scheme, M, N, K, S))

            def call(out, ws=None, c=case, a=dA, b=dB):
                oz.gemm(ex, c[1], c[2], c[3], 1.0, a, c[3], b, c[2], 0.0, out, c[2], scheme=c[0], slices=c[4],
                        workspace=ws)

            call(own, w)
            ex.synchronize()
            ops[case] = (call, dC, own.download((M, N), np.float64).view(np.uint64), (dA, dB, own, w))
        st = C.c_void_p(ex.stream())
        graphs = []
        ops[first][0](ops[first][1])  # the workspace is allocated here
        ex.synchronize()
        try:
            for case in (first, second):
                graph, gexec = C.c_void_p(), C.c_void_p()
                assert hip.hipStreamBeginCapture(st, 1) == 0  # thread-local capture mode
                try:
                    ops[case][0](ops[case][1])
                finally:
                    ended = hip.hipStreamEndCapture(st, C.byref(graph))
                assert ended == 0
                assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, C.c_size_t(0)) == 0
                graphs.append((case, graph, gexec))
            for _ in range(3):
                for case, _, gexec in graphs:
                    _, out, want, _ = ops[case]
                    out.upload(np.full(want.shape, np.nan))
                    assert hip.hipGraphLaunch(gexec, st) == 0
                    ex.synchronize()
                    np.testing.assert_array_equal(out.download(want.shape, np.float64).view(np.uint64), want)
                ops[second][0](ops[second][1])  # eager, between the replays
                ex.synchronize()
        finally:
            for _, graph, gexec in graphs:
                hip.hipGraphExecDestroy(gexec)
                hip.hipGraphDestroy(graph)
