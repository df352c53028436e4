"""Stage times as the headers describe them: they add up, and step2_ms holds steps 1 and 2 where those are one launch."""
import numpy as np
import pytest

from test_gpu_parity import gen_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [1, 2])
@pytest.mark.parametrize("M,N,K,S,together", [(300, 200, 700, 6, True), (100, 90, 3000, 6, True),
                                              (2000, 1900, 2500, 4, True), (3000, 1900, 2500, 4, False),
                                              (600, 500, 5000, 4, False)])
def test_stages(ex, orc, scheme, M, N, K, S, together):
    import ozablas_amd as oz

    A, B = gen_pair(orc, M, N, K, 1.0, 3)
    ws = (oz.WorkspaceScheme1 if scheme == 1 else oz.WorkspaceScheme2)(ex, M, N, K, S)
    dA, dB, dC = ex.to_device(A), ex.to_device(B), ex.alloc(8 * M * N)
    runs = []
    for _ in range(6):
        t = oz.OzaTimings()
        (oz.ozaki_scheme1_gemm if scheme == 1 else oz.ozaki_scheme2_gemm)(ws, dA, dB, dC, t)
        runs.append([t.step1_ms, t.step2_ms, t.step3_ms, t.step4_ms, t.total_ms])
    for r in runs:
        assert min(r) >= 0 and abs(sum(r[:4]) - r[4]) < 1e-2 + 1e-3 * r[4], r
    one, two = (np.median([r[i] for r in runs[1:]]) for i in (0, 1))
    assert two > 0
    # reading the operands at 8 TB/s is the least that step 1 takes by itself
    assert (one < two) if together else one > 8.0 * K * (M + N) / 8e12 * 1e3, runs
    ws.free()
