"""Workgroups of one item on the CPU model of the LDS ring: with Q slots an item may be shorter than the ring
when no other follows (chain_start_deep repeats its last stage, ozablas_amd/csrc/igemm_core.hpp)."""
import pytest

from test_ring_model import WAVES, check


def single(nit, Q, ksteps, idle=False):
    last = nit - 1
    ops = [("dma", i, (0, min(i, last))) for i in range(Q)]
    ops += [("vmw", Q - 1), ("lgw",), ("bar",), ("rd", 0, (0, 0))]
    refetch = 0
    for it in range(last):
        own = it + Q < nit
        ops += [("rd", it % Q, (0, it))] * (ksteps - 1)
        ops += [("vmw", Q - 2), ("lgw",), ("bar",), ("rd", (it + 1) % Q, (0, it + 1))]
        ops.append(("dma", it % Q, (0, it + Q) if own else (0, refetch)))
        refetch += not own
    assert refetch <= last  # never past the item's last stage
    ops += [("rd", last % Q, (0, last))] * (ksteps - 1)
    ops += [("lgw",), ("bar",), ("dma", last % Q, (0, refetch)), ("vmw", 0)]
    return [op for op in ops if op[0] not in ("rd", "lgw")] if idle else ops


@pytest.mark.parametrize("Q", [4, 8])
def test_single_items_of_any_length(Q):
    for nit in range(1, 3 * Q):
        full = single(nit, Q, 4)
        assert not check([full] * WAVES), nit
        assert not check([full] * (WAVES - 1) + [single(nit, Q, 4, idle=True)]), nit
