"""Rings of more than two slots (mainloop_chain with STAGES = Q, ozablas_amd/csrc/igemm_core.hpp) on the CPU
model of the LDS ring: Q stages of an item are issued before it starts, stage i + Q (its own, or the next
item's) when stage i has been read, and a wait leaves the Q - 2 later stages outstanding.  One load per
stage here stands for the LPS loads of a wave.  Items have at least Q stages."""
import itertools

import pytest

from test_ring_model import WAVES, check


def workgroup(items, Q, ksteps, stores, idle=False, slack=0):
    ops, base = [], 0
    ops += [("dma", i, (0, i)) for i in range(Q)]  # chain_start_deep
    for x, nit in enumerate(items):
        more = x + 1 < len(items)

        def slot(i):
            return (base + i) % Q

        def src(i):  # past the last item: its stages again, read by nobody
            return (x, i) if i < nit else (x + 1 if more else x, i - nit)

        ops += [("vmw", Q - 1), ("lgw",), ("bar",), ("rd", slot(0), (x, 0))]
        for it in range(nit - 1):
            ops += [("rd", slot(it), (x, it))] * (ksteps - 1)
            ops += [("vmw", Q - 2 + slack), ("lgw",), ("bar",), ("rd", slot(it + 1), (x, it + 1))]
            ops.append(("dma", slot(it + Q), src(it + Q)))
        ops += [("rd", slot(nit - 1), (x, nit - 1))] * (ksteps - 1)
        ops += [("lgw",), ("bar",), ("dma", slot(nit + Q - 1), src(nit + Q - 1))]
        ops += [("vm", "store")] * stores
        base = (base + nit) % Q
    ops.append(("vmw", 0))
    return [op for op in ops if op[0] not in ("rd", "lgw", "vm")] if idle else ops


@pytest.mark.parametrize("Q,ksteps", [(4, 2), (4, 1), (8, 2)])
@pytest.mark.parametrize("stores", [0, 3])
def test_deep_ring_protocol(Q, ksteps, stores):
    for n in range(1, 4):
        for items in itertools.product(range(Q, Q + 4), repeat=n):
            full = workgroup(items, Q, ksteps, stores)
            assert not check([full] * WAVES), items
            bad = check([full] * (WAVES - 1) + [workgroup(items, Q, ksteps, stores, idle=True)])
            assert not bad, f"items {items}: {bad[:3]}"


def test_one_more_outstanding_stage_is_caught():
    """Planted on the CPU: a stage entered with its own loads outstanding."""
    assert check([workgroup((5, 6), 4, 2, 0, slack=1)] * WAVES)


def test_items_shorter_than_the_ring_are_caught():
    """Why such shapes take the two-slot ring: the stage after next would be the item's after next."""
    assert check([workgroup((3, 5), 4, 2, 0)] * WAVES)
