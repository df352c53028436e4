"""The relaxed first wait of mainloop_chain together with the work counters that Scheme I's large calls take their
items from (first_claims, publish_claim, ozablas_amd/csrc/k_igemm.hip), on the CPU model of the LDS ring: thread 0's
atomic and LDS write, the barrier of the publication, and waves with nothing to compute, which keep the loads, waits
and barriers (mainloop_idle)."""
import itertools

import pytest

from test_ring_entry_wait import entry_wait
from test_ring_model import WAVES, chain_start, check


def claimed(items, ksteps, wave, stores, outstanding=1, idle=False):
    ops, base = [], 0
    if wave == 0:
        ops += [("vm", "atomic"), ("vmw", 0)]  # first_claims
    ops += [("vmw", 0), ("lgw",), ("bar",)]
    chain_start(ops, 0, items[0])
    for x, nit in enumerate(items):
        more = x + 1 < len(items)
        body = []
        entry_wait(body, x, nit, base, (x + 1, items[x + 1]) if more else None, ksteps, outstanding)
        if idle:
            body = [op for op in body if op[0] not in ("rd", "lgw")]
        ops += body
        if not idle:
            if more and wave == 0:
                ops.append(("vm", "atomic"))
            ops += [("vm", "store")] * stores
        if more:  # publish_claim: only thread 0's wave waits for its ticket
            if wave == 0:
                ops.append(("vmw", stores))  # the ticket is older than the stores
            ops += [("lgw",), ("bar",)]
        base = (base + nit) & 1
    ops.append(("vmw", 0))
    return ops


@pytest.mark.parametrize("ksteps", [2, 4])
@pytest.mark.parametrize("stores", [0, 1, 8])
@pytest.mark.parametrize("idle", [False, True])
def test_claims_keep_the_ring_protocol(ksteps, stores, idle):
    for n in range(1, 5):
        for items in itertools.product((1, 2, 3, 4), repeat=n):
            waves = [claimed(items, ksteps, w, stores, idle=idle and w == WAVES - 1) for w in range(WAVES)]
            bad = check(waves)
            assert not bad, f"items {items}: {bad[:3]}"


def test_one_more_outstanding_operation_is_caught():
    """Planted on the CPU: two stages' loads outstanding at the entry."""
    assert check([claimed((2, 3), 4, w, 0, outstanding=2) for w in range(WAVES)])
