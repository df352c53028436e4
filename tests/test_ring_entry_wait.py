"""The relaxed first wait of mainloop_chain (ozablas_amd/csrc/igemm_core.hpp) on the CPU model of the LDS ring
(test_ring_model): an item with at least two stages enters when at most one stage's loads are
outstanding -- stage 1's, or the previous item's stores -- instead of none, and reads its first
fragments before it issues anything.  One load per stage here stands for the LPS loads of a wave."""
import itertools

import pytest

from test_ring_model import WAVES, check, chain_start, mainloop_chain


def entry_wait(ops, x, nit, base, nxt, ksteps, outstanding=1):
    body = []
    mainloop_chain(body, x, nit, base, nxt, ksteps)
    assert body[0] == ("vmw", 0)
    body[0] = ("vmw", outstanding if nit >= 2 else 0)
    if nit == 1:  # the first fragment read comes before the issue of chain stage 1
        assert body[3][0] == "dma" and body[4][0] == "rd"
        body[3], body[4] = body[4], body[3]
    ops += body


def workgroup(items, ksteps, stores, outstanding=1):
    ops, base = [], 0
    chain_start(ops, 0, items[0])
    for x, nit in enumerate(items):
        nxt = (x + 1, items[x + 1]) if x + 1 < len(items) else None
        entry_wait(ops, x, nit, base, nxt, ksteps, outstanding)
        ops += [("vm", "store")] * stores
        base = (base + nit) & 1
    ops.append(("vmw", 0))
    return ops


@pytest.mark.parametrize("ksteps", [2, 4])
@pytest.mark.parametrize("stores", [0, 1, 8])
def test_relaxed_entry_keeps_the_ring_protocol(ksteps, stores):
    for n in range(1, 5):
        for items in itertools.product((1, 2, 3, 4), repeat=n):
            bad = check([workgroup(items, ksteps, stores)] * WAVES)
            assert not bad, f"items {items}: {bad[:3]}"


def test_one_more_outstanding_operation_is_caught():
    """Planted on the CPU: two stages' loads outstanding at the entry leave stage 0 unread-able."""
    bad = check([workgroup((2, 3), 4, 0, outstanding=2)] * WAVES)
    assert any(b.startswith(("R1", "R2")) for b in bad)
