"""Waves without fragments (mainloop_idle, ozablas_amd/csrc/igemm_core.hpp) on the CPU model of the LDS ring:
they issue their loads and meet the barriers of every item beside waves that compute."""
import itertools

import pytest

from test_ring_entry_wait import workgroup
from test_ring_model import WAVES, check


def idle(ops):
    """A wave's operations without its fragment reads, their waits and its stores."""
    return [op for op in ops if op[0] not in ("rd", "lgw", "vm")]


@pytest.mark.parametrize("stores", [0, 8])
def test_idle_waves_keep_the_ring_protocol(stores):
    for n in range(1, 4):
        for items in itertools.product((1, 2, 3, 4), repeat=n):
            full = workgroup(items, 4, stores)
            for active in range(1, WAVES):
                bad = check([full] * active + [idle(full)] * (WAVES - active))
                assert not bad, f"items {items}, {active} active waves: {bad[:3]}"


def test_a_missing_barrier_is_caught():
    """Planted on the CPU: an idle wave that skips its last barrier."""
    full = workgroup((2, 3), 4, 0)
    short = idle(full)
    del short[max(i for i, op in enumerate(short) if op[0] == "bar")]
    assert check([full] * (WAVES - 1) + [short])
