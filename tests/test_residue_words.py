"""Scheme II's residues from 32-bit words (int_words and sym_residue, ozablas_amd/csrc/oza_device.hpp, with the constants
of make_residue_consts and the word counts of residue_words, slice_core.hpp), transcribed: the symmetric residue of
every integer that a word count is used for, with each intermediate inside its width.  Host only."""
import random

import numpy as np
import pytest


def consts(m):
    p, w = 2 ** 32 % m, []
    for _ in range(13):
        w.append(p)
        p = p * 256 % m
    wt = [[(m - w[4 * n + k]) % m for k in range(4)] for n in range(3)]
    init = [w[4 * n + 3] * 128 % m for n in range(3)]
    assert all(x < 256 for row in wt for x in row)
    return wt, init, pow(m, -1, 2 ** 32)


def int_words(t, nd):
    """t: an integer-valued float64; the device's operations, each exact."""
    out = []
    for _ in range(nd - 1):
        top = np.floor(t * 2.0 ** -32)
        lo = int(t) - int(top) * 2 ** 32  # fma(-top, 2^32, t): exact if it fits 53 bits
        assert 0 <= lo < 2 ** 32 and float(lo) == lo
        out.append(lo)
        t = top
    assert -2 ** 31 <= int(t) < 2 ** 31
    out.append(int(t) % 2 ** 32 ^ 0x80000000)
    return out


def sym_residue(words, wt, init, m, minv):
    d = init
    for n, x in enumerate(words):
        d += sum((x >> 8 * k & 0xff) * wt[n][k] for k in range(4))
    assert d < 2 ** 20
    p = d * minv % 2 ** 32
    p -= p >> 31 << 32  # as a signed number
    return p * m >> 32


def words_for(kparam):
    return 1 if kparam <= 30 else 2 if kparam <= 62 else 3


@pytest.mark.parametrize("nd", [1, 2, 3])
def test_symmetric_residue(orc, nd):
    kparams = [k for k in range(1, 76) if words_for(k) == nd]
    assert max(kparams) == {1: 30, 2: 62, 3: 75}[nd]
    top = 2.0 ** max(kparams)
    rng = random.Random(nd)
    ts = [0.0, 1.0, -1.0, top, -top, np.nextafter(top, 0), -np.nextafter(top, 0)]
    ts += [s * 2.0 ** k for k in range(max(kparams)) for s in (1, -1)] + [s * (2.0 ** k - 1) for k in range(2, 53) for s in (1, -1) if 2.0 ** k <= top]
    ts += [float(round(rng.uniform(-1, 1) * 2.0 ** rng.choice(kparams))) for _ in range(600)]
    for m in (int(m) for m in orc.moduli()):
        wt, init, minv = consts(m)
        near = [float(m * q + r) for q in (0, 1, -1, 5, -7) for r in (-m // 2, m // 2, (m + 1) // 2, 1 - m // 2)]
        for t in ts + near:
            got = sym_residue(int_words(t, nd), wt, init[nd - 1], m, minv)
            want = int(t) % m
            assert got == (want if want <= m // 2 else want - m), (m, t)


def test_largest_kparam_has_its_words(orc):
    for S in range(1, 21):
        for K in (1, 2, 3, 100, 137438):
            assert orc.kparam(S, K) <= 75
