"""product_digit (ozablas_amd/csrc/oza_device.hpp) and the byte weights of crt_host.cpp, transcribed: the digit of an
INT32 product is its plain residue, with every intermediate inside 32 bits; and the grouped CRT of test_crt_groups
with multipliers for plain residues, whose constants have the same bounds.  Host only."""
import random

import pytest

from test_crt_groups import tables, value


def digit(v, m):
    minv, p, d = pow(m, -1, 1 << 32), (1 << 32) % m, (1 << 63) % m
    u = v + 2 ** 31
    assert 0 <= u < 1 << 32
    for k in range(4):
        wt = (m - p) % m
        assert wt < 256
        d += (u >> (8 * k) & 0xff) * wt
        p = p * 256 % m
    assert d < (1 << 18) + 256
    return (d * minv % (1 << 32)) * m >> 32


def test_product_digit(orc):
    top = 2 ** 31 - 1
    rng = random.Random(7)
    for m in (int(m) for m in orc.moduli()):
        vs = [0, 1, -1, m, -m] + [e + k for e in (top, -top) for k in range(-300, 301)] + [-2 ** 31] + [rng.randint(-top, top) for _ in range(3000)]
        for v in vs:
            assert not -2 ** 31 <= v < 2 ** 31 or digit(v, m) == v % m, (m, v)


@pytest.mark.parametrize("S", range(1, 21))
def test_grouped_crt_of_plain_residues(orc, S):
    moduli = [int(m) for m in orc.moduli()[:S]]
    M, groups, amb = tables(moduli)
    plain = []
    for s0, E, _, _ in groups:
        ms = moduli[s0:s0 + 3]
        P = E[0] * ms[0]
        w = sum(pow(M // m, -1, m) * pow(e, -1, m) * e for m, e in zip(ms, E)) % P
        plain.append((s0, E, w * (M // P), (w << 32) // P))
    limbs = (M.bit_length() + 1 + 31) // 32
    rng = random.Random(S)
    half = M // 2
    xs = [x % M for x in (0, 1, 2, M - 1, M - 2, half, half - 1, half + 1, M // 3, 2 * M // 3)]
    xs += [rng.randrange(M) for _ in range(400)]
    xs += [rng.randrange(int(0.43 * M), int(0.57 * M) + 1) % M for _ in range(400)]  # the ambiguous fractions
    for x in xs:
        assert value([x % m for m in moduli], M, plain, amb, limbs) == (x - M if x >= half else x), (S, x)
