"""The integer steps of Scheme II's reconstruction (crt_value, ozablas_amd/csrc/recon_core.hpp, with the
constants of crt_host.cpp), transcribed: group sums u_g, the quotient estimate with its ambiguous
fractions, and Y = X - q M, against the definition (X mod M, minus M from floor(M/2) on), with every
intermediate inside the width the device holds it in; and the stored digit of an INT32 product
(stored_digit, oza_device.hpp).  Host only; the device code is checked bit
for bit by the GPU parity tests."""
import random

import pytest


def tables(moduli):
    M = 1
    for m in moduli:
        M *= m
    groups, err = [], 0
    for s0 in range(0, len(moduli), 3):
        ms = moduli[s0:s0 + 3]
        P = 1
        for m in ms:
            P *= m
        E = [P // m for m in ms]
        w = sum(-2 ** 32 * pow(M // m, -1, m) * pow(e, -1, m) * e for m, e in zip(ms, E)) % P
        err += sum((m - 1) * e for m, e in zip(ms, E))
        groups.append((s0, E, w * (M // P), (w << 32) // P))
    err += 2 + (0 if M >> 64 else (1 << 31) // M)
    return M, groups, (1 << 32) - err


def value(c, M, groups, amb, limbs):
    h, cols = 1 << 31, [0] * limbs
    for s0, E, R, F in groups:
        assert all(e < 1 << 16 for e in E) and F < 1 << 32
        u = sum(x * e for x, e in zip(c[s0:], E))
        assert u < 1 << 32
        h += u * F
        cols = [col + u * (R >> (32 * l) & 0xffffffff) for l, col in enumerate(cols)]
    q = h >> 32
    assert h < 1 << 64 and q < 1 << 32
    neg = (1 << 160) - M
    cols = [col + q * (neg >> (32 * l) & 0xffffffff) for l, col in enumerate(cols)]
    assert all(col + (1 << 33) < 1 << 64 for col in cols)
    y = sum(col << (32 * l) for l, col in enumerate(cols)) & ((1 << (32 * limbs)) - 1)
    if y >> (32 * limbs - 1):
        y -= 1 << (32 * limbs)
    assert abs(y) < 0.57 * M + 1
    if (h & 0xffffffff) >= amb and y >= M // 2:
        y -= M
    return y


@pytest.mark.parametrize("S", range(1, 21))
def test_grouped_crt(orc, S):
    moduli = [int(m) for m in orc.moduli()[:S]]
    M, groups, amb = tables(moduli)
    assert amb >= 0.94 * (1 << 32)
    limbs = (M.bit_length() + 1 + 31) // 32
    rng = random.Random(S)
    half = M // 2
    edges = {0, 1, 2, M - 1, M - 2, half, half - 1, half + 1, M // 3, 2 * M // 3}
    xs = [x % M for x in edges] + [rng.randrange(M) for _ in range(400)]
    xs += [rng.randrange(int(0.43 * M), int(0.57 * M) + 1) % M for _ in range(400)]  # the ambiguous fractions
    for x in xs:
        want = x - M if x >= half else x
        assert value([-x * pow(2, -32, m) % m for m in moduli], M, groups, amb, limbs) == want, (S, x)


def test_stored_digit(orc):
    top = 137438 * 125 ** 2  # the largest |C_s| of an accepted K
    rng = random.Random(7)
    for m in (int(m) for m in orc.moduli()):
        minv, bias = pow(m, -1, 1 << 32), -(-2 ** 31 // m) * m
        vs = [0, 1, -1, m, -m, top, -top, top - m, m - top] + [rng.randint(-top, top) for _ in range(3000)]
        for v in vs:
            u = v + bias
            assert 0 <= u < 1 << 32
            assert (u * minv % (1 << 32)) * m >> 32 == -v * pow(2, -32, m) % m, (m, v)
