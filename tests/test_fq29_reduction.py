"""CPU model of the 29-bit Montgomery reduction whose first seven steps take a
multiple of m that is -1 mod 2^29 (zkmetal_amd/csrc/field29.hpp n(i),
curve29.hpp q_m / q_red): the constants, the value mod m, the bound
ab / 2^261 + (1 + 2^-29) m, and no column past 64 bits at the largest limbs
the products take."""
import os
import random
import re

import pytest

from oracle import bn254 as B

MASK = (1 << 29) - 1
R = 1 << 261
RED = 7
SRC = os.path.join(os.path.dirname(__file__), "..", "zkmetal_amd", "csrc", "field29.hpp")


def limbs(x):
    return [(x >> (29 * i)) & MASK for i in range(9)]


def val(a):
    return sum(v << (29 * i) for i, v in enumerate(a))


def consts(name):
    body = open(SRC).read().split("struct %s {" % name, 1)[1].split("\n};", 1)[0]
    pinv = int(re.search(r"kPinv = (0x[0-9a-f]+)u", body).group(1), 16)

    def table(fn):
        sw = body.split("uint32_t %s(int i) {" % fn, 1)[1].split("default: return", 1)
        cases = re.findall(r"case (\d): return (0x[0-9a-f]+)u", sw[0])
        return [int(v, 16) for _, v in sorted(cases)] + [int(re.match(r"\s*(0x[0-9a-f]+)u", sw[1]).group(1), 16)]

    return pinv, table("p"), table("n")


def product(a, b, pinv, P, N):
    m, t, acc = [0] * 9, [0] * 9, 0

    def red(j, d):
        return N[d - 1] if j < RED else P[d]

    for k in range(9):
        for j in range(k):
            acc += a[j] * b[k - j] + m[j] * red(j, k - j)
        acc += a[k] * b[0]
        assert acc < 1 << 64
        m[k] = (acc if k < RED else (acc & 0xFFFFFFFF) * pinv) & MASK
        if k >= RED:
            acc += m[k] * P[0]
            assert acc & MASK == 0 and acc < 1 << 64
        acc >>= 29
    for k in range(9, 17):
        if k - 9 < RED:
            acc += m[k - 9] * red(k - 9, 9)
        for j in range(k - 8, 9):
            acc += a[j] * b[k - j] + m[j] * red(j, k - j)
        assert acc < 1 << 64
        t[k - 9] = acc & MASK
        acc >>= 29
    t[8] = acc
    assert acc < 1 << 32
    return t


@pytest.mark.parametrize("name,mod", [("Bn254Fp", B.P), ("Bn254Fr", B.R_ORDER)])
def test_reduction_with_the_multiple(name, mod):
    pinv, P, N = consts(name)
    assert val(P) == mod and pinv == (-pow(mod, -1, 1 << 29)) % (1 << 29)
    assert val(N) << 29 == pinv * mod + 1
    rnd = random.Random(29)
    top = limbs(8 * mod - 1)
    # limbs up to 2^30 (two normalised values added), values up to 8.5 m
    wide = [MASK * 2] * 8 + [(17 * mod // 2) >> 232]
    cases = [(limbs(0), top), (top, top), (limbs(1), limbs(1)), (wide, limbs(8 * mod)), (limbs(mod), limbs(mod))]
    cases += [(limbs(rnd.randrange(17 * mod // 2)), limbs(rnd.randrange(8 * mod))) for _ in range(3000)]
    for a, b in cases:
        r = val(product(a, b, pinv, P, N))
        assert (r * R - val(a) * val(b)) % mod == 0
        assert r * R < val(a) * val(b) + mod * (R + (R >> 29))
