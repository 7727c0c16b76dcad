"""GPU unit tests of the lane-team point arithmetic of the merge, reduction
and tail kernels (team29.hpp) against the affine group law: additions with
random Z, identities, doubling and cancellation mixed in one wave, on BN254
G1, Grumpkin and BN254 G2."""
import random

import pytest

from oracle import bn254 as B
from oracle import bn254_g2 as G2
from oracle import grumpkin as GK
import test_gpu_g2 as g2t

pytestmark = pytest.mark.gpu


def _cases(pts, neg):
    out = [(pts[i], pts[i + 1]) for i in range(len(pts) - 1)]
    P = pts[0]
    # the exceptions between ordinary additions: a wave's branches diverge
    special = [(P, P), (P, neg(P)), (P, None), (None, P), (None, None), (pts[1], pts[1])]
    for k, c in enumerate(special):
        out.insert(3 * k + 1, c)
    return out


@pytest.mark.parametrize("n", [1, 37])
@pytest.mark.parametrize("curve", ["bn254", "grumpkin"])
def test_g1_add_dbl(engine, curve, n):
    C, p, order, op = (B, B.P, B.R_ORDER, 9) if curve == "bn254" else (GK, B.R_ORDER, B.P, 11)
    rnd = random.Random(71)
    pts = [C.mul(C.G, rnd.randrange(1, order)) for _ in range(24)]
    cases = _cases(pts, C.neg)[-n:] if n == 1 else (_cases(pts, C.neg) * 2)[:n]
    R = 1 << 256

    def enc(pt):
        if pt is None:
            return bytes(128)
        z = rnd.randrange(1, p)
        zz, zzz = z * z % p, z * z * z % p
        return b"".join((v * R % p).to_bytes(32, "little") for v in (pt[0] * zz, pt[1] * zzz, zz, zzz))

    def dec(buf, i):
        X, Y, ZZ, ZZZ = (int.from_bytes(bytes(buf[128 * i + 32 * k:128 * i + 32 * k + 32]), "little") for k in range(4))
        assert max(X, Y, ZZ, ZZZ) < p  # canonical
        # x = X / ZZ: the Montgomery factors cancel
        return None if ZZ == 0 else (X * pow(ZZ, -1, p) % p, Y * pow(ZZZ, -1, p) % p)

    Pb = b"".join(enc(a) for a, _ in cases)
    Qb = b"".join(enc(b) for _, b in cases)
    add, dbl = engine.test_xyzz(op, Pb, Qb), engine.test_xyzz(op + 1, Pb, Qb)
    for i, (a, b) in enumerate(cases):
        assert dec(add, i) == C.add(a, b), i
        assert dec(dbl, i) == C.add(a, a), i


def test_g2_add_dbl(engine):
    rnd = random.Random(72)
    pts = [G2.mul(G2.G2, rnd.randrange(1, 1 << 64)) for _ in range(20)]
    cases = _cases(pts, G2.neg)
    Pb = b"".join(g2t._host_xyzz(a, g2t._rz(rnd)) for a, _ in cases)
    Qb = b"".join(g2t._host_xyzz(b, g2t._rz(rnd)) for _, b in cases)
    add, dbl = engine.test_g2(7, Pb, Qb), engine.test_g2(8, Pb, Qb)
    for i, (a, b) in enumerate(cases):
        assert g2t._xyzz_affine(add, i) == G2.add(a, b), i
        assert g2t._xyzz_affine(dbl, i) == G2.add(a, a), i
