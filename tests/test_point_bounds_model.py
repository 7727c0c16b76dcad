"""CPU model of the point additions that hand stored points to one another
between the kernels: the bucket loop's (curve29.hpp, curve_g2.hpp), the lane
teams' (zkmetal_amd/csrc/team29.hpp) and the one-lane G2 addition and doubling
(curve_g2.hpp), limb for limb, on single and merged products with the reduction
digits of curve29.hpp (q_m, q_red).

What it pins: the one bound of a stored point (X < 6.5p, Y < 3.5p, ZZ, ZZZ <
2p per component, limbs normalised) holds for what either form stores and is
enough for what either form loads, doubling and cancellation included; no
column passes 64 bits and no limb wraps on the way."""
import random

import pytest

from oracle import bn254 as B
from oracle import bn254_g2 as G2
from test_fq29_model import MASK, P, PINV, PL, R, U64, fq_add, fq_csub, fq_sub, iz2, kpr, limbs, lt, sub_lazy, val

RED = 7
NL = limbs((PINV * P + 1) >> 29)
ZERO = limbs(0)
STORED = (6.5, 3.5, 2, 2)  # the bound of a stored point's X, Y, ZZ, ZZZ


def prod(pairs, k=0, e=None, borrow=1):
    """sum of a b over one or two pairs, / 2^261, - e + k p (k = 0: no
    subtraction): fq_mul(_x2, _x3), fq_mul_sub, fq_mul_add(_sub).  The kernels
    keep a column in one or two accumulators; their sum is this one."""
    for a, b in pairs:
        assert len(pairs) == 1 or all(v < 1 << 29 for v in a)
        assert all(v < 3 << 29 for v in a + b)
    s = sum(val(a) * val(b) for a, b in pairs)
    assert s < P * R // 2
    d = [x - y for x, y in zip(kpr(k, borrow), e)] if k else [0] * 9
    assert all(x >= 0 for x in d), "negative limb of k p - e"
    m, t, acc = [0] * 9, [0] * 9, 0

    def red(j, n):
        return NL[n - 1] if j < RED else PL[n]

    for c in range(17):
        if c >= 9:
            acc += d[c - 9]
            if c - 9 < RED:
                acc += m[c - 9] * red(c - 9, 9)
        for j in range(max(0, c - 8), min(c + 1, 9)):
            acc += sum(a[j] * b[c - j] for a, b in pairs)
            if j < c:
                acc += m[j] * red(j, c - j)
        assert acc < U64, "column overflow"
        if c < 9:
            m[c] = (acc if c < RED else (acc & 0xFFFFFFFF) * PINV) & MASK
            if c >= RED:
                acc += m[c] * PL[0]
                assert acc & MASK == 0 and acc < U64
        else:
            t[c - 9] = acc & MASK
        acc >>= 29
    t[8] = acc + d[8]
    assert t[8] < 1 << 29
    off = k * P - (val(e) if k else 0)
    assert (val(t) - off - s * pow(R, -1, P)) % P == 0
    assert (val(t) - off) * R < s + P * (R + (R >> 29)) + R
    return t


# ---- an element: its components (one for G1, two for G2)

def each(f, *xs):
    return tuple(f(*c) for c in zip(*xs))


def eadd(a, b):
    return each(fq_add, a, b)


def esub(k, a, b):
    return each(lambda x, y: fq_sub(k, x, y), a, b)


def below(a, bound):
    for c in a:
        lt(c, bound)
    return a


def zero(a):
    below(a, 2)
    return all(iz2(c) for c in a)


def team_mul(a, b):
    """TeamFieldG1::mul, TeamFieldG2::mul"""
    if len(a) == 1:
        return (prod([(a[0], b[0])]),)
    z = [x - y for x, y in zip(kpr(10), b[1])]
    assert all(0 <= v < 1 << 30 for v in z)
    return (prod([(a[0], b[0]), (a[1], z)]), prod([(a[0], b[1]), (a[1], b[0])]))


def stored(p):
    for c, bound in zip(p, STORED):
        below(c, bound)
        assert all(v <= MASK for x in c for v in x)
    return p


def team_dbl(a):
    X, Y, ZZ, ZZZ = stored(a)
    U = eadd(Y, Y)
    xx, V = below(team_mul(X, X), 1.75), below(team_mul(U, U), 1.85)
    M = eadd(eadd(xx, xx), xx)
    S, W, ZZ3, MM = team_mul(X, V), team_mul(U, V), team_mul(ZZ, V), team_mul(M, M)
    X3 = below(esub(3, MM, eadd(S, S)), 4.5)
    Y3 = esub(2, team_mul(M, esub(5, S, X3)), team_mul(W, Y))
    return stored((X3, Y3, below(ZZ3, 1.5), below(team_mul(W, ZZZ), 1.5)))


def team_add(a, b):
    stored(a), stored(b)
    U1, S1, U2, S2 = team_mul(a[0], b[2]), team_mul(a[1], b[3]), team_mul(a[2], b[0]), team_mul(a[3], b[1])
    Pp, Rr = esub(2, U2, U1), esub(2, S2, S1)
    d0, d1 = esub(2, U1, U2), esub(2, S1, S2)
    PP, RR, zz, zzz = team_mul(d0, d0), team_mul(d1, d1), team_mul(a[2], b[2]), team_mul(a[3], b[3])
    Q, ZZ3, PPP = team_mul(U1, PP), team_mul(zz, PP), team_mul(Pp, PP)
    T = each(lambda q, c: [2 * x + y for x, y in zip(q, c)], Q, PPP)
    X3 = esub(5, RR, T)
    Y3 = esub(2, team_mul(Rr, esub(7, Q, X3)), team_mul(PPP, S1))
    r = stored((X3, Y3, below(ZZ3, 1.5), below(team_mul(PPP, zzz), 1.5)))
    if zero(PP) or zero(RR) or zero(zz):
        aid, bid = zero(a[2]), zero(b[2])
        if zero(PP) and zero(RR) and not aid and not bid:
            r = team_dbl(a)
        if aid:
            r = b
        if bid:
            r = a
    return r


# ---- G2Arith: one lane per point

def red4(a):
    return fq_csub(2, lt(a, 4) or a)


def red8(a):
    return fq_csub(2, fq_csub(4, lt(a, 8) or a))


def m2(a, b, k=0, e=(None, None), kb=2):
    """mul2m<K, KB>"""
    n = sub_lazy(kb, ZERO, b[1])
    return (prod([(a[0], b[0]), (a[1], n)], k, e[0]), prod([(a[0], b[1]), (a[1], b[0])], k, e[1]))


def mul2(a, b):
    below(a, 2), below(b, 2)
    t0, t1 = prod([(a[0], b[0])]), prod([(a[1], b[1])])
    t2 = prod([(fq_add(*a), fq_add(*b))])
    return (red4(fq_sub(2, t0, t1)), red8(fq_sub(3, t2, fq_add(t0, t1))))


def sqr2(a):
    below(a, 2)
    t = prod([(a[0], a[1])])
    return (prod([(fq_add(*a), fq_sub(2, *a))]), red4(fq_add(t, t)))


def sub2(a, b):
    return each(red4, esub(2, a, b))


def lane_dbl(p):
    """G2Arith::dbl: a stored point, brought below 2p first"""
    stored(p)
    X, Y = each(red8, p[0]), each(red4, p[1])
    U = each(red4, eadd(Y, Y))
    V = sqr2(U)
    W, S = mul2(U, V), mul2(X, V)
    xx = sqr2(X)
    M = each(red8, eadd(eadd(xx, xx), xx))
    X3 = sub2(sub2(sqr2(M), S), S)
    Y3 = sub2(mul2(M, sub2(S, X3)), mul2(W, Y))
    return stored((X3, Y3, mul2(V, p[2]), mul2(W, p[3])))


def lane_add(a, q):
    """G2Arith::add"""
    stored(a), stored(q)
    U1, S1 = m2(a[0], q[2]), m2(a[1], q[3])
    below(U1, 1.2), below(S1, 1.2)
    Pp, Rr = below(m2(q[0], a[2], 2, U1), 3.2), below(m2(q[1], a[3], 2, S1), 3.2)

    def lz(v):
        return [2 * x for x in v]

    PP = (prod([(fq_add(*Pp), sub_lazy(4, *Pp))]), prod([(lz(Pp[0]), Pp[1])]))
    below(PP, 1.3)
    PPP, Q = m2(Pp, PP), m2(U1, PP)
    T = each(lambda u, v: [2 * x + y for x, y in zip(u, v)], Q, PPP)
    below(T, 4)
    X3 = each(red8, (prod([(fq_add(*Rr), sub_lazy(4, *Rr))], 4, T[0], 3), prod([(lz(Rr[0]), Rr[1])], 4, T[1], 3)))
    M2 = m2(S1, PPP)
    Y3 = each(red4, m2(Rr, esub(2, Q, X3), 2, M2, kb=4))
    r = below(X3, 2), below(Y3, 2), below(m2(m2(a[2], q[2]), PP), 2), below(m2(m2(a[3], q[3]), PPP), 2)
    aid, qid = zero(a[2]), zero(q[2])
    if zero(PP) and zero(each(red4, Rr)) and not aid and not qid:
        r = lane_dbl(a)
    if aid:
        r = q
    return a if qid else r


# ---- the bucket loop's additions of an affine table point

def run_g1(a, q):
    """Arith::qxyzz_madd_run (its columns in fixed order; the sums are these):
    the new accumulator and whether the two cancelled"""
    X, Y, ZZ, ZZZ = (c[0] for c in stored(a))
    x2, y2 = q[0][0], q[1][0]
    Pp, Rr = prod([(x2, ZZ)], 7, X), prod([(y2, ZZZ)], 5, Y)
    lt(Pp, 8.5), lt(Rr, 6.5)
    PP, RR = prod([(Pp, Pp)]), prod([(Rr, Rr)])
    lt(PP, 1.6), lt(RR, 1.6)
    PPP, Q = prod([(Pp, PP)]), prod([(X, PP)])
    X3 = fq_sub(5, RR, [2 * x + y for x, y in zip(Q, PPP)])
    Y3 = prod([(Rr, sub_lazy(7, Q, X3)), (Y, sub_lazy(2, ZERO, PPP))])
    r = stored(((X3,), (Y3,), (prod([(ZZ, PP)]),), (prod([(ZZZ, PPP)]),)))
    assert iz2(PP) == (PP[0] in (0, PL[0]) and iz2(PP))  # the one-limb screen misses none
    cancel = False
    if iz2(PP):
        cancel = not iz2(RR)
        if not cancel:
            r = team_dbl((q[0], q[1], (limbs(R % P),), (limbs(R % P),)))
    return r, cancel


def run_g2(a, q):
    """G2Arith::madd_run"""
    for c in a:
        below(c, 2)
    Pp, Rr = below(m2(q[0], a[2], 2, a[0]), 3.1), below(m2(q[1], a[3], 2, a[1]), 3.1)
    PP = (prod([(fq_add(*Pp), sub_lazy(4, *Pp))]), prod([([2 * v for v in Pp[0]], Pp[1])]))
    PPP, Q = below(m2(Pp, PP), 1.1), below(m2(a[0], PP), 1.1)
    T = below(each(lambda u, v: [2 * x + y for x, y in zip(u, v)], Q, PPP), 4)
    X3 = each(red8, (prod([(fq_add(*Rr), sub_lazy(4, *Rr))], 4, T[0], 3),
                     prod([([2 * v for v in Rr[0]], Rr[1])], 4, T[1], 3)))
    Y3 = each(red4, m2(Rr, esub(2, Q, X3), 2, m2(a[1], PPP), kb=4))
    r = tuple(below(c, 2) for c in (X3, Y3, m2(a[2], PP), m2(a[3], PPP)))
    cancel = False
    if zero(PP):
        cancel = not zero(each(red4, Rr))
        if not cancel:
            one = (limbs(R % P), ZERO)
            r = lane_dbl((q[0], q[1], one, one))
    return r, cancel


# ---- points

def xyzz(pt, rnd, g2):
    """a stored point of an affine one: random Z, every component lifted by a
    random multiple of p within its bound"""
    if pt is None:
        return tuple((ZERO,) * (2 if g2 else 1) for _ in range(4))
    if g2:
        z = (rnd.randrange(1, P), rnd.randrange(P))
        zz = G2.mul2(z, z)
        zzz = G2.mul2(zz, z)
        c = (G2.mul2(pt[0], zz), G2.mul2(pt[1], zzz), zz, zzz)
    else:
        z = rnd.randrange(1, P)
        zz, zzz = z * z % P, z * z * z % P
        c = ((pt[0] * zz % P,), (pt[1] * zzz % P,), (zz,), (zzz,))

    def lift(v, bound):
        v = v * R % P
        return limbs(v + P * rnd.randrange(int((bound * P - 1 - v) // P) + 1))

    return tuple(tuple(lift(v, b) for v in comp) for comp, b in zip(c, STORED))


def affine(pt):
    ri = pow(R, -1, P)
    X, Y, ZZ, ZZZ = ([val(c) * ri % P for c in comp] for comp in pt)
    if len(X) == 1:
        return None if ZZ == [0] else (X[0] * pow(ZZ[0], -1, P) % P, Y[0] * pow(ZZZ[0], -1, P) % P)
    if ZZ == [0, 0]:
        return None
    return (G2.mul2(tuple(X), G2.inv2(tuple(ZZ))), G2.mul2(tuple(Y), G2.inv2(tuple(ZZZ))))


def pairs_of(C, rnd, n):
    pts = [C.mul(C.G2 if C is G2 else C.G, rnd.randrange(1, B.R_ORDER)) for _ in range(n)]
    a, b = pts[:2]
    return list(zip(pts, pts[1:])) + [(a, a), (a, C.neg(a)), (a, None), (None, b), (None, None)]


@pytest.mark.parametrize("C", [B, G2], ids=["g1", "g2"])
def test_team_operations_at_the_stored_bound(C):
    rnd = random.Random(41)
    g2 = C is G2
    for a, b in pairs_of(C, rnd, 12):
        A, Bq = xyzz(a, rnd, g2), xyzz(b, rnd, g2)
        s = team_add(A, Bq)
        assert affine(s) == C.add(a, b)
        assert affine(team_dbl(A)) == C.add(a, a)
        # chained on what they store
        assert affine(team_add(s, team_dbl(s))) == C.mul(C.add(a, b), 3)


def test_lane_operations_at_the_stored_bound():
    rnd = random.Random(42)
    for a, b in pairs_of(G2, rnd, 8):
        A, Bq = xyzz(a, rnd, True), xyzz(b, rnd, True)
        s = lane_add(A, Bq)
        assert affine(s) == G2.add(a, b)
        assert affine(lane_dbl(A)) == G2.add(a, a)
        assert affine(team_add(s, A)) == G2.add(G2.add(a, b), a)


def test_lane_additions_of_merged_points():
    """the bucket reduction by lanes on buckets that the merge's teams stored:
    equal ones double, opposite ones cancel, others add"""
    rnd = random.Random(43)
    k = [rnd.randrange(1, B.R_ORDER) for _ in range(6)]
    pts = [G2.mul(G2.G2, x) for x in k]
    for i in range(60):
        a, b = pts[i % 5], pts[i % 5 + 1]
        # the same sum from two buckets' partials
        s, t = (team_add(xyzz(a, rnd, True), xyzz(b, rnd, True)) for _ in range(2))
        want = G2.add(a, b)
        assert affine(lane_add(s, t)) == G2.add(want, want)
        if i < 6:
            u = team_add(xyzz(G2.neg(a), rnd, True), xyzz(G2.neg(b), rnd, True))
            assert affine(lane_add(s, u)) is None
            assert affine(lane_add(lane_add(s, xyzz(a, rnd, True)), t)) == G2.add(G2.add(want, want), a)


@pytest.mark.parametrize("C", [B, G2], ids=["g1", "g2"])
def test_bucket_runs_and_their_merge(C):
    """runs of table points (a repeat, a cancellation), then the merge of two
    runs by a team, and in G2 the lane addition of two such buckets"""
    rnd = random.Random(44)
    g2, step = C is G2, run_g2 if C is G2 else run_g1
    one = (limbs(R % P), ZERO) if g2 else (limbs(R % P),)

    def table(pt):
        return tuple(tuple(limbs(v * R % P) for v in (c if g2 else (c,))) for c in pt)

    def run(pts):
        acc, want = None, None
        for pt in pts:
            q = table(pt)
            if acc is None:
                acc, cancel = (q[0], q[1], one, one), False
            else:
                acc, cancel = step(acc, q)
            want = C.add(want, pt)
            if cancel:
                assert want is None and affine(acc) is None
                acc = None
            else:
                assert affine(acc) == want
        return acc, want

    for _ in range(4):
        pts = [C.mul(C.G2 if g2 else C.G, rnd.randrange(1, B.R_ORDER)) for _ in range(6)]
        a, wa = run([pts[0], pts[0], pts[1], C.neg(C.add(C.add(pts[0], pts[0]), pts[1])), pts[2], pts[3]])
        b, wb = run([pts[4], pts[5], pts[4]])
        s = team_add(a, b)
        assert affine(s) == C.add(wa, wb)
        assert affine(team_add(s, a)) == C.add(C.add(wa, wb), wa)
        if g2:
            assert affine(lane_add(s, team_add(b, a))) == C.mul(C.add(wa, wb), 2)
