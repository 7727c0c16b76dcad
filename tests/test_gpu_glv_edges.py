"""The decomposition's truncated products where a carry from the part left out
could reach the quotient, and the digits' extremes, against the oracle."""
import random

import pytest

import zkmetal_amd as zk
from helpers import result_affine
from oracle import bn254 as B
from oracle import ref

pytestmark = pytest.mark.gpu

G1 = 0x24CCEF014A773D2CF7A7BD9D4391EB18D  # the rounding constants of the split
G2 = 0x2D91D232EC7E0B3D7


def fe(x):
    return x.to_bytes(32, "little")


def _edges():
    rnd = random.Random(5)
    ks = []
    for g in (G1, G2):
        top = (B.R_ORDER * g) >> 256
        for m in [1, 2, top] + [rnd.randrange(1, top) for _ in range(300)]:
            k = ((m << 256) - 1) // g  # k g just below m 2^256, k + 1 just above
            ks += [k, k + 1]
    return [k for k in ks if k < B.R_ORDER]


@pytest.fixture(scope="module")
def engine():
    e = zk.MetalMSM()
    yield e
    e.close()


def test_split_at_quotient_edges(engine):
    ks = _edges()
    out = engine.test_glv(b"".join(fe(k) for k in ks))
    for i, k in enumerate(ks):
        rec = bytes(out[48 * i:48 * i + 48])
        got = (int.from_bytes(rec[:16], "little"), int.from_bytes(rec[16:32], "little"),
               bool(int.from_bytes(rec[32:36], "little")), bool(int.from_bytes(rec[36:40], "little")))
        assert got == B.glv_decompose(k), hex(k)


@pytest.mark.parametrize("c", [2, 7, 8, 11, 13, 16])
def test_digits_at_their_extremes(engine, c):
    # halves whose windows are all half, all half + 1, all ones, alternating
    half = 1 << (c - 1)
    pats = []
    for d in (half, half + 1, half - 1, (1 << c) - 1, 1):
        x = sum(d << (c * w) for w in range(128 // c + 1))
        pats += [x % 2**126, (x << c) % 2**126, x % 2**64]
    ks = [(u + v * B.LAMBDA) % B.R_ORDER for u in pats for v in pats] + _edges()[:200]
    n = len(ks)
    sc = b"".join(fe(k) for k in ks)
    engine.srs_generate(11, n)
    engine.set_window_bits(c)
    try:
        got = result_affine(engine.msm_batch_resident(sc, [n])[0])
    finally:
        engine.set_window_bits(0)
    assert got == B.mul(B.G, ref.scalar_dot(sc, zk.gen_scalars(11, n, 0).tobytes(), n))
