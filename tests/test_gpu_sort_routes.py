"""The sort's routes at their edges against the closed form: a segment just
within and just past the one-block sort (16384 entries, 4096 buckets), and
segments on either side of the one-block histogram scan (128 tiles)."""
import pytest

import zkmetal_amd as zk
from helpers import result_affine
from oracle import bn254 as B
from oracle import ref

pytestmark = pytest.mark.gpu

SEED = 0x50B7


@pytest.fixture(scope="module")
def eng():
    e = zk.MetalMSM()
    e.set_window_shift(e.SHIFT_OFF)
    e.srs_generate(SEED, (1 << 18) + 1)
    yield e
    e.close()


def _check(eng, n, dist):
    sc = zk.gen_scalars(SEED + n, n, dist)
    got = result_affine(eng.msm_batch_resident(sc, [n])[0])
    assert got == B.mul(B.G, ref.scalar_dot(sc.tobytes(), zk.gen_scalars(SEED, n, 0).tobytes(), n))


@pytest.mark.parametrize("n", [1, 511, 8192, 8193])
@pytest.mark.parametrize("c", [2, 13, 14])
def test_one_block_sort_edges(eng, n, c):
    eng.set_window_bits(c)
    try:
        for dist in (0, 1):
            _check(eng, n, dist)
    finally:
        eng.set_window_bits(0)


@pytest.mark.parametrize("n", [1 << 18, (1 << 18) + 1])
def test_one_block_scan_edges(eng, n):
    for parts in (1, 2):
        eng.set_pipeline_parts(parts)
        try:
            _check(eng, n, 1)
        finally:
            eng.set_pipeline_parts(0)
