"""The sort's routes at their edges against the closed form: a segment just
within and just past the one-block sort (16384 entries, 4096 buckets), and
segments on either side of the one-block histogram scan (128 tiles)."""
import numpy as np
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


@pytest.mark.parametrize("n", [8193, 12320, 40000])
@pytest.mark.parametrize("odd", [None, 63, 64, 8192])
def test_second_pass_with_one_low_byte(eng, n, odd):
    # keys that differ in their high bytes only (ranked without matching), and
    # the same with one entry of another low byte (matched) at a wave's edge
    rng = np.random.default_rng(SEED + n)
    k = 1 + 256 * rng.integers(0, 120, n, dtype=np.uint64)
    if odd is not None:
        k[odd] += 77
    sc = np.zeros((n, 4), np.uint64)
    sc[:, 0] = k
    sc = sc.reshape(-1).view(np.uint8)
    eng.set_window_bits(16)
    try:
        got = result_affine(eng.msm_batch_resident(sc, [n])[0])
    finally:
        eng.set_window_bits(0)
    assert got == B.mul(B.G, ref.scalar_dot(sc.tobytes(), zk.gen_scalars(SEED, n, 0).tobytes(), n))
