"""G2 sums of equal buckets that the merge stored: neighbouring buckets of the
lowest window hold copies of one point each, another point for every pair, so
that the bucket reduction by lanes doubles points left by the lane teams;
against the closed form."""
import numpy as np
import pytest

import zkmetal_amd as zk
from oracle import bn254_g2 as G

pytestmark = pytest.mark.gpu

SEED = 0x62D0


# a forced width whose buckets are reduced by lanes, and the default one there
@pytest.mark.parametrize("n,c", [(150001, 16), (300000, 0)])
def test_equal_merged_buckets(engine, n, c):
    m = 1 << 14
    buf = zk.DeviceBuffer(m * 128)
    engine.g2_points_generate(SEED, m, buf)
    table = np.frombuffer(buf.download(), dtype=np.uint8).reshape(m, 128)
    bucket = np.random.default_rng(n).permutation(n) % (2 * m - 1)
    scalars = np.zeros((n, 4), dtype=np.uint64)
    scalars[:, 0] = bucket + 1
    engine.set_window_bits(c)
    try:
        got = engine.g2_msm(np.ascontiguousarray(table[bucket // 2]).reshape(-1), scalars.view(np.uint8).reshape(-1))
    finally:
        engine.set_window_bits(0)
    keys = zk.gen_scalars(SEED, m, 0).reshape(m, 32)
    weight = np.bincount(bucket // 2, weights=bucket + 1, minlength=m)
    total = sum(int.from_bytes(k.tobytes(), "little") * int(w) for k, w in zip(keys, weight))
    assert G.jacobian_bytes_to_affine(got) == G.mul(G.G2, total % G.R_ORDER)
