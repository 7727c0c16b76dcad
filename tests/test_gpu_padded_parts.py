"""A window-shifted MSM split into eight parts, one window each, at sizes that
do not fill their last sort tile, after a larger call on the same engine has
left digits of its own in the buffers; against the closed form."""
import pytest

import zkmetal_amd as zk
from helpers import result_affine
from oracle import bn254 as B
from oracle import ref

pytestmark = pytest.mark.gpu

SEED = 0x8BA2


def test_padding_of_one_window_parts():
    top = 1 << 17
    keys = zk.gen_scalars(SEED, top, 0)
    e = zk.MetalMSM()
    try:
        e.srs_generate(SEED, top)
        e.set_window_shift(e.SHIFT_ALL)
        for n in (top, 5001, 1, 2047, 70001):
            sc = zk.gen_scalars(SEED + n, n, 0)
            for parts in (8, 5):
                e.set_pipeline_parts(parts)
                print(f"n={n} parts={parts}", flush=True)
                got = result_affine(e.msm_batch_resident(sc, [n])[0])
                assert got == B.mul(B.G, ref.scalar_dot(sc.tobytes(), keys[:n].tobytes(), n))
    finally:
        e.close()
