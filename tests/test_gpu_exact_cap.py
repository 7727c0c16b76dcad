"""A cap on the engine's memory of exactly what a call takes: the call keeps
its tuned window width."""
import pytest

import zkmetal_amd as zk

pytestmark = pytest.mark.gpu

SEED = 0xCA9


@pytest.mark.parametrize("n", [2048, 1 << 14])
def test_call_at_its_own_cap(n):
    gen, free, capped = zk.MetalMSM(), zk.MetalMSM(), zk.MetalMSM()
    try:
        gen.srs_generate(SEED, n)
        pts, sc = gen.srs_download(n), zk.gen_scalars(SEED + 1, n, 0)
        want = free.msm(pts, sc)
        width = free.last_timing()["window_bits"]
        capped.set_workspace_limit(free.workspace_bytes())
        assert capped.msm(pts, sc) == want
        assert capped.last_timing()["window_bits"] == width
        assert capped.workspace_bytes() == free.workspace_bytes()
    finally:
        for e in (gen, free, capped):
            e.close()
