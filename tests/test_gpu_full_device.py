"""A device with no room for the tuned plan and no cap set: the call runs on
the narrow-window plan with the same result, also when it meets the limit
after larger buffers were in place, and the engine goes on."""
import pytest

import zkmetal_amd as zk

pytestmark = pytest.mark.gpu

SEED = 0xF011


def test_plain_call_on_a_full_device():
    n = 1 << 14
    gen, e = zk.MetalMSM(), zk.MetalMSM()
    try:
        gen.srs_generate(SEED, n)
        pts, sc = gen.srs_download(n), zk.gen_scalars(SEED + 1, n, 0)
        want = gen.msm(pts, sc)
        e.set_window_bits(10)
        assert e.msm(pts, sc) == want
        need = e.workspace_bytes()
        e.close()
        e = zk.MetalMSM()
        zk._check(zk.lib().zkmsm_test_device_memory(e.handle, need + (1 << 20)), "test_device_memory")
        for _ in range(2):
            assert e.msm(pts, sc) == want
            assert e.last_timing()["window_bits"] == 10
        # no room for either plan: refused, and well again with room
        f = zk.MetalMSM()
        try:
            zk._check(zk.lib().zkmsm_test_device_memory(f.handle, 8 << 20), "test_device_memory")
            with pytest.raises(zk.MSMError) as err:
                f.msm(pts, sc)
            assert err.value.status == zk.ERR_ALLOC_FAILED
            zk._check(zk.lib().zkmsm_test_device_memory(f.handle, 0), "test_device_memory")
            assert f.msm(pts, sc) == want
            assert f.last_timing()["window_bits"] == 16
        finally:
            f.close()
    finally:
        e.close()
        gen.close()


def test_resident_batch_on_a_full_device():
    counts = [512] * 64
    e = zk.MetalMSM()
    try:
        e.srs_generate(SEED, 1 << 12)
        sc = zk.gen_scalars(SEED + 2, sum(counts), 0)
        ds = zk.DeviceBuffer(sc.nbytes)
        ds.upload(sc)
        zk._check(zk.lib().zkmsm_test_device_memory(e.handle, e.workspace_bytes() + (160 << 20)), "test_device_memory")
        lean = e.msm_batch_resident(ds, counts)
        assert e.workspace_bytes() < 160 << 20  # the shifted buckets alone take 300 MB
        zk._check(zk.lib().zkmsm_test_device_memory(e.handle, 0), "test_device_memory")
        assert e.msm_batch_resident(ds, counts) == lean
        assert e.workspace_bytes() > 300 << 20
    finally:
        e.close()
