"""A cap on the engine's memory that leaves room only for the narrow-window
plan: the call still runs (lean plan) and gives the same bytes, on a plain
call and on the window-shifted resident table."""
import pytest

import zkmetal_amd as zk

pytestmark = pytest.mark.gpu

SEED = 0x1EA4


@pytest.mark.parametrize("n", [2048, 1 << 14])
def test_capped_plain_call(n):
    gen = zk.MetalMSM()
    e = zk.MetalMSM()
    try:
        gen.srs_generate(SEED, n)
        pts, sc = gen.srs_download(n), zk.gen_scalars(SEED + 1, n, 0)
        want = gen.msm(pts, sc)
        # what the narrow windows need (a forced width of 8 or 10 bits), and
        # nothing for 13 or 16 bits' buckets
        e.set_window_bits(10 if n > 4096 else 8)
        assert e.msm(pts, sc) == want
        need = e.workspace_bytes()
        e.close()
        e = zk.MetalMSM()
        e.set_workspace_limit(need + (1 << 20))
        assert e.msm(pts, sc) == want
        assert e.workspace_bytes() <= need + (1 << 20)
    finally:
        e.close()
        gen.close()


def test_capped_resident_call():
    n = 700
    e = zk.MetalMSM()
    try:
        e.srs_generate(SEED, 1 << 12)
        sc = zk.gen_scalars(SEED + 2, n, 0)
        ds = zk.DeviceBuffer(sc.nbytes)
        ds.upload(sc)
        want = e.msm_batch_resident(ds, [n])
        e.close()
        e = zk.MetalMSM()
        e.srs_generate(SEED, 1 << 12)
        e.set_workspace_limit(e.workspace_bytes() + (3 << 20))  # the shifted buckets take 4.7 MB
        assert e.msm_batch_resident(ds, [n]) == want
    finally:
        e.close()


def test_capped_call_of_many_lanes():
    # a cap that leaves no room for the third wave's merge records
    n = 1 << 17
    gen = zk.MetalMSM()
    e = zk.MetalMSM()
    try:
        gen.srs_generate(SEED, n)
        pts, sc = gen.srs_download(n), zk.gen_scalars(SEED + 3, n, 0)
        want = e.msm(pts, sc)
        need = e.workspace_bytes()
        e.close()
        e = zk.MetalMSM()
        e.set_workspace_limit(need - (8 << 20))
        assert e.msm(pts, sc) == want
        assert e.workspace_bytes() <= need - (8 << 20)
    finally:
        e.close()
        gen.close()
