"""Ray queries of every split: one ray per wave up to full waves, chunks by
position only and with the rest from the counter, ends of waves and chunks, from
host (up to 4096 rays through pinned memory) and from device memory: each ray's answer is the one it gets in a call of
its own size class, and the instance is the customIndex."""
import numpy as np
import pytest

from helpers import gpu_context, random_rays
from raygun_amd import procgen, rgrt
from raygun_amd.hiptime import DeviceBuffer
from raygun_amd.records import HIT

pytestmark = pytest.mark.gpu

SIMDS = 1024  # a full MI355X; the sizes below surround its switches


@pytest.mark.parametrize("n", [1, 3, SIMDS, SIMDS + 1, 4 * SIMDS - 1, 4 * SIMDS, 4 * SIMDS + 1, 32 * SIMDS + 1, 5 * 64 * SIMDS + 65, 1_000_003])
def test_hits_do_not_depend_on_the_call_size(n):
    print(f"[case] ray counts {n}", flush=True)
    setup = procgen.config2(64, 64, tris_per_mesh=500, num_instances=12)
    ctx, inst = gpu_context(setup)
    try:
        inst["customIndex"] = inst["customIndex"][::-1].copy()
        ctx.build_tlas(inst)
        rays = random_rays(n, 7, radius=70.0)
        rays["tmax"] = 300.0
        got = ctx.trace_rays(rays)
        dr, dh = DeviceBuffer(rays.nbytes), DeviceBuffer(n * HIT.itemsize)
        try:
            dr.upload(rays)
            dh.upload(np.zeros(n, HIT))
            for _ in range(2):  # the counter is cleared for each call
                ctx.trace_rays_device(dr.address, n, 0xFF, dh.address)
            ctx.synchronize()
            back = np.zeros(n, HIT)
            assert dh.L.hipMemcpy(back.ctypes.data, dh.ptr, back.nbytes, 2) == 0  # hipMemcpyDeviceToHost
        finally:
            dr.close()
            dh.close()
        assert np.array_equal(back.view(np.uint8), got.view(np.uint8))
        pick = np.unique(np.linspace(0, n - 1, 200).astype(np.int64))
        few = ctx.trace_rays(rays[pick])
        assert np.array_equal(few.view(np.uint8), got[pick].view(np.uint8))
        if n > 1000:
            assert 0.2 < np.mean(got["instance"] != 0xFFFFFFFF) <= 1.0
            assert got["instance"][got["instance"] != 0xFFFFFFFF].max() < len(inst)
    finally:
        ctx.close()


@pytest.mark.parametrize("n", [1, 5000])
def test_a_context_without_images_answers_ray_queries(n):
    print(f"[case] rays without images {n}", flush=True)
    setup = procgen.config2(64, 64, tris_per_mesh=500, num_instances=12)
    ctx, inst = gpu_context(setup)
    bare = ctx.shared(width=0, height=0)
    try:
        bare.build_tlas(inst)
        rays = random_rays(n, 3, radius=70.0)
        rays["tmax"] = 300.0
        assert np.array_equal(bare.trace_rays(rays).view(np.uint8), ctx.trace_rays(rays).view(np.uint8))
    finally:
        bare.close()
        ctx.close()
