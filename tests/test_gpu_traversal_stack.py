"""The traversal's stack past its LDS part: long thin triangles fanned about a
line overlap in every box, so rays along it keep more entries waiting than
there are in LDS, in one and in two levels; the oracle's traversal counts them.
Every distance equals, bit for bit, the oracle's brute force in 32 bits over
all triangles with the same watertight test. Calls of few rays have a ray or a
few per wave; above 32,768 the waves are full, and every second ray passes the
fan's end with fewer entries, so a wave has lanes on both sides of the limit."""
import numpy as np
import pytest

import oracle_py
from raygun_amd import rgrt
from raygun_amd.records import INSTANCE, MATERIAL, NO_HIT, RAY, VERTEX

pytestmark = pytest.mark.gpu

LDS_ENTRIES = 16  # kLdsStack in trace.hip


def fan(n, seed):
    """n slivers through the z axis's neighbourhood, each as long as the scene."""
    rng = np.random.default_rng(seed)
    a = rng.uniform(0, 2 * np.pi, n)
    p = np.zeros((n, 3, 3))
    p[:, 0] = np.stack([np.cos(a), np.sin(a), rng.uniform(-1, 1, n)], 1)
    p[:, 1] = np.stack([-np.cos(a), -np.sin(a), rng.uniform(-1, 1, n)], 1)
    p[:, 2] = p[:, 1] + rng.normal(0, 0.05, (n, 3))
    v = np.zeros(3 * n, VERTEX)
    v["position"] = p.reshape(-1, 3)
    v["normal"][:, 2] = 1.0
    return v, np.arange(3 * n, dtype=np.uint32)


@pytest.mark.parametrize("tris,instances,rays", [(1, 1, 1), (2, 3, 63), (700, 1, 65), (700, 40, 1000), (700, 2, 40_000)])
def test_hits_with_entries_past_the_lds_stack(tris, instances, rays):
    print(f"[case] stack tris={tris} instances={instances}", flush=True)
    v, i = fan(tris, 3)
    rng = np.random.default_rng(5)
    inst = np.zeros(instances, INSTANCE)
    inst["transform"] = [1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0]
    inst["transform"][:, [3, 7, 11]] = rng.uniform(-0.02, 0.02, (instances, 3))
    inst["customIndex"] = np.arange(instances)
    inst["mask"] = 0xFF
    inst["flags"] = 1
    r = np.zeros(rays, RAY)
    r["origin"] = np.stack([rng.uniform(-0.1, 0.1, rays), rng.uniform(-0.1, 0.1, rays), np.full(rays, -2.0)], 1)
    r["dir"] = np.stack([rng.normal(0, 0.01, rays), rng.normal(0, 0.01, rays), np.ones(rays)], 1)
    r["tmin"], r["tmax"] = 0.0, 100.0
    if rays > 32_768:
        r["origin"][1::2, 0] += 1.0
    ctx = rgrt.Context(16, 16)
    osc = oracle_py.OracleScene(v, i, np.zeros(0, MATERIAL))
    try:
        ctx.upload_geometry(v, i)
        inst["blas"] = ctx.build_blas(0, 0, tris, len(v))
        ctx.build_tlas(inst)
        assert osc.build_blas(0, 0, tris) == inst["blas"][0]
        osc.build_tlas(inst)
        depth = osc.stack_depths(r)
        if tris > 2:
            assert np.all(depth[::2] > LDS_ENTRIES)
        if rays > 32_768:
            spills = depth[:rays // 64 * 64].reshape(-1, 64) > LDS_ENTRIES
            assert not np.any(np.all(spills, 1)) and np.median(depth[1::2]) > 4
        got = ctx.trace_rays(r)
        t, instance, _ = osc.trace_rays_brute32(r)
        hit = instance != NO_HIT
        assert np.array_equal(got["instance"] != NO_HIT, hit)
        assert np.array_equal(got["t"][hit], t[hit])
        if tris > 2:
            assert np.count_nonzero(got["instance"] != NO_HIT) > rays // 2
    finally:
        ctx.close()
