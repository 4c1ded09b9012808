"""Wide trees on both sides of the numbering's switch from one workgroup to a
sort by level (more than 32768 leaves): random triangles, clusters whose
subtrees are deep and uneven, and equal centroids (Morton ties broken by
index), and of the box refit's switch to a middle pass (2^18 leaves). Node for
node the oracle's trees, as built, refitted and rebuilt."""
import numpy as np
import pytest

import oracle_py
from raygun_amd import rgrt
from raygun_amd.records import MATERIAL, VERTEX

pytestmark = pytest.mark.gpu


def soup(n, shape, seed):
    rng = np.random.default_rng(seed)
    if shape == "random":
        c = rng.uniform(-10, 10, (n, 3))
    elif shape == "clusters":
        c = rng.choice(rng.uniform(-10, 10, (9, 3)), n) + rng.normal(0, 1, (n, 3)) * 10.0 ** rng.uniform(-6, 0, (n, 1))
    else:  # a few places, thousands of triangles in each
        c = rng.integers(-2, 3, (n, 3)).astype(float)
    v = np.zeros(3 * n, VERTEX)
    v["position"] = (c[:, None] + rng.normal(0, 0.05, (n, 3, 3)) * (shape != "ties")).reshape(-1, 3)
    v["normal"][:, 1] = 1.0
    return v, np.arange(3 * n, dtype=np.uint32)


@pytest.mark.parametrize("n,shape", [(32768, "random"), (32769, "random"), (50_001, "clusters"), (40_000, "ties"),
                                     (140_000, "clusters"), ((1 << 18) - 1, "random"), (1 << 18, "clusters"),
                                     (300_001, "ties")])
def test_wide_trees_equal_the_oracles(n, shape):
    print(f"[case] wide numbering {n} {shape}", flush=True)
    v, i = soup(n, shape, 3)
    moved, _ = soup(n, shape, 4)
    ctx, osc = rgrt.Context(16, 16), oracle_py.OracleScene(v, i, np.zeros(0, MATERIAL))
    try:
        ctx.upload_geometry(v, i)
        b = ctx.build_blas(0, 0, n, len(v))
        assert osc.build_blas(0, 0, n) == b

        def same(what):
            for compressed in (False, True):
                assert np.array_equal(ctx.export_blas_wide(b, compressed), osc.export_blas_wide(b, compressed)), what

        same("built")
        ctx.update_vertices(0, moved)
        osc.update_vertices(0, moved)
        ctx.refit_blas(b)
        osc.refit_blas(b)
        same("refitted")
        osc.rebuild_blas(b)
        ctx.rebuild_blas(b)
        same("rebuilt")
        if n <= 1 << 18:
            ctx.rebuild_blas_noalloc(b)
            same("rebuilt in the fixed scratch")
    finally:
        ctx.close()
