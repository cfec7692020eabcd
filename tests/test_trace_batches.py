"""Ray batches at the sizes where the traversal kernels split their work
differently, against the oracle: hits bit for bit (the kernels only hand rays
out differently; each ray's own arithmetic does not change)."""
import os

import numpy as np
import pytest

from bulbit_amd import scenes

THREADS = max(1, min(16, len(os.sched_getaffinity(0))))


@pytest.fixture(scope="module")
def small():
    from bulbit_amd.gpu import GpuScene
    from oracle import OracleScene

    sc, _ = scenes.icosphere_scene(level=3)
    return GpuScene(sc), OracleScene(sc)


# one ray; below, at and past the fewest rays a wave starts with (8); one
# wave and one block more; past 8 per wave of a full grid (some 6,000 to 8,000
# waves); and past 128 per wave, where the shared counter takes over
@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 8, 9, 64, 65, 129, 70001, 1_050_001])
@pytest.mark.parametrize("any_hit", [False, True])
def test_batch_sizes(small, n, any_hit):
    g, o = small
    bmin, bmax = o.world_bounds()
    rays = scenes.random_rays(bmin, bmax, n, seed=n, t_max=3.0 if any_hit else np.inf)
    hits, _ = g.trace(rays, any_hit=any_hit)
    want, _ = o.trace(rays, any_hit=any_hit, threads=THREADS)
    assert np.array_equal(hits["prim"], want["prim"])
    if not any_hit:
        for f in ("t", "u", "v"):
            assert np.array_equal(hits[f].view(np.int32), want[f].view(np.int32)), f


def _same(g, o, rays, any_hit):
    hits, _ = g.trace(rays, any_hit=any_hit)
    want, _ = o.trace(rays, any_hit=any_hit, threads=THREADS)
    assert np.array_equal(hits["prim"], want["prim"])
    if not any_hit:
        for f in ("t", "u", "v"):
            assert np.array_equal(hits[f].view(np.int32), want[f].view(np.int32)), f
    return float(np.mean(want["prim"] >= 0))


# The traversal records hold boxes rounded outwards and are tested with a
# margin; the exact box of a leaf decides before a hit counts.  Rays that sit
# at the margins' ends: directions along axes and nearly so (also negative
# zero), of lengths other than one, from far away, over ranges that start or
# lie behind the origin, and rays the library must finish but that hit nothing
KINDS = ["axis", "near_axis", "negative_zero", "long", "short", "far", "negative_range", "empty_range",
         "infinite_origin"]


def _hard_rays(kind, bmin, bmax, n=40_000):
    rng = np.random.default_rng(KINDS.index(kind) + 100)
    rays = scenes.random_rays(bmin, bmax, n, seed=KINDS.index(kind) + 200)
    i, axis = np.arange(n), rng.integers(0, 3, n)
    if kind in ("axis", "near_axis", "negative_zero"):
        other = {"axis": 0.0, "near_axis": 1e-30, "negative_zero": -0.0}[kind]
        d = np.full((n, 3), other, np.float32)
        d[i, axis] = np.where(rng.random(n) < 0.5, 1.0, -1.0)
        if kind == "near_axis":  # some components just small, some far below what 1 / d can hold
            d = np.where(np.abs(d) < 0.5, d * 10.0 ** rng.uniform(-10, 26, (n, 3)), d).astype(np.float32)
        rays["d"] = d
    elif kind == "long":
        rays["d"] *= (10.0 ** rng.uniform(0, 12, n))[:, None].astype(np.float32)
        rays["t_min"] = 0.0
    elif kind == "short":
        rays["d"] *= (10.0 ** rng.uniform(-6, 0, n))[:, None].astype(np.float32)
    elif kind == "far":
        target = rays["o"].copy()
        rays["o"] = target - rays["d"] * (10.0 ** rng.uniform(1, 5, n))[:, None].astype(np.float32)
    elif kind == "negative_range":
        rays["t_min"] = -rng.uniform(0, 10, n)
        rays["t_max"] = rays["t_min"] + rng.uniform(0, 10, n).astype(np.float32)
    elif kind == "empty_range":
        rays["t_max"] = rays["t_min"] - 1.0
    elif kind == "infinite_origin":
        rays["o"][i, axis] = np.where(rng.random(n) < 0.5, np.inf, -np.inf)
    return rays


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("any_hit", [False, True])
def test_rays_at_the_margins(small, kind, any_hit):
    g, o = small
    bmin, bmax = o.world_bounds()
    hit = _same(g, o, _hard_rays(kind, bmin, bmax), any_hit)
    assert (hit > 0.0) == (kind not in ("empty_range", "infinite_origin"))


# scenes whose coordinates are large against their details, small, spread
# over many magnitudes, or flat
@pytest.mark.gpu
@pytest.mark.parametrize("place", ["offset", "small", "large", "mixed", "flat"])
def test_scenes_at_the_margins(place):
    from bulbit_amd.gpu import GpuScene
    from oracle import OracleScene

    sc, _ = scenes.icosphere_scene(level=3)
    p = sc.positions.astype(np.float64)
    if place == "offset":
        p += [4096.0, -300.0, 77.7]
    elif place == "small":
        p *= 1e-2  # below this the reference's epsilon on the determinant misses every triangle
    elif place == "large":
        p *= 1e9
    elif place == "mixed":
        p[:642] = p[:642] * 1e-3 + [0.0, 5.0, 0.0]
    else:
        p[:, 1] = 0.25
    sc.positions = p.astype(np.float32)
    g, o = GpuScene(sc), OracleScene(sc)
    bmin, bmax = o.world_bounds()
    rays = scenes.random_rays(bmin, bmax, 60_000, seed=3)
    if place in ("mixed", "flat"):  # aim at the geometry
        tri = sc.positions[sc.indices[np.random.default_rng(4).integers(0, len(sc.indices), len(rays))]]
        rays["o"] = np.float32([0.3, 6.0, 2.0]) + 0.1 * rays["d"]
        rays["d"] = tri.mean(1) - rays["o"]
        rays["t_min"] = 0.0
    else:
        rays["t_min"] = 0.0
    hit = _same(g, o, rays, False)
    assert hit > 0.01
    rays["t_max"] = np.float32(1.0) if place in ("mixed", "flat") else np.float32(0.3 * np.linalg.norm(bmax - bmin))
    _same(g, o, rays, True)


# The film at the path order's edges: strips of 8 pixels (widths 1, 7, 8, 9,
# 65), one sample, fewer, as many and more than the film kernel takes at a
# time (8), and several passes of unequal sample counts; every sample's value
# is fixed by its pixel and number, so the film equals the sum of one-sample
# films in sample order bit for bit
@pytest.mark.gpu
@pytest.mark.parametrize("width,height,spp,paths", [(1, 1, 3, 0), (7, 5, 8, 0), (8, 8, 2, 0), (9, 3, 9, 0), (65, 33, 17, 0),
                                                    (65, 33, 17, 65 * 33 * 5), (16, 40, 7, 16 * 40 * 3)])
def test_film_equals_its_samples(small, width, height, spp, paths):
    g, _ = small
    cam = scenes.make_camera((0.0, 2.4, 5.2), (0.0, 0.9, 0.0), 38.0, 0.0, 5.0, width, height)
    s, c, _ = g.render(cam, scenes.render_params(spp, max_bounces=3, seed=5, wavefront_paths=paths))
    film = g.new_film(cam)
    for k in range(spp):
        ws, wc, _ = g.render(cam, scenes.render_params(1, max_bounces=3, seed=5, sample_begin=k), film=film)
    assert np.array_equal(c, wc) and np.array_equal(s.view(np.int32), ws.view(np.int32))
    assert np.any(s > 0) or width == 1
