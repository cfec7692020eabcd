"""The work that programs of this framework have it do, as cases for timing
and comparing: ray batches, renders, batches of renders, and the radiance
cache alone and inside a render.  Every case goes through the public entry
points (bulbit_amd.gpu, bulbit_amd.nrc and the C ABI below them) with device
buffers, as bench.py and the examples call them.

A case is a dict of plain values; "kind" names the path and the other entries
its sizes and options.  The sizes are those of bench.py's workloads, of the
tests and of the README, cut where a scene would take long to generate, and
odd ones beside them.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from bulbit_amd import capi, scenes
from bulbit_amd.gpu import GpuScene, render_batch
from bulbit_amd.nrc import Nrc

SHAPES = {"64x4": (64, 4), "128x5": (128, 5)}  # hidden width and layers of the two networks
ENC_USED, ENC, OUT, OUT_PAD = 74, 80, 3, 16    # the cache's input and output, as stored


def listed():
    return [
        # picking and probing: a handful of rays, where the call itself is the cost
        {"name": "trace_few", "kind": "trace", "scene": "icosphere", "level": 4, "rays": 61, "any_hit": False,
         "camera": False, "noalloc": False},
        # one large closest-hit batch of incoherent rays (BVH::Intersect over a ray set), an odd count
        {"name": "trace_closest", "kind": "trace", "scene": "icosphere", "level": 7, "rays": 1000003,
         "any_hit": False, "camera": False, "noalloc": False},
        # visibility over a large set of bounded segments (BVH::IntersectAny)
        {"name": "trace_any", "kind": "trace", "scene": "icosphere", "level": 7, "rays": 4194304, "any_hit": True,
         "camera": False, "noalloc": False},
        # the README example: one analytic sphere, 640 x 360 at 16 spp
        {"name": "render_readme", "kind": "render", "scene": "readme", "level": 0, "lights": 0, "width": 640,
         "height": 360, "spp": 16, "bounces": 8, "filter": "box", "graph": False},
        # one progressive frame of an interactive preview: 1 spp, where launches and short tails count
        {"name": "render_preview", "kind": "render", "scene": "icosphere", "level": 6, "lights": 64, "width": 1280,
         "height": 720, "spp": 1, "bounces": 8, "filter": "box", "graph": False},
        # the benchmark's frame: 1.31 M triangles, 1080p, 64 spp, 8 bounces (the largest case)
        {"name": "render_frame", "kind": "render", "scene": "icosphere", "level": 8, "lights": 64, "width": 1920,
         "height": 1080, "spp": 64, "bounces": 8, "filter": "box", "graph": False},
        # textures in every slot, normal maps, alpha cut-outs, every BxDF, the Gaussian filter, ragged sizes
        {"name": "render_textured", "kind": "render", "scene": "textured", "level": 6, "lights": 16, "width": 801,
         "height": 451, "spp": 8, "bounces": 8, "filter": "gaussian", "graph": False},
        # the large-scene generator: metallic-roughness spheres on a plane, many area lights, 12 bounces
        {"name": "render_many_lights", "kind": "render", "scene": "spheres", "level": 5, "lights": 1024,
         "width": 1920, "height": 1080, "spp": 4, "bounces": 12, "filter": "box", "graph": False},
        # several uneven scenes rendered by one call, as the batched workload does
        {"name": "render_batch", "kind": "batch", "jobs": 8, "max_level": 6, "spp": 16, "sizes": 303},
        # one frame of the cached path tracer with online training (4 Adam steps), 64-wide network
        {"name": "cached_frame", "kind": "cached", "scene": "readme", "level": 0, "lights": 0, "width": 1920,
         "height": 1080, "spp": 1, "bounces": 8, "net": "64x4", "steps": 4, "primary": True, "direct": False},
        # inference of the wide network over a frame's worth of query rows, an odd count
        {"name": "cache_query", "kind": "query", "net": "128x5", "rows": 2000003},
        # the wide network's training loop: 4 Adam steps of 65,536 rows
        {"name": "cache_train", "kind": "train", "net": "128x5", "rows": 65536, "steps": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "render", "render", "render", "batch", "cached", "query", "train"])
    if kind == "trace":
        return {"kind": kind, "scene": rng.choice(["icosphere", "icosphere", "textured", "readme", "spheres"]),
                "level": rng.randint(3, 7), "rays": _log_int(rng, 1, 4000000), "any_hit": rng.random() < 0.5,
                "camera": rng.random() < 0.5, "noalloc": rng.random() < 0.25}
    if kind in ("render", "cached"):
        width = _log_int(rng, 64, 1920)
        height = max(36, min(1080, int(width * rng.uniform(0.4, 1.2))))
        most = max(1, min(64, 16000000 // (width * height)))
        case = {"kind": kind, "scene": rng.choice(["readme", "icosphere", "icosphere", "textured", "spheres"]),
                "level": rng.randint(3, 7), "lights": _log_int(rng, 4, 1024), "width": width, "height": height,
                "spp": _log_int(rng, 1, most), "bounces": rng.randint(2, 12)}
        if kind == "render":
            return {**case, "filter": rng.choice(["box", "tent", "gaussian"]), "graph": rng.random() < 0.25}
        return {**case, "spp": min(case["spp"], 4), "net": rng.choice(sorted(SHAPES)), "steps": rng.randint(0, 4),
                "primary": rng.random() < 0.5, "direct": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "jobs": rng.randint(2, 10), "max_level": rng.randint(5, 6), "spp": rng.randint(1, 16),
                "sizes": rng.randint(0, 9999)}
    net = rng.choice(sorted(SHAPES))
    if kind == "query":
        return {"kind": kind, "net": net, "rows": _log_int(rng, 1, 4000000)}
    return {"kind": kind, "net": net, "rows": _log_int(rng, 64, 131072), "steps": rng.randint(1, 4)}


# ------------------------------------------------------------------- scenes

def _textured(width, height, level, seed, n_lights):
    """The displaced icosphere with spherical texture coordinates, its face
    groups cycling through textured materials of every kind, some with normal
    maps and alpha, over a checkered ground, with a dim environment."""
    sc, cam = scenes.icosphere_scene(width, height, level=level, seed=seed, n_lights=n_lights)
    rng = np.random.default_rng(seed)
    p = sc.positions.astype(np.float64) - np.array([0.0, 1.05, 0.0])
    r = np.maximum(np.linalg.norm(p, axis=1), 1e-9)
    uvs = np.stack([3.0 * ((np.arctan2(p[:, 2], p[:, 0]) / (2 * np.pi)) % 1.0),
                    2.0 * np.arccos(np.clip(p[:, 1] / r, -1, 1)) / np.pi], 1)
    ground = len(sc.positions) - 3 * n_lights - 4
    uvs[ground:] = 0.0
    uvs[ground:ground + 4] = [[0, 0], [8, 0], [8, 8], [0, 8]]
    sc.uvs = uvs.astype(np.float32)

    def image(h, w, c):
        return sc.add_texture(scenes.image_texture(
            rng.uniform(0.05, 0.95, (h, w, c) if c > 1 else (h, w)).astype(np.float32)))

    def constant(v):
        return sc.add_texture(scenes.constant_texture(v))

    albedo, rough = image(256, 512, 3), image(64, 64, 1)
    metal = sc.add_texture(scenes.image_texture((rng.random((32, 32)) > 0.5).astype(np.float32)))
    check = sc.add_texture(scenes.checker_texture(constant(0.05), constant(0.5), (8.0, 8.0), 1))
    yy, xx = np.mgrid[0:64, 0:64] / 64.0
    normal = sc.add_texture(scenes.image_texture(np.stack(
        [0.5 + 0.3 * np.sin(6 * np.pi * xx), 0.5 + 0.3 * np.cos(4 * np.pi * yy), np.full((64, 64), 0.9)],
        2).astype(np.float32)))
    cut = np.where(rng.random((32, 32)) < 0.4, 0.0, 1.0).astype(np.float32)
    cut[:8] = 0.5  # fractional rows
    alpha = sc.add_texture(scenes.image_texture(cut))
    floor = sc.add_texture(scenes.checker_texture(constant((0.8, 0.8, 0.8)), constant((0.2, 0.3, 0.6)), (4.0, 4.0), 3))

    def mat(m, **slots):
        for k, v in slots.items():
            setattr(m, k, v)
        return m

    mats = [
        mat(scenes.diffuse((1, 1, 1)), tex_color=albedo),
        mat(scenes.conductor(scenes.GOLD_ETA, scenes.GOLD_K, 0.3), tex_u_roughness=check, tex_v_roughness=check),
        mat(scenes.metallic_roughness((0.9, 0.6, 0.3), 0.0, 0.5), tex_color=albedo, tex_u_roughness=rough,
            tex_v_roughness=rough, tex_metallic=metal),
        mat(scenes.dielectric(1.5, roughness=0.3, energy_compensation=1), tex_u_roughness=rough,
            tex_v_roughness=rough),
        mat(scenes.diffuse((0.7, 0.7, 0.7)), tex_normal=normal),
        mat(scenes.conductor(scenes.GOLD_ETA, scenes.GOLD_K, 0.2, energy_compensation=1), tex_normal=normal),
        mat(scenes.diffuse((0.8, 0.7, 0.6)), tex_u_roughness=check),
        mat(scenes.diffuse((0.6, 0.9, 0.6)), tex_alpha=alpha),
        mat(scenes.metallic_roughness((0.5, 0.5, 0.9), 1.0, 0.3), tex_alpha=alpha, tex_normal=normal),
        mat(scenes.diffuse((1, 1, 1)), tex_color=floor),
    ]
    base, faces = len(sc.materials), 20 * 4 ** level
    sc.materials += mats
    sc.prims[:faces, 2] = base + (np.arange(faces) // 256) % (len(mats) - 1)
    sc.prims[faces:faces + 2, 2] = len(sc.materials) - 1
    sc.add_infinite_light((0.05, 0.06, 0.08))
    return sc, cam


def _scene(case, seed, width, height):
    """(SceneData, camera) of a case"""
    kind, lights = case["scene"], case.get("lights", 64)
    if kind == "readme":  # no seeded part: the camera moves a little instead
        sc, cam = scenes.readme_scene(width, height)
        t = 0.01 * (seed % 997)
        pos = (3.0 * math.cos(t) - 0.4 * math.sin(t), 2.0, 5.0)
        return sc, scenes.make_camera(pos, (0.0, 1.0, 0.0), 35.0, 0.01, 6.0, width, height)
    if kind == "spheres":
        return scenes.large_scene(width, height, n_spheres=64, level=min(case["level"], 5), n_lights=lights,
                                  seed=5150 + seed % 100000)
    if kind == "textured":
        return _textured(width, height, case["level"], 2026 + seed % 100000, lights)
    return scenes.icosphere_scene(width, height, level=case["level"], seed=2026 + seed % 100000, n_lights=lights)


def _prims(case):
    kind, lights = case["scene"], case.get("lights", 64)
    if kind == "readme":
        return 1
    faces = 20 * 4 ** (min(case["level"], 5) if kind == "spheres" else case["level"])
    return faces * (64 if kind == "spheres" else 1) + 2 + lights


def _rays(case, seed, g, cam):
    """the batch's rays as a device tensor of 8 floats each"""
    n = case["rays"]
    lo, hi = np.array(g.info.world_min[:]), np.array(g.info.world_max[:])
    if case["camera"]:  # a pinhole at the camera's place: neighbours run together
        gen = np.random.default_rng(seed)
        side = max(1, int(math.isqrt(n)))
        i = np.arange(n)
        x = ((i % side) + gen.random(n)) / side - 0.5
        y = ((i // side) + gen.random(n)) / max(1, -(-n // side)) - 0.5
        eye = np.array(cam.position[:], np.float64)
        fwd = 0.5 * (lo + hi) - eye
        fwd /= np.linalg.norm(fwd)
        right = np.cross(fwd, [0.0, 1.0, 0.0])
        right /= np.linalg.norm(right)
        up = np.cross(right, fwd)
        d = fwd + 0.7 * x[:, None] * right + 0.5 * y[:, None] * up
        rays = np.zeros(n, capi.RAY_DTYPE)
        rays["o"] = eye
        rays["d"] = d / np.linalg.norm(d, axis=1, keepdims=True)
        rays["t_min"] = np.float32(1e-4)
        rays["t_max"] = 0.75 * np.linalg.norm(hi - lo) if case["any_hit"] else np.inf
    else:
        t_max = 0.25 * float(np.linalg.norm(hi - lo)) if case["any_hit"] else np.inf
        rays = scenes.random_rays(lo, hi, n, seed, t_max=t_max)
    return torch.from_numpy(rays.view(np.float32).reshape(n, 8)).to("cuda")


# -------------------------------------------------------------------- cache

def _layers(net):
    width, hidden = SHAPES[net]
    return [(ENC if l == 0 else width, OUT_PAD if l == hidden else width) for l in range(hidden + 1)]


def _weights(net, seed):
    """Xavier-uniform weights, the padding zero, k-major per layer"""
    rng = np.random.default_rng(seed)
    shapes, out = _layers(net), []
    for l, (k, n) in enumerate(shapes):
        last = l == len(shapes) - 1
        a = math.sqrt(6.0 / ((ENC_USED if l == 0 else k) + (OUT if last else n)))
        m = rng.uniform(-a, a, (k, n)).astype(np.float32)
        if l == 0:
            m[ENC_USED:] = 0
        if last:
            m[:, OUT:] = 0
        out.append(m)
    return out


def _rows(n, seed):
    """feature rows as a render makes them, and smooth radiance targets"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    raw = torch.rand((n, 16), generator=gen, device="cuda")
    for c in (3, 6):
        v = 2.0 * raw[:, c:c + 3] - 1.0
        raw[:, c:c + 3] = v / v.norm(dim=1, keepdim=True).clamp_min(1e-6)
    raw[:, 13:] = 0.0
    base = 0.6 + 0.3 * torch.sin(2 * math.pi * raw[:, 0]) * torch.cos(math.pi * raw[:, 1]) + 0.2 * raw[:, 2]
    target = torch.stack([base, 0.8 * base + 0.1 * raw[:, 8], 0.5 * base + 0.2 * raw[:, 12]], 1)
    return raw, target.contiguous()


def _net(case, seed):
    width, layers = SHAPES[case["net"]]
    net = Nrc(seed=1 + seed % 100000, width=width, layers=layers)
    net.set_weights(np.concatenate([m.ravel() for m in _weights(case["net"], seed)]))
    return net


# ------------------------------------------------------------------ the cases

def prepare(case, seed):
    kind = case["kind"]
    if kind == "trace":
        sc, cam = _scene(case, seed, 640, 360)
        g = GpuScene(sc)
        return {"kind": kind, "case": case, "scene": g, "rays": _rays(case, seed, g, cam),
                "hits": torch.empty((case["rays"], 4), dtype=torch.int32, device="cuda")}
    if kind in ("render", "cached"):
        sc, cam = _scene(case, seed, case["width"], case["height"])
        if kind == "render" and case["filter"] != "box":
            scenes.set_filter(cam, case["filter"])
        g = GpuScene(sc)
        state = {"kind": kind, "case": case, "scene": g, "camera": cam, "film": g.new_film(cam), "frame": 0,
                 "seed": seed % 100000}
        if kind == "cached":
            state["net"] = _net(case, seed)
            state["cache"] = scenes.cache_params(train_steps=case["steps"], query_primary=case["primary"],
                                                 query_direct=case["direct"])
        return state
    if kind == "batch":
        jobs = []
        for spec in scenes.batch_workload_specs(case["jobs"], seed=case["sizes"]):
            spec = {**spec, "level": min(spec["level"], case["max_level"]), "seed": seed % 100000,
                    "scene_seed": spec["scene_seed"] + seed % 100000}
            sc, cam, params = scenes.batch_workload_job(spec, spp=case["spp"])
            g = GpuScene(sc)
            jobs.append((g, cam, params, g.new_film(cam)))
        return {"kind": kind, "jobs": jobs}
    raw, target = _rows(case["rows"] * case.get("steps", 1), seed)
    state = {"kind": kind, "case": case, "net": _net(case, seed), "raw": raw, "target": target}
    if kind == "query":
        state["out"] = torch.empty((case["rows"], OUT), dtype=torch.float32, device="cuda")
    return state


def run(state):
    kind = state["kind"]
    if kind == "trace":
        case, hits = state["case"], state["hits"]
        trace = state["scene"].trace_noalloc_device if case["noalloc"] else state["scene"].trace_device
        trace(state["rays"].data_ptr(), case["rays"], hits.data_ptr(), any_hit=case["any_hit"])
        return {"prim": hits[:, 0], "t": hits.view(torch.float32)[:, 1], "uv": hits.view(torch.float32)[:, 2:]}
    if kind in ("render", "cached"):
        case, (total, count) = state["case"], state["film"]
        total.zero_()
        count.zero_()
        params = scenes.render_params(case["spp"], max_bounces=case["bounces"], seed=state["seed"],
                                      sample_begin=state["frame"] * case["spp"], graph=int(case.get("graph", False)))
        state["frame"] = (state["frame"] + 1) % 4096  # the next frame takes new samples
        if kind == "render":
            state["scene"].render_device(state["camera"], params, total.data_ptr(), count.data_ptr())
            return {"sum": total, "count": count}
        state["scene"].render_cached_device(state["net"], state["camera"], params, state["cache"], total.data_ptr(),
                                            count.data_ptr())
        return {"sum": total, "count": count, "weights": state["net"].weights()}
    if kind == "batch":
        for _, _, _, (total, count) in state["jobs"]:
            total.zero_()
            count.zero_()
        render_batch(state["jobs"])
        return [list(film) for _, _, _, film in state["jobs"]]
    case, net, raw = state["case"], state["net"], state["raw"]
    if kind == "query":
        out = state["out"]
        capi.check(net.lib.bbgpu_nrc_query(net.h, raw.data_ptr(), case["rows"], out.data_ptr(), None),
                   "bbgpu_nrc_query", net.lib)
        return out
    loss = ctypes.c_float()
    n, steps = case["rows"], case["steps"]
    for s in range(steps):  # the loss is read after the last step only
        capi.check(net.lib.bbgpu_nrc_train(net.h, raw[n * s:].data_ptr(), state["target"][n * s:].data_ptr(), n, 1,
                                           ctypes.byref(loss) if s == steps - 1 else None, None, None),
                   "bbgpu_nrc_train", net.lib)
    return {"weights": net.weights(), "loss": loss.value}


def _ray_work(prims):
    """bytes and operations one ray cannot do without: a root-to-leaf walk of
    a binary tree (both children's boxes per level: 64 bytes, 2 x 18
    operations) and one triangle (48 bytes, about 60 operations)"""
    depth = max(1.0, math.log2(max(2, prims)))
    return 64.0 * depth + 48.0, 36.0 * depth + 60.0


def work(case):
    kind = case["kind"]
    if kind in ("query", "train"):
        shapes = _layers(case["net"])
        params = sum(k * n for k, n in shapes)
        used = sum((ENC_USED if l == 0 else k) * (OUT if l == len(shapes) - 1 else n)
                   for l, (k, n) in enumerate(shapes))
        if kind == "query":
            return {"bytes": case["rows"] * (13 + 3) * 4.0 + 2.0 * params, "flops": 2.0 * used * case["rows"]}
        # Adam reads and writes the fp32 weights and both moments
        per_step = case["rows"] * (13 + 3) * 4.0 + 24.0 * params
        return {"bytes": per_step * case["steps"], "flops": 6.0 * used * case["rows"] * case["steps"]}
    if kind == "batch":
        # mean job of the generator: 0.44 Mpixel, 16 spp, two rays a sample
        paths = case["jobs"] * 440000.0 * case["spp"]
        return {"bytes": case["jobs"] * 440000.0 * 32, "flops": paths * 2 * _ray_work(20 * 4 ** case["max_level"])[1]}
    prims = _prims(case)
    scene_bytes = prims * (64.0 + 48.0)  # every inner node's two boxes and every triangle once
    ray_bytes, ray_flops = _ray_work(prims)
    if kind == "trace":
        n = case["rays"]
        return {"bytes": 48.0 * n + min(scene_bytes, n * ray_bytes), "flops": n * ray_flops}
    # a camera ray and a shadow ray a sample at least; the film read and written
    pixels = case["width"] * case["height"]
    rays = 2.0 * pixels * case["spp"]
    got = {"bytes": 32.0 * pixels + min(scene_bytes, rays * ray_bytes), "flops": rays * ray_flops}
    if kind == "cached":
        shapes = _layers(case["net"])
        got["flops"] += 2.0 * sum(k * n for k, n in shapes) * (0.4 * pixels + 3 * 65536 * case["steps"])
    return got


def tolerance(case):
    kind = case["kind"]
    if kind == "trace":
        # whole numbers and the float32 operations of the reference in its order: bit for bit
        return "exact"
    if kind in ("render", "batch"):
        # Paths are chaotic: a last-bit change of a sine flips a few of them.
        # Films of the CPU restatement with the C library's float sines
        # against correctly rounded ones: untextured scenes 1e-4 in the
        # 2-norm and 0.05 in one pixel, with alpha textures (a hash of the
        # ray's bits decides) 6e-3 and 1.9.  Four times that, to the most
        # that a comparison takes; counts are equal.
        if case.get("scene") == "textured":
            return {"rel": 0.025, "max": 0.99}
        return {"rel": 4e-4, "max": 0.2}
    if kind == "cached":
        # bf16 predictions, and weights that Adam moves by about one learning
        # rate whatever the gradient's size: the rows' order is not fixed
        return {"rel": 0.02, "max": 0.5}
    if kind == "query":
        return {"rel": 0.01, "max": 0.1}
    return {"rel": 0.01, "max": 0.1}


# ------------------------------------------------- the same in 64 bits

def _encode64(raw):
    x = raw[:, :3].double()
    cols = []
    for f in range(12):
        for a in range(3):
            if len(cols) < 64:
                arg = math.pi * 2.0 ** f * x[:, a]
                cols += [torch.sin(arg), torch.cos(arg)]
    return torch.cat([torch.stack(cols, 1), raw[:, 3:13].double(),
                      torch.zeros((len(raw), ENC - ENC_USED), dtype=torch.float64, device=raw.device)], 1)


def _forward64(ws, raw):
    h = _encode64(raw)
    for w in ws[:-1]:
        h = torch.relu(h @ w)
    return (h @ ws[-1])[:, :OUT]


def _exact_trace(case, seed):
    """brute force over all triangles; hits decided in 64 bits"""
    if case["scene"] in ("readme", "textured") or case["any_hit"] or _prims(case) * case["rays"] > 2e9:
        return None
    sc, cam = _scene(case, seed, 640, 360)
    box = type("Box", (), {})()  # the corners the rays are drawn in: the bounds of all primitives
    tri = sc.positions[sc.indices]
    box.info = type("Info", (), {"world_min": list(tri.min((0, 1))), "world_max": list(tri.max((0, 1)))})()
    rays = _rays(case, seed, box, cam).double()
    p = torch.from_numpy(tri.astype(np.float64)).to("cuda")
    e1, e2 = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    best = torch.zeros((len(rays), 3), dtype=torch.float64, device="cuda")
    for i in range(0, len(rays), max(1, int(2e7 // len(p)))):
        r = rays[i:i + max(1, int(2e7 // len(p)))]
        o, d = r[:, None, 0:3], r[:, None, 4:7]
        pv = torch.linalg.cross(d.expand(-1, len(p), -1), e2[None].expand(len(r), -1, -1))
        inv = 1.0 / (e1[None] * pv).sum(2)
        tv = o - p[None, :, 0]
        u = (tv * pv).sum(2) * inv
        qv = torch.linalg.cross(tv, e1[None].expand(len(r), -1, -1))
        v = (d * qv).sum(2) * inv
        t = (e2[None] * qv).sum(2) * inv
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= r[:, None, 3]) & (t <= r[:, None, 7])
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        k = t.argmin(1, keepdim=True)
        found = torch.cat([t.gather(1, k), u.gather(1, k), v.gather(1, k)], 1)
        best[i:i + len(r)] = torch.where(torch.isfinite(found[:, :1]), found, torch.zeros_like(found))
    return {"prim": None, "t": best[:, 0], "uv": best[:, 1:]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "trace":
        return _exact_trace(case, seed)
    if kind not in ("query", "train"):
        return None  # films have no 64-bit counterpart: each path's course depends on its roundings
    ws = [torch.from_numpy(w).to("cuda").double() for w in _weights(case["net"], seed)]
    n = case["rows"]
    if kind == "query":
        raw, _ = _rows(n, seed)
        return torch.cat([_forward64(ws, raw[i:i + 262144]) for i in range(0, n, 262144)])
    raw, target = _rows(n * case["steps"], seed)
    m, v = [torch.zeros_like(w) for w in ws], [torch.zeros_like(w) for w in ws]
    loss = 0.0
    for s in range(case["steps"]):
        for w in ws:
            w.requires_grad_(True)
        y = _forward64(ws, raw[n * s:n * (s + 1)])
        t = target[n * s:n * (s + 1)].double()
        value = ((y - t) ** 2 / (y.detach() ** 2 + 0.01)).mean()
        grads = torch.autograd.grad(value, ws)
        loss = float(value)
        with torch.no_grad():
            for k, g in enumerate(grads):
                if k == len(ws) - 1:
                    g[:, OUT:] = 0
                m[k] = 0.9 * m[k] + 0.1 * g
                v[k] = 0.99 * v[k] + 0.01 * g * g
                step = (m[k] / (1 - 0.9 ** (s + 1))) / (torch.sqrt(v[k] / (1 - 0.99 ** (s + 1))) + 1e-8)
                ws[k] = (ws[k] - 1e-3 * step).detach()
    return {"weights": torch.cat([w.reshape(-1) for w in ws]), "loss": loss}
