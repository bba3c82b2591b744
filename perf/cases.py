"""Workloads of the path-trace library, one pass at a time, for timing.

Each case is one call (or the few calls of one frame) that a program makes
through the binding in `snake-vk_amd/snkpt.py`, on the scenes that the library
generates: the 4k-triangle room (1; 4 at 1080p), the 1.02M-triangle field of
spheres (2), the room with 10,000 emissive triangles (3) and the 16 rooms of
11k-1.74M triangles of the batched workload (5).

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) what the program holds before the call, on the GPU
    run(state)          one pass; its outputs
    work(case)          bytes and operations one pass cannot do without
    exact(case, seed)   run's outputs in 64 bits, where they have such a value
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "snake-vk_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import raysets  # noqa: E402
import snkpt  # noqa: E402

# triangles, rays per pixel of a path-traced frame at the scene's own depth
# (camera, extension and shadow rays), nodes and triangles an average ray visits
SCENES = {1: (4004, 5.7, 8.0, 2.0), 2: (1024002, 2.3, 12.2, 2.25), 3: (14004, 1.4, 9.0, 2.0),
          4: (4004, 3.2, 8.0, 2.0)}
TRIS5 = (286260, 11060, 24684, 116316, 358836, 1713516, 75660, 310284, 1739796, 180660, 152916, 16164, 693924, 29276,
         294884, 148260)


def listed():
    return [
        # a particle system's collision rays against the room: the smallest call, latency counts
        {"name": "contacts_room_16k", "kind": "contacts", "scene": 1, "variant": 0, "n": 16384},
        # the library's headline: one cosine bounce per primary hit of a 1080p frame, closest hit with barycentrics
        {"name": "bounce_rays_1080p", "kind": "trace", "scene": 2, "variant": 0, "w": 1920, "h": 1080, "any": False},
        # shadow rays of an oddly sized viewport
        {"name": "shadow_rays_1283x717", "kind": "trace", "scene": 2, "variant": 0, "w": 1283, "h": 717, "any": True},
        # a preview frame: few pixels, so launches and the readback count
        {"name": "frame_room_256", "kind": "frame", "scene": 1, "variant": 0, "w": 256, "h": 256, "depth": 4, "rr": 0,
         "gbuffer": False, "half": False, "accumulate": False},
        # a full frame of the large scene with Russian roulette
        {"name": "frame_million_1080p", "kind": "frame", "scene": 2, "variant": 0, "w": 1920, "h": 1080, "depth": 8,
         "rr": 3, "gbuffer": False, "half": False, "accumulate": False},
        # the renderer's own form: rasterised G-buffer in, accumulated RGBA16F image out
        {"name": "frame_gbuffer_1080p", "kind": "frame", "scene": 4, "variant": 0, "w": 1920, "h": 1080, "depth": 8,
         "rr": 3, "gbuffer": True, "half": True, "accumulate": True},
        # ReSTIR direct light of 10,000 emitters along the camera's orbit, then the temporal resolve
        {"name": "restir_taa_1080p", "kind": "restir", "scene": 3, "variant": 0, "w": 1920, "h": 1080, "spatial": 5,
         "candidates": 32},
        # a radiance-cache frame: NEE + BRDF probe at the primary hit, the network for the rest, one training step
        {"name": "cache_room_1080p", "kind": "cache", "scene": 4, "variant": 0, "w": 1920, "h": 1080, "paths": 32768,
         "mis": True},
        # 64 views of 16 scenes in one replayed graph: the largest call
        {"name": "batch_64_views", "kind": "batch", "scenes": 16, "first": 0, "per_scene": 4, "scale": 1.0},
        # a dynamic scene: new transforms, the acceleration structure built again, a frame's camera rays traced
        {"name": "rebuild_million", "kind": "rebuild", "scene": 2, "variant": 0, "w": 1280, "h": 720},
        # the network alone, serving: a million queries
        {"name": "cache_infer_1m", "kind": "infer", "n": 1000003},
        # the network alone, training: one optimiser step, then the new network asked
        {"name": "cache_train_64k", "kind": "train", "n": 65536, "probe": 4096},
    ]


def _log(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))


def draw(rng):
    kind = rng.choice(["contacts", "trace", "trace", "frame", "frame", "restir", "cache", "batch", "rebuild", "infer",
                       "train"])
    if kind == "contacts":
        return {"kind": kind, "scene": rng.choice([1, 2]), "variant": 0, "n": _log(rng, 1000, 2000000)}
    if kind == "infer":
        return {"kind": kind, "n": _log(rng, 1000, 1000000)}
    if kind == "train":
        return {"kind": kind, "n": _log(rng, 4096, 131072), "probe": _log(rng, 256, 16384)}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 8), "first": rng.randint(0, 8), "per_scene": rng.randint(1, 4),
                "scale": round(rng.uniform(0.5, 1.0), 3)}
    w, h = _log(rng, 96, 1920), _log(rng, 64, 1080)
    if kind == "restir":
        return {"kind": kind, "scene": 3, "variant": 0, "w": w, "h": h, "spatial": rng.randint(1, 5),
                "candidates": rng.choice([8, 16, 32])}
    if kind == "cache":
        return {"kind": kind, "scene": 4, "variant": 0, "w": w, "h": h, "paths": _log(rng, 4096, 65536),
                "mis": rng.random() < 0.5}
    scene = rng.choice([1, 2, 5, 5])
    case = {"kind": kind, "scene": scene, "variant": rng.randint(0, 15) if scene == 5 else 0, "w": w, "h": h}
    if kind == "trace":
        return {**case, "any": rng.random() < 0.5}
    if kind == "rebuild":
        return case
    return {**case, "depth": rng.randint(2, 8), "rr": rng.choice([0, 3]), "gbuffer": rng.random() < 0.3,
            "half": rng.random() < 0.3, "accumulate": rng.random() < 0.3}


# ---------------------------------------------------------------- scenes ----
@functools.lru_cache(maxsize=None)
def _scene(config, variant):
    """The scene's host arrays: loaded assets, the same for every seed."""
    return snkpt.SceneData(config, variant)


def _context(config, variant):
    ctx = snkpt.Context(0)
    ctx.load_scene(_scene(config, variant))
    ctx.build_accel()
    return ctx


def _camera(scene, frame, w, h, rng):
    """The scene's camera moved by up to 0.5 % of its distance from the origin."""
    cam = scene.camera(frame, w, h)
    view = np.array(cam.view, np.float64).reshape(4, 4).T
    proj = np.array(cam.proj, np.float64).reshape(4, 4).T
    pos = np.array(cam.cam_pos[:3], np.float64)
    d = rng.uniform(-1.0, 1.0, 3) * 0.005 * np.linalg.norm(pos)
    move = np.eye(4)
    move[:3, 3] = -d
    view = view @ move
    for k, v in enumerate(view.T.reshape(-1)):
        cam.view[k] = v
    for k, v in enumerate((proj @ view).T.reshape(-1)):
        cam.proj_view[k] = v
    for a in range(3):
        cam.cam_pos[a] = pos[a] + d[a]
    return cam


def _primary_rays(cam, w, h):
    m = torch.from_numpy(raysets.camera_matrix(cam)).cuda()
    ys, xs = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float64),
                            torch.arange(w, device="cuda", dtype=torch.float64), indexing="ij")
    one = torch.ones_like(xs)
    clip = torch.stack([(xs + 0.5) / w * 2 - 1, (ys + 0.5) / h * 2 - 1, one, one], -1).reshape(-1, 4)
    p = clip @ m.T
    o = torch.tensor(list(cam.cam_pos[:3]), dtype=torch.float64, device="cuda")
    d = p[:, :3] / p[:, 3:4].clamp_min(1e-6) - o
    d = d / d.norm(dim=1, keepdim=True)
    org = torch.zeros(w * h, 4, device="cuda")
    org[:, :3] = o.float()
    dirs = torch.full((w * h, 4), 1e30, device="cuda")
    dirs[:, :3] = d.float()
    return org, dirs


def _world(ctx, scene):
    """(T, 12) world triangles, the first triangle of each instance and the scene's largest extent."""
    tris = torch.from_numpy(np.frombuffer(ctx.export(6).tobytes(), np.float32).reshape(-1, 12).copy()).cuda()
    inst = scene.arrays()[2]
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(inst[:, 4] // 3)]).astype(np.int64)).cuda()
    v = tris[:, :9].reshape(-1, 3)
    return tris, off, float((v.max(0).values - v.min(0).values).max())


def _emitters(scene, tris, off):
    em = np.ctypeslib.as_array(scene.s.emissive_instances, (scene.s.n_emissive,)).astype(np.int64)
    ends = off.cpu().numpy()
    ids = torch.from_numpy(np.concatenate([np.arange(ends[i], ends[i + 1]) for i in em])).cuda()
    t = tris[ids, :9]
    area = torch.linalg.cross(t[:, 3:6] - t[:, 0:3], t[:, 6:9] - t[:, 0:3]).norm(dim=1)
    return t, area / area.sum()


def _gbuffer(ctx, scene, cam, w, h):
    """The G-buffer images of RaytracingResources, from traced camera rays."""
    org, dirs = _primary_rays(cam, w, h)
    t, inst, prim, _, _ = ctx.trace(org, dirs)
    tris, off, _ = _world(ctx, scene)
    hit = t >= 0
    ii = torch.where(hit, inst, torch.zeros_like(inst)).long()
    tri = tris[off[ii] + torch.where(hit, prim, torch.zeros_like(prim)).long()]
    v0, v1, v2 = tri[:, 0:3], tri[:, 3:6], tri[:, 6:9]
    n = torch.linalg.cross(v1 - v0, v2 - v0)
    n = n / n.norm(dim=1, keepdim=True).clamp_min(1e-30)
    d3 = dirs[:, :3]
    n = torch.where(((n * d3).sum(1) > 0)[:, None], -n, n)
    pv = torch.tensor(np.array(cam.proj_view, np.float32).reshape(4, 4).T.copy()).cuda()
    clip = (org[:, :3] + d3 * t[:, None]) @ pv[:, :3].T + pv[:, 3]
    one = torch.ones_like(t)
    _, _, inst5, _, mats = scene.arrays()
    mi = torch.from_numpy(inst5[:, 3].astype(np.int64)).cuda()[ii]
    m = torch.from_numpy(mats.view(np.float32).copy()).cuda()[mi]
    flags = torch.from_numpy(mats[:, 12].astype(np.int32)).cuda()[mi]
    albedo = torch.cat([torch.round(m[:, 8:11].clamp(-1, 1) * 127.0), 127.0 * one[:, None]], 1)
    return {"depth": torch.where(hit, clip[:, 2] / clip[:, 3], one).reshape(h, w).contiguous(),
            "normal": torch.cat([n, one[:, None]], 1).half().reshape(h, w, 4).contiguous(),
            "albedo": albedo.to(torch.int8).reshape(h, w, 4).contiguous(),
            "rma": torch.stack([m[:, 5], m[:, 6], one, one], 1).half().reshape(h, w, 4).contiguous(),
            "mat_flags": torch.where(hit, flags, torch.zeros_like(flags)).to(torch.int16).reshape(h, w).contiguous()}


# --------------------------------------------------------------- network ----
LO, HI = (-1.0, 0.0, -1.0), (1.0, 2.0, 1.0)


def _samples(n, seed):
    """Points of the room with unit directions and normals, materials, and a smooth radiance as target."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    s = torch.zeros(n, 16, device="cuda")
    lo, hi = torch.tensor(LO, device="cuda"), torch.tensor(HI, device="cuda")
    x = lo + (hi - lo) * torch.rand(n, 3, device="cuda", generator=g)
    d = torch.randn(n, 3, device="cuda", generator=g)
    nn = torch.randn(n, 3, device="cuda", generator=g)
    s[:, 0:3] = x
    s[:, 3:6] = d / d.norm(dim=1, keepdim=True)
    s[:, 6:9] = nn / nn.norm(dim=1, keepdim=True)
    s[:, 9] = 0.05 + 0.95 * torch.rand(n, device="cuda", generator=g)
    s[:, 10:13] = 0.1 + 0.8 * torch.rand(n, 3, device="cuda", generator=g)
    base = 0.5 + 0.4 * torch.sin(3 * x[:, 0]) * torch.cos(2 * x[:, 2]) + 0.2 * x[:, 1]
    s[:, 13] = base
    s[:, 14] = 0.8 * base + 0.1 * s[:, 3]
    s[:, 15] = 0.6 * base + 0.1 * s[:, 11]
    return s


def _weights(seed):
    """A network as training leaves one: Glorot-scaled layers, grid features of some tenths."""
    rng = np.random.default_rng(seed)
    mlp = np.zeros(snkpt.CACHE_MLP_PARAMS, np.float32)
    for k in range(4):
        mlp[4096 * k:4096 * (k + 1)] = rng.uniform(-1, 1, 4096) * math.sqrt(6.0 / 128)
    mlp[16384:16384 + 192] = rng.uniform(-1, 1, 192) * math.sqrt(6.0 / 67)
    grid = rng.random(snkpt.CACHE_GRID_PARAMS, dtype=np.float32)
    grid -= 0.5
    grid *= 0.6
    return mlp, grid


def _network(seed):
    ctx = snkpt.Context(0)
    ctx.cache_reset(1 + seed % 1000, LO, HI)
    mlp, grid = _weights(seed)
    ctx.cache_set_params(0, mlp)
    ctx.cache_set_params(1, grid)
    return ctx


def _encode64(grid, s):
    """The 64 network inputs of samples `s` (float64)."""
    inv = 1.0 / max(b - a for a, b in zip(LO, HI))
    p = ((s[:, 0:3] - torch.tensor(LO, dtype=torch.float64, device=s.device)) * inv).clamp(0, 1)
    x = torch.zeros(s.shape[0], 64, dtype=torch.float64, device=s.device)
    b = math.exp((math.log(2048.0) - math.log(16.0)) / 15)
    for lv in range(16):
        r = math.floor(16.0 * b ** lv + 1e-6)
        q = p * r
        c = q.floor().clamp_max(r - 1)
        f, c = q - c, c.long()
        for k in range(8):
            bit = [k & 1, (k >> 1) & 1, k >> 2]
            w = torch.ones_like(f[:, 0])
            for a in range(3):
                w = w * (f[:, a] if bit[a] else 1 - f[:, a])
            i, j, m = (c[:, a] + bit[a] for a in range(3))
            if (r + 1) ** 3 <= 1 << 19:
                at = i + j * (r + 1) + m * (r + 1) ** 2
            else:
                at = (i ^ (j * 2654435761) ^ (m * 805459861)) & ((1 << 19) - 1)
            x[:, 2 * lv:2 * lv + 2] += w[:, None] * grid[lv, at].double()
    x[:, 32:38] = 0.5 * (s[:, 3:9] + 1)
    x[:, 38:42] = s[:, 9:13]
    x[:, 42:54:2] = torch.sin(math.pi * s[:, 3:9])
    x[:, 43:54:2] = torch.cos(math.pi * s[:, 3:9])
    return x


def _network64(seed, samples):
    """The network's three outputs for `samples`, in 64 bits."""
    mlp, grid = _weights(seed)
    grid = torch.from_numpy(grid).to(samples.device).view(16, 1 << 19, 2)
    w = torch.from_numpy(mlp).to(samples.device).double()
    out = []
    for s in samples.double().split(1 << 17):
        x = _encode64(grid, s)
        for k in range(4):
            x = (x @ w[4096 * k:4096 * (k + 1)].view(64, 64).T.contiguous()).clamp_min(0)
        out.append(x @ w[16384:16384 + 192].view(3, 64).T.contiguous())
    return torch.cat(out)


# ------------------------------------------------------------------ cases ----
def _settings(case, st, **kw):
    st["frame"] += 1
    return snkpt.default_settings(seed=st["seed"], frame=st["frame"] - 1, **kw)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    st = {"kind": kind, "case": case, "seed": 1 + seed % 0x7FFFFFFF, "frame": 0}
    if kind in ("infer", "train"):
        st["ctx"] = _network(seed)
        st["samples"] = _samples(case["n"], seed)
        if kind == "train":
            st["probe"] = _samples(case["probe"], seed + 1)
        return st
    if kind == "batch":
        st["batch"], st["stream"] = snkpt.Batch(0), torch.cuda.Stream()
        st["outs"] = []
        for k in range(case["scenes"]):
            var = (case["first"] + k) % 16
            sid = st["batch"].add_scene(_context(5, var))
            for v in range(case["per_scene"]):
                _, w, h = snkpt.scene_view(5, 4 * var + v)
                w, h = max(64, int(w * case["scale"])), max(64, int(h * case["scale"]))
                out = torch.zeros(h, w, 4, device="cuda")
                st["batch"].add_view(sid, _camera(_scene(5, var), 4 * var + v, w, h, rng), w, h,
                                     st["seed"] + 4 * var + v, out)
                st["outs"].append(out)
        torch.cuda.synchronize()
        return st
    scene = _scene(case["scene"], case["variant"])
    ctx = st["ctx"] = _context(case["scene"], case["variant"])
    if kind == "contacts":
        n = case["n"]
        info = ctx.accel_info()
        lo = torch.tensor(list(info.scene_lo), device="cuda")
        hi = torch.tensor(list(info.scene_hi), device="cuda")
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        r = 0.01 + 0.07 * torch.rand(n, 1, device="cuda", generator=g)
        d = torch.randn(n, 3, device="cuda", generator=g)
        d = d / d.norm(dim=1, keepdim=True)
        p = lo + (hi - lo) * torch.rand(n, 3, device="cuda", generator=g)
        speed = 30.0 * torch.rand(n, 1, device="cuda", generator=g)
        st["org"] = torch.cat([p - d * r, torch.zeros_like(r)], 1).contiguous()
        st["dir"] = torch.cat([d, speed / 120.0 + 2 * r], 1).contiguous()
        m4 = np.array(scene.arrays()[3], np.float32)
        m4[1:, 12] += 0.01  # last frame's transforms: everything but the ground moved
        ctx.set_prev_transforms(m4)
        return st
    w, h = case["w"], case["h"]
    cam = st["cam"] = _camera(scene, 0, w, h, rng)
    if kind == "trace":
        org, dirs = _primary_rays(cam, w, h)
        t, inst, prim, _, _ = ctx.trace(org, dirs)
        tris, off, ext = _world(ctx, scene)
        if case["any"]:
            st["org"], st["dir"] = raysets.shadow_rays_torch(org, dirs, t, *_emitters(scene, tris, off), seed=seed,
                                                             scale=ext)
        else:
            st["org"], st["dir"] = raysets.secondary_rays_torch(org, dirs, t, inst, prim, tris, off, ext, seed=seed)
        # one size for every seed: as many rays as a view of the scene usually hits, spread evenly over the hits
        n = _traced(case)
        at = torch.arange(n, device="cuda") * st["org"].shape[0] // n
        st["org"], st["dir"] = st["org"][at].contiguous(), st["dir"][at].contiguous()
        return st
    if kind == "rebuild":
        st["org"], st["dir"] = _primary_rays(cam, w, h)
        _, _, st["inst"], m4, _ = (np.array(a) for a in scene.arrays())
        st["moved"] = []
        for _ in range(8):
            m = np.array(m4, np.float32)
            m[1:, 12:15] += rng.uniform(-0.05, 0.05, (m.shape[0] - 1, 3)).astype(np.float32)
            st["moved"].append(m)
        return st
    st["out"] = torch.zeros(h, w, 4, device="cuda", dtype=torch.float16 if case.get("half") else torch.float32)
    if kind == "frame" and case["gbuffer"]:
        st["gbuffer"] = _gbuffer(ctx, scene, cam, w, h)
    if kind == "restir":
        st["scene"] = scene
        st["image"] = torch.zeros(h, w, 4, device="cuda")
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        coarse = torch.randn(1, 2, 9, 9, device="cuda", generator=g)
        flow = torch.nn.functional.interpolate(coarse, size=(h, w), mode="bilinear", align_corners=True)[0]
        st["motion"] = (flow.permute(1, 2, 0) * (1.0 / w)).half().contiguous()  # about a pixel
    if kind == "cache":
        ctx.cache_reset(1 + seed % 1000)
    return st


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "batch":
        s = _settings(case, st, mode=snkpt.MODE_PT, max_depth=6, rr_start=3)
        st["batch"].render(s, use_graph=True, stream=st["stream"])
        return st["outs"]
    ctx = st["ctx"]
    if kind == "infer":
        return ctx.cache_infer(st["samples"])
    if kind == "train":
        loss = ctx.cache_train(st["samples"], lr=2.5e-3)
        return {"loss": loss, "mlp": ctx.cache_params(0), "radiance": ctx.cache_infer(st["probe"])}
    if kind == "contacts":
        return ctx.trace_contacts(st["org"], st["dir"])
    if kind == "trace":
        if case["any"]:
            return ctx.trace(st["org"], st["dir"], any_hit=True, with_uv=False)[:3]
        return ctx.trace(st["org"], st["dir"])
    if kind == "rebuild":
        ctx.set_instances(st["inst"], st["moved"][st["frame"] % len(st["moved"])])
        ctx.build_accel()
        st["frame"] += 1
        return ctx.trace(st["org"], st["dir"])
    w, h, out = case["w"], case["h"], st["out"]
    if kind == "frame":
        s = _settings(case, st, max_depth=case["depth"], rr_start=case["rr"])
        if case["accumulate"]:
            s.flags |= snkpt.FLAG_ACCUMULATE
        fmt = snkpt.FORMAT_RGBA16F if case["half"] else snkpt.FORMAT_RGBA32F
        if case["gbuffer"]:
            ctx.render_gbuffer(st["cam"], s, st["gbuffer"], out, w, h, fmt)
        else:
            ctx.render(st["cam"], s, out, w, h, fmt)
    elif kind == "restir":
        s = _settings(case, st, mode=snkpt.MODE_RESTIR, max_depth=1, num_spatial_resamples=case["spatial"],
                      restir_candidates=case["candidates"])
        ctx.render(st["scene"].camera(s.frame % 64, w, h), s, st["image"], w, h)
        ctx.taa_resolve(st["image"], out, st["motion"], w, h, reset=s.frame == 0)
    else:
        s = _settings(case, st, mode=snkpt.MODE_CACHE, max_depth=8, rr_start=3, cache_query_depth=1,
                      cache_train_paths=case["paths"], cache_lr=2.5e-3, cache_ema=0.0,
                      flags=snkpt.FLAG_CACHE_INDIRECT | snkpt.FLAG_CACHE_TRAIN_AT_QUERY |
                      (snkpt.FLAG_CACHE_MIS if case["mis"] else 0))
        ctx.render(st["cam"], s, out, w, h)
    return out


# ------------------------------------------------------------------- work ----
def _tris(case):
    return TRIS5[case["variant"]] if case["scene"] == 5 else SCENES[case["scene"]][0]


def _traced(case):
    return max(1, int(case["w"] * case["h"] * (0.6 if case["scene"] == 2 else 0.9)))


def _ray_flops(nodes, tris):
    return nodes * 8 * 6 * 2 + tris * 60  # six fused slab planes of eight boxes, a watertight triangle test


def work(case):
    kind = case["kind"]
    if kind in ("infer", "train"):
        n = case["n"]
        mlp = 2.0 * (4 * 64 * 64 + 64 * 16)
        grid = 32.0 * (1 << 20)
        if kind == "infer":  # sample read, radiance written, each grid entry read once at most
            return {"bytes": 68.0 * n + min(grid, 512.0 * n), "flops": (mlp + 16 * 8 * 8) * n}
        touched = min(8.4e6, 128.0 * n)  # grid entries with a gradient: masters, moments and copies read and written
        return {"bytes": 64.0 * n + 72.0 * touched, "flops": 3 * mlp * n + mlp * case["probe"]}
    if kind == "batch":
        px = tris = 0
        for k in range(case["scenes"]):
            var = (case["first"] + k) % 16
            tris += TRIS5[var]
            for v in range(case["per_scene"]):
                _, w, h = snkpt.scene_view(5, 4 * var + v)
                px += max(64, int(w * case["scale"])) * max(64, int(h * case["scale"]))
        return {"bytes": 16.0 * px + 66.0 * tris, "flops": 4.6 * px * _ray_flops(10, 2)}
    tris = _tris(case)
    nodes, per = (10.0, 2.0) if case["scene"] == 5 else SCENES[case["scene"]][2:]
    scene_bytes = 66.0 * tris  # leaf records of 48 B, a node of 80 B for four to five triangles
    if kind == "contacts":
        return {"bytes": 92.0 * case["n"] + min(scene_bytes, 300.0 * case["n"]),
                "flops": case["n"] * _ray_flops(3, 1)}
    px = case["w"] * case["h"]
    if kind == "trace":
        n = _traced(case)
        return {"bytes": (44.0 if case["any"] else 52.0) * n + min(scene_bytes, 1100.0 * n),
                "flops": n * _ray_flops(nodes, per)}
    if kind == "rebuild":  # vertices and indices read, world and leaf triangles and nodes written; rays traced
        return {"bytes": tris * (48.0 + 48.0 + 48.0 + 18.0) + 52.0 * px, "flops": px * _ray_flops(nodes, per)}
    if kind == "frame":
        rays = 4.6 if case["scene"] == 5 else SCENES[case["scene"]][1]
        b = (8.0 if case["half"] else 16.0) + (32.0 if case["accumulate"] else 0.0) + (26.0 if case["gbuffer"] else 0.0)
        return {"bytes": b * px + scene_bytes, "flops": rays * px * _ray_flops(nodes, per)}
    if kind == "restir":
        # image, history and motion; two reservoirs and G-buffers of history; 64 B of one emitter per candidate
        return {"bytes": (16 + 76 + 2 * 100) * px + 0.64e6,
                "flops": px * (1.4 * _ray_flops(nodes, per) + (case["candidates"] + 6 * case["spatial"]) * 100.0)}
    return {"bytes": 16.0 * px + scene_bytes + 32.0 * (1 << 20) + 72.0 * min(8.4e6, 128.0 * case["paths"]),
            "flops": 0.56 * px * (3 * _ray_flops(nodes, per) + 34816.0) + 3 * 34816.0 * case["paths"]}


# ------------------------------------------------------------------ exact ----
def _world64(scene):
    """World triangles (T, 3, 3) of the scene's arrays, in 64 bits."""
    pos, idx, inst, m4, _ = scene.arrays()
    out = []
    for xf, i0, v0, _, n in np.asarray(inst, np.int64):
        v = np.asarray(pos, np.float64)[np.asarray(idx[i0:i0 + n], np.int64) + v0]
        m = np.asarray(m4[xf], np.float64).reshape(4, 4).T
        out.append((v @ m[:3, :3].T + m[:3, 3]).reshape(-1, 3, 3))
    return torch.from_numpy(np.concatenate(out)).cuda()


def _closest64(tris, org, dirs):
    """t of the closest hit of every ray, -1 where there is none (both faces; Moeller and Trumbore 1997)."""
    a, e1, e2 = tris[:, 0], tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0]
    n = torch.linalg.cross(e1, e2)
    best = []
    for o, d in zip(org.double().split(max(1, (1 << 25) // tris.shape[0])),
                    dirs.double().split(max(1, (1 << 25) // tris.shape[0]))):
        # det = -d.n, t = (o - a).n / det, u = (d x (o - a)).e2 ..., as products over all pairs
        det = -(d[:, :3] @ n.T)
        t = (o[:, :3] @ n.T - (a * n).sum(1)) / det
        # w = d x (o - a): w.e2 = d.((o - a) x e2) = (d x o).e2 - d.(a x e2)
        w = torch.linalg.cross(d[:, :3], o[:, :3])
        u = (w @ e2.T - d[:, :3] @ torch.linalg.cross(a, e2).T) / -det
        v = (w @ e1.T - d[:, :3] @ torch.linalg.cross(a, e1).T) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t >= o[:, 3:]) & (t <= d[:, 3:])
        t = torch.where(ok, t, torch.full_like(t, math.inf)).min(1).values
        best.append(torch.where(t.isfinite(), t, torch.full_like(t, -1.0)))
    return torch.cat(best)


def exact(case, seed):
    kind = case["kind"]
    if kind == "infer":
        y = _network64(seed, _samples(case["n"], seed))
        return torch.cat([y, torch.zeros_like(y[:, :1])], 1)
    if kind == "train":
        s = _samples(case["n"], seed)
        y = _network64(seed, s)
        loss = ((y - s[:, 13:16].double()) ** 2 / (y * y + 0.01)).mean()
        # the step itself divides each gradient by its own size: a value near zero has no stable sign
        return {"loss": float(loss), "mlp": None, "radiance": None}
    if kind == "trace" and not case["any"] and case["w"] * case["h"] * _tris(case) <= 8e9:
        st = prepare(case, seed)
        return [_closest64(_world64(_scene(case["scene"], case["variant"])), st["org"], st["dir"]), None, None, None,
                None]
    # frames are random walks whose later choices follow the roundings of the earlier ones, an any-hit ray
    # returns whichever occluder it meets first, and the rest would take minutes without a tree
    return None
