"""GPU parity: the HIP LBVH->BVH8 build is bit-exact against the CPU twin, and
HIP traversal returns bit-identical hits (and visit counts) to the CPU BVH8
traversal, which itself matches brute force."""
import sys

import numpy as np
import pytest

from helpers import as_bits, assert_bits_equal, gpu_trace, make_ctx, scene_world, tri_soup_ctx
from oracle import binding as O

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _compare_build(ctx, world):
    b = O.Bvh(world)
    info = ctx.accel_info()
    assert info.num_triangles == b.n
    assert info.num_nodes == b.num_nodes, (info.num_nodes, b.num_nodes)
    assert info.depth == b.depth and info.binary_depth == b.binary_depth
    assert_bits_equal(ctx.export(6), world.reshape(-1), "world triangles")
    assert_bits_equal(ctx.export(0), b.keys, "sorted Morton keys")
    assert_bits_equal(ctx.export(1), b.ids, "sorted triangle ids")
    if b.n >= 2:
        assert_bits_equal(ctx.export(2), b.child, "radix-tree children")
        assert_bits_equal(ctx.export(7), b.leafify, "leaf-cluster flags")
    assert_bits_equal(ctx.export(3), b.aabb, "binary boxes")
    assert_bits_equal(ctx.export(4), b.nodes, "BVH8 nodes")
    assert_bits_equal(ctx.export(5), b.leaf, "leaf triangles")
    return b


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7, 64, 1000])
def test_build_bitexact_random_soup(gpu, n):
    _say(f"build soup n={n}")
    rng = np.random.default_rng(100 + n)
    pos = rng.uniform(-5, 5, (3 * n, 3)).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32)
    ctx = tri_soup_ctx(pos, idx)
    world = O.flatten(pos, idx, np.array([[0, 0, 0, 0, 3 * n]], np.uint32), np.eye(4, dtype=np.float32))
    b = _compare_build(ctx, world)
    import raysets
    org, dr = raysets.random_rays(4096, [-5] * 3, [5] * 3, seed=n)
    rays = np.concatenate([org, dr], 1)
    g = gpu_trace(ctx, rays)
    c = b.trace(rays)
    for k, name in enumerate(["t", "inst", "prim", "u", "v", "nodes visited", "tris visited"]):
        assert_bits_equal(g[k], c[k], name)


def test_build_bitexact_duplicate_keys(gpu):
    """Many triangles with identical Morton codes exercise the index tie-break."""
    _say("build duplicate keys")
    rng = np.random.default_rng(3)
    base = rng.uniform(0, 1, (3, 3)).astype(np.float32)
    pos = np.concatenate([base + np.float32(1e-7) * k for k in range(300)] +
                         [rng.uniform(0, 1, (300, 3)).astype(np.float32)])
    idx = np.arange(pos.shape[0], dtype=np.uint32)
    ctx = tri_soup_ctx(pos, idx)
    world = O.flatten(pos, idx, np.array([[0, 0, 0, 0, idx.size]], np.uint32), np.eye(4, dtype=np.float32))
    _compare_build(ctx, world)


def test_empty_scene_all_miss(gpu):
    import snkpt
    ctx = snkpt.Context(0)
    ctx.set_instances(np.zeros((0, 5), np.uint32), np.eye(4, dtype=np.float32).reshape(1, 16))
    ctx.set_materials([])
    ctx.set_lights(None, None)
    ctx.build_accel()
    assert ctx.accel_info().num_triangles == 0
    rays = np.zeros((100, 8), np.float32)
    rays[:, 4] = 1.0
    rays[:, 7] = 1e30
    t, inst, prim, u, v, nv, tv = gpu_trace(ctx, rays)
    assert (t == -1).all() and (inst.view(np.uint32) == 0xFFFFFFFF).all()


def test_room_build_and_trace_parity(gpu):
    import raysets
    import snkpt
    _say("room: build")
    scene = snkpt.SceneData(1)
    ctx = make_ctx(scene)
    world = scene_world(scene)
    b = _compare_build(ctx, world)
    lo, hi = world[:, :9].reshape(-1, 3).min(0), world[:, :9].reshape(-1, 3).max(0)
    org, dr = raysets.random_rays(50000, lo, hi, seed=9)
    porg, pdr = raysets.primary_rays(scene.camera(0, 128, 128), 128, 128)
    rays = np.concatenate([np.concatenate([org, dr], 1), np.concatenate([porg, pdr], 1)])
    # tmin/tmax windows as the reference uses them (RayGen.rgen:172-174, :114-116)
    rays[::7, 3] = 0.01
    rays[::7, 7] = 1000.0
    rays[1::7, 3] = 0.001
    rays[1::7, 7] = 0.5
    _say("room: closest hit")
    g = gpu_trace(ctx, rays)
    c = b.trace(rays)
    for k, name in enumerate(["t", "inst", "prim", "u", "v", "nodes visited", "tris visited"]):
        assert_bits_equal(g[k], c[k], name)
    w = O.trace_brute(world, rays)
    for k, name in enumerate(["t", "inst", "prim", "u", "v"]):
        assert_bits_equal(g[k], w[k], name + " vs brute force")
    _say("room: any hit")
    ga = gpu_trace(ctx, rays, any_hit=True)
    ca = b.trace(rays, any_hit=True)
    for k, name in enumerate(["t", "inst", "prim", "u", "v", "nodes visited", "tris visited"]):
        assert_bits_equal(ga[k], ca[k], "any-hit " + name)
    assert np.array_equal(ga[0] >= 0, w[0] >= 0)


def test_axis_parallel_and_grazing_rays(gpu):
    import snkpt
    scene = snkpt.SceneData(1)
    ctx = make_ctx(scene)
    world = scene_world(scene)
    b = O.Bvh(world)
    rng = np.random.default_rng(4)
    n = 6000
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = rng.uniform(-1.2, 1.2, (n, 3)) + np.array([0, 1, 0])
    axis = rng.integers(0, 3, n)
    sign = rng.choice([-1.0, 1.0], n)
    rays[np.arange(n), 4 + axis] = sign
    # a third of them lie exactly in wall planes (y = 0, x = +-1, z = -1)
    rays[: n // 3, 1] = 0.0
    rays[n // 3: 2 * n // 3, 0] = 1.0
    rays[:, 7] = 1e30
    g = gpu_trace(ctx, rays)
    c = b.trace(rays)
    w = O.trace_brute(world, rays)
    for k, name in enumerate(["t", "inst", "prim", "u", "v"]):
        assert_bits_equal(g[k], c[k], name)
        assert_bits_equal(g[k], w[k], name + " vs brute force")


def test_spheres_1m_build_and_incoherent_parity(gpu):
    """1.02M-triangle scene: bit-exact build; incoherent secondary rays match the
    CPU BVH8 bit for bit and brute force on a subsample."""
    import torch

    import raysets
    import snkpt
    _say("spheres: generate + build")
    scene = snkpt.SceneData(2)
    ctx = make_ctx(scene)
    world = scene_world(scene)
    b = _compare_build(ctx, world)
    _say("spheres: primary + secondary rays")
    w, h = 480, 270
    porg, pdr = raysets.primary_rays(scene.camera(0, w, h), w, h)
    po, pd = torch.from_numpy(porg).cuda(), torch.from_numpy(pdr).cuda()
    t, inst, prim, _, _ = ctx.trace(po, pd)
    inst_np = scene.arrays()[2]
    off = np.concatenate([[0], np.cumsum(inst_np[:, 4] // 3)]).astype(np.int64)
    wt = torch.from_numpy(world[:, :].copy()).cuda()
    so, sd = raysets.secondary_rays_torch(po, pd, t, inst, prim, wt, torch.from_numpy(off).cuda(), 100.0, seed=1)
    rays = torch.cat([so, sd], 1).cpu().numpy()
    assert rays.shape[0] > 0.5 * w * h
    _say(f"spheres: trace {rays.shape[0]} secondary rays")
    g = gpu_trace(ctx, rays)
    c = b.trace(rays)
    for k, name in enumerate(["t", "inst", "prim", "u", "v", "nodes visited", "tris visited"]):
        assert_bits_equal(g[k], c[k], name)
    sub = rays[::64][:1024]
    wb = O.trace_brute(world, sub)
    gs = [x[::64][:1024] for x in g]
    agree = (as_bits(gs[1]) == as_bits(wb[1])) & (as_bits(gs[2]) == as_bits(wb[2]))
    assert agree.mean() >= 0.9999 or (~agree).sum() <= 0, f"{(~agree).sum()} id mismatches vs brute force"
    tt = (gs[0] >= 0)
    rel = np.abs(gs[0][tt] - wb[0][tt]) / np.maximum(np.abs(wb[0][tt]), 1e-30)
    assert rel.max() <= 1e-5


def test_invalid_rays_miss_fast(gpu):
    """NaN / inf / zero-direction / empty-interval rays are immediate misses on
    the GPU too (no full-tree walk), matching the oracle."""
    import time

    import snkpt
    scene = snkpt.SceneData(2)
    ctx = make_ctx(scene)
    rng = np.random.default_rng(0)
    n = 1 << 16
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = rng.uniform(-40, 40, (n, 3))
    d = rng.normal(size=(n, 3))
    rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 7] = 1e30
    bad = rng.choice(n, 64, replace=False)
    rays[bad[:16], 4] = np.nan
    rays[bad[16:32], 1] = np.inf
    rays[bad[32:48], 4:7] = 0.0
    rays[bad[48:], 3] = 5.0
    rays[bad[48:], 7] = 1.0
    g = gpu_trace(ctx, rays)
    assert (g[0][bad] == -1).all() and (g[5][bad] == 0).all()
    import torch
    t0 = time.perf_counter()
    gpu_trace(ctx, rays, counted=False)
    assert time.perf_counter() - t0 < 2.0


def test_parallel_axis_rays_cull_on_gpu(gpu):
    """Vertical and axis-aligned rays on the 1.02M-triangle scene: bit-identical
    to the CPU twin (hits and visit counts) and few nodes visited."""
    import snkpt
    scene = snkpt.SceneData(2)
    ctx = make_ctx(scene)
    world = scene_world(scene)
    b = O.Bvh(world)
    rng = np.random.default_rng(8)
    n = 4096
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0] = rng.uniform(-60, 60, n)
    rays[:, 1] = rng.choice([0.01, 1.0, 5.0, 30.0], n)
    rays[:, 2] = rng.uniform(-60, 60, n)
    axis = rng.integers(0, 3, n)
    rays[np.arange(n), 4 + axis] = rng.choice([-1.0, 1.0], n)
    rays[:, 7] = 1e30
    g = gpu_trace(ctx, rays)
    c = b.trace(rays)
    for k, name in enumerate(["t", "inst", "prim", "u", "v", "nodes visited", "tris visited"]):
        assert_bits_equal(g[k], c[k], name)
    assert g[5].max() < 400
    w = O.trace_brute(world, rays[:256])
    for k in range(5):
        assert_bits_equal(g[k][:256], w[k], "brute force")


def test_rebuild_after_new_transforms_matches_cpu_twin(gpu):
    """A dynamic frame: new instance transforms, same meshes (only the
    transforms are uploaded again).  The rebuilt BVH8 equals the CPU twin of
    the moved scene bit for bit, and tracing sees the moved geometry."""
    import snkpt
    scene = snkpt.SceneData(1)
    ctx = make_ctx(scene)
    pos, idx, inst, m4, _ = scene.arrays()
    m4 = np.asarray(m4, np.float32).reshape(-1, 16).copy()
    for k in range(3):
        moved = m4.copy()
        moved[1:, 13] += 0.05 * (k + 1)  # column-major: y translation of every transform but the first
        ctx.set_instances(inst, moved)
        ctx.build_accel()
        world = O.flatten(pos, idx, inst, moved)
        b = O.Bvh(world)
        assert np.array_equal(ctx.export(4), b.nodes), k
        assert_bits_equal(ctx.export(6), world.reshape(-1), f"world triangles, update {k}")
        rays = np.zeros((4096, 8), np.float32)
        rng = np.random.default_rng(k)
        rays[:, 0:3] = rng.uniform(-0.9, 0.9, (4096, 3)) + np.array([0, 1.0, 0], np.float32)
        d = rng.normal(size=(4096, 3)).astype(np.float32)
        rays[:, 4:7] = d / np.linalg.norm(d, axis=1, keepdims=True)
        rays[:, 7] = 1e30
        g = gpu_trace(ctx, rays)
        c = b.trace(rays)
        for j, name in enumerate(["t", "inst", "prim", "u", "v"]):
            assert_bits_equal(g[j], c[j], name)


def test_ray_counts_around_band_edges(gpu):
    """The persistent traversal deals the rays out in bands of (blocks x 64) and
    splits the last, partial band evenly; ray counts at and around the chunk and band
    edges, of four-wave blocks (up to 22 x 64 rays per CU) and of two large blocks per CU, (closest and any hit) must each trace every ray once,
    bit-identical to the CPU twin."""
    import torch

    import raysets
    import snkpt
    scene = snkpt.SceneData(1)
    ctx = make_ctx(scene)
    world = scene_world(scene)
    b = O.Bvh(world)
    assert b.depth - 1 <= 8  # the 8-entry stack variant: two blocks of 16 waves per CU
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    band = 16 * cus * 2 * 64  # 16 bands of the large blocks; cus * 256 rays fill a four-wave block per CU
    counts = sorted({1, 63, 64, 65, 1000, cus * 256 - 1, cus * 256, cus * 256 + 1, cus * 1024 + 63, band - 1, band, band + 1, band + 777, 2 * band + 4097})
    lo, hi = world[:, :9].reshape(-1, 3).min(0), world[:, :9].reshape(-1, 3).max(0)
    org, dr = raysets.random_rays(counts[-1], lo, hi, seed=21)
    rays = np.concatenate([org, dr], 1)
    for any_hit in (False, True):
        c = b.trace(rays, any_hit=any_hit)
        for n in counts:
            _say(f"band edges: n={n} (band {band}) any_hit={any_hit}")
            g = gpu_trace(ctx, rays[:n], any_hit=any_hit)
            for k, name in enumerate(["t", "inst", "prim", "u", "v", "nodes visited", "tris visited"]):
                assert_bits_equal(g[k], c[k][:n], f"n={n} {name}")


def test_autotuned_launch_shapes_keep_every_hit(gpu):
    """snkpt_build_accel's autotuner picks a launch shape per kind; every shape
    (refill threshold, steps per check, resident blocks) gives the same hits
    bit for bit, closest and any hit, as the oracle's traversal."""
    import torch

    import raysets
    import snkpt
    scene = snkpt.SceneData(2)
    ctx = snkpt.Context(0)
    ctx.load_scene(scene)
    ctx.build_accel()
    t0 = ctx.trace_tuning()
    print("autotuned:", t0.as_dict(), flush=True)
    assert not t0.fixed and t0.ms[0] > 0 and t0.ms[1] > 0
    assert t0.refill_lanes[0] in (4, 8, 16) and t0.steps_per_check[0] in (3, 4)
    org, dr = raysets.random_rays(200_000, scene_lo(ctx), scene_hi(ctx), seed=8)
    o, d = torch.from_numpy(org).cuda(), torch.from_numpy(dr).cuda()
    ref = None
    for refill, steps, bpc in ((8, 4, 16), (1, 3, 3), (64, 4, 1), (16, 3, 12)):
        t = snkpt.TraceTuning()
        t.refill_lanes[:] = [refill, refill]
        t.steps_per_check[:] = [steps, steps]
        t.blocks_per_cu[:] = [bpc, bpc]
        ctx.set_trace_tuning(t)
        assert ctx.trace_tuning().fixed == 1
        got = [[x.cpu().numpy() for x in ctx.trace(o, d, any_hit=a)[:3]] for a in (False, True)]
        if ref is None:
            ref = got
            continue
        for a in range(2):
            for k in range(3):
                assert_bits_equal(got[a][k], ref[a][k], f"shape {(refill, steps, bpc)} any={a} field {k}")
    c = O.Bvh(scene_world(scene)).trace(np.concatenate([org, dr], 1))
    assert_bits_equal(ref[0][0], c[0], "t vs oracle")
    assert_bits_equal(ref[0][2], c[2], "prim vs oracle")
    bad = snkpt.TraceTuning()
    bad.refill_lanes[:] = [0, 8]
    bad.steps_per_check[:] = [4, 4]
    bad.blocks_per_cu[:] = [16, 16]
    with pytest.raises(snkpt.SnkptError):
        ctx.set_trace_tuning(bad)
    ctx.set_trace_tuning(None)
    ctx.build_accel()
    assert ctx.trace_tuning().fixed == 0


def scene_lo(ctx):
    return list(ctx.accel_info().scene_lo)


def scene_hi(ctx):
    return list(ctx.accel_info().scene_hi)
