"""GPU parity of the ray hand-out: the same rays traced in calls of every size
class (one ray, part of a wave, the edges of 64-ray chunks, of the blocks and bands of
a launch, and of the lines between eight lanes per ray, small blocks and large blocks)
and with directions whose inverses leave the range of the short reciprocal return the
hits of the CPU BVH8 traversal bit for bit.  A counted call always has a lane per ray."""
import numpy as np
import pytest

from helpers import assert_bits_equal, make_ctx, scene_world
from oracle import binding as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def room(gpu):
    import raysets
    import snkpt
    scene = snkpt.SceneData(1)
    ctx = make_ctx(scene)
    bvh = O.Bvh(scene_world(scene))
    org, dr = raysets.random_rays(400003, [-1, 0, -1], [1, 2, 1], seed=5)
    rays = np.concatenate([org, dr], 1)
    return ctx, bvh, rays, bvh.trace(rays, any_hit=False), bvh.trace(rays, any_hit=True)


@pytest.fixture(scope="module")
def field(gpu):
    """1.02M triangles: a deeper tree, another stack variant, the groups' line at 2^17."""
    import raysets
    import snkpt
    scene = snkpt.SceneData(2)
    ctx = make_ctx(scene)
    bvh = O.Bvh(scene_world(scene))
    assert bvh.depth == ctx.accel_info().depth >= 8
    info = ctx.accel_info()
    org, dr = raysets.random_rays(360449, list(info.scene_lo), list(info.scene_hi), seed=6)
    rays = np.concatenate([org, dr], 1)
    return ctx, rays, bvh.trace(rays, any_hit=False), bvh.trace(rays, any_hit=True)


def _trace(ctx, rays, any_hit, counted=False):
    import torch
    o = torch.from_numpy(np.ascontiguousarray(rays[:, :4])).cuda()
    d = torch.from_numpy(np.ascontiguousarray(rays[:, 4:])).cuda()
    return [None if a is None else a.cpu().numpy() for a in ctx.trace(o, d, any_hit=any_hit, counted=counted)]


def _check(ctx, rays, n, closest, first, counted):
    for any_hit, want in ((False, closest), (True, first)):
        got = _trace(ctx, rays[:n], any_hit, counted)
        for k, name in enumerate(["t", "inst", "prim"]):
            assert_bits_equal(got[k], want[k][:n], f"{name}, {n} rays, any hit {any_hit}")
        if not any_hit:
            for k, name in ((3, "u"), (4, "v")):
                assert_bits_equal(got[k], want[k][:n], f"{name}, {n} rays")


# counted: a lane per ray from the first ray on; blocks of 4 waves take 256 rays, a band of
# them is 64 rays a block
@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 65, 1000, 4097, 32768, 32769, 65535, 65536, 65537, 70000])
def test_call_sizes(room, n, counted):
    ctx, _, rays, closest, first = room
    _check(ctx, rays, n, closest, first, counted)


# on both sides of the groups' line (81,920 in a tree of depth 7) and of the small blocks'
# (22 waves' lanes on each of 256 CUs), then of bands of two large blocks per CU
@pytest.mark.parametrize("n", [81919, 81920, 81921, 100003, 360447, 360448, 360449, 393215, 393217, 400003])
def test_call_sizes_around_the_lines(room, n):
    ctx, bvh, rays, closest, first = room
    assert bvh.depth == 7
    _check(ctx, rays, n, closest, first, False)


@pytest.mark.parametrize("n", [5, 16385, 131071, 131072, 131073, 200003, 360448, 360449])
def test_call_sizes_of_a_deeper_tree(field, n):
    ctx, rays, closest, first = field
    _check(ctx, rays, n, closest, first, False)


@pytest.mark.parametrize("counted", [False, True])
def test_extreme_directions(room, counted):
    """Components at and beyond both ends of the short reciprocal's range, zeros of
    both signs, unnormalised rays, and rays that miss at once (zero, NaN, empty)."""
    ctx, bvh, rays, _, _ = room
    rng = np.random.default_rng(9)
    r = rays[:4096].copy()
    mag = np.array([0.0, -0.0, 1e-30, 1e-20, 2.0 ** -61, 2.0 ** -60, 1e-10, 1.0, 1e10, 2.0 ** 60, 2.0 ** 61], np.float32)
    for k in range(4096):
        for a in rng.permutation(3)[:rng.integers(1, 3)]:
            r[k, 4 + a] = mag[rng.integers(len(mag))] * (1 if rng.random() < 0.5 else -1)
    r[0, 4:7] = 0.0
    r[1, 4] = np.nan
    r[2, 3], r[2, 7] = 2.0, 1.0
    for any_hit in (False, True):
        want = bvh.trace(r, any_hit=any_hit)
        got = _trace(ctx, r, any_hit, counted)
        for k, name in enumerate(["t", "inst", "prim"]):
            assert_bits_equal(got[k], want[k], f"{name}, any hit {any_hit}")
