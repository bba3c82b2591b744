"""GPU: the cache's queries give the same bits whatever the call's size (rows of
inputs up to 40,960 queries, level by level above), against the FP64 oracle's
encoding at the line between the two and at ragged sizes."""
import numpy as np
import pytest

from oracle import binding as O

pytestmark = pytest.mark.gpu
LO, HI = [-1.0, 0.0, -1.0], [1.0, 2.0, 1.0]


@pytest.fixture(scope="module")
def net(gpu):
    import snkpt
    import torch
    ctx = snkpt.Context(0)
    ctx.cache_reset(3, LO, HI)
    rng = np.random.default_rng(4)
    grid = (rng.uniform(-1, 1, O.GRID_PARAMS) * 0.3).astype(np.float32)
    ctx.cache_set_params(1, grid)
    n = 70001
    s = np.zeros((n, 16), np.float32)
    s[:, 0:3] = rng.uniform([-1.1, -0.1, -1.1], [1.1, 2.1, 1.1], (n, 3))  # some outside the box
    s[:8, 0:3] = [[a, b, c] for a in (-1, 1) for b in (0, 2) for c in (-1, 1)]  # its corners
    d = rng.normal(size=(n, 6))
    s[:, 3:6] = d[:, :3] / np.linalg.norm(d[:, :3], axis=1, keepdims=True)
    s[:, 6:9] = d[:, 3:] / np.linalg.norm(d[:, 3:], axis=1, keepdims=True)
    s[:, 9:13] = rng.uniform(0.05, 1, (n, 4))
    t = torch.from_numpy(s).cuda()
    full = ctx.cache_infer(t).cpu().numpy()
    enc = ctx.cache_params(4).reshape(n, 64).copy()
    return ctx, s, t, full, enc, grid


@pytest.mark.parametrize("n", [1, 65, 32767, 32768, 32769, 40959, 40960, 40961, 65535, 70001])
def test_same_bits_at_every_size(net, n):
    ctx, _, t, full, enc, _ = net
    y = ctx.cache_infer(t[:n].contiguous()).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), full[:n].view(np.uint32))
    assert np.array_equal(ctx.cache_params(4).view(np.uint16), enc[:n].reshape(-1).view(np.uint16))


def test_encoding_matches_oracle(net):
    _, s, _, _, enc, grid = net
    pick = np.r_[0:64, 32700:32800, 40900:41000, 69900:70001]
    want = O.cache_encode(O.CacheGeom(LO, HI), grid, s[pick])
    # FP16 grid entries and an FP16 result: the tolerance of the row-wise encoding's test
    assert np.allclose(enc[pick].astype(np.float64), want, rtol=4e-3, atol=2e-3)


@pytest.mark.parametrize("n", [65, 70001])
@pytest.mark.parametrize("shift", [1, 2, 3])
def test_samples_need_a_floats_alignment_only(net, n, shift):
    import torch
    ctx, s, _, full, enc, _ = net
    buf = torch.zeros(n * 16 + 4, device="cuda")
    t = buf[shift:shift + n * 16].view(n, 16)
    t.copy_(torch.from_numpy(s[:n]))
    assert t.data_ptr() % 16 == 4 * shift
    y = ctx.cache_infer(t).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), full[:n].view(np.uint32))
    assert np.array_equal(ctx.cache_params(4).view(np.uint16), enc[:n].reshape(-1).view(np.uint16))


@pytest.mark.parametrize("first,w,h", [(70001, 97, 53), (1000, 300, 200), (70001, 300, 200), (41000, 300, 200)])
def test_encoded_inputs_after_a_frame(gpu, first, w, h):
    """The encoded inputs read back after a cache frame without training are those of
    the frame's queries whatever layout the encodings before and in the frame took, and
    those of each replay after a captured frame's replay."""
    import snkpt
    import torch

    from helpers import make_ctx
    scene = snkpt.SceneData(1)
    ctx = make_ctx(scene)
    info = ctx.accel_info()
    lo, hi = list(info.scene_lo), list(info.scene_hi)
    rng = np.random.default_rng(first + w)
    ctx.cache_reset(3, lo, hi)
    grid = (rng.uniform(-1, 1, O.GRID_PARAMS) * 0.3).astype(np.float32)
    ctx.cache_set_params(1, grid)
    s = np.zeros((first, 16), np.float32)
    s[:, 0:3] = rng.uniform(lo, hi, (first, 3))
    s[:, 3:13] = rng.uniform(0.1, 0.9, (first, 10))
    t = torch.from_numpy(s).cuda()
    cam = scene.camera(0, w, h)
    out = torch.zeros(h, w, 4, device="cuda")
    st = snkpt.default_settings(mode=snkpt.MODE_CACHE, max_depth=4, seed=5, cache_query_depth=1,
                                flags=snkpt.FLAG_NO_STATS | snkpt.FLAG_NO_TRAIN)

    def check():
        q = ctx.cache_params(5).reshape(-1, 16)
        enc = ctx.cache_params(4).reshape(-1, 64).astype(np.float64)
        assert enc.shape[0] == first and q.shape[0] > 0.3 * w * h
        k = min(first, q.shape[0])
        # FP16 grid entries and an FP16 result: the tolerance of the encoding's own test
        want = O.cache_encode(O.CacheGeom(lo, hi), grid, q[:k])
        assert np.allclose(enc[:k], want, rtol=4e-3, atol=2e-3)
        assert not enc[q.shape[0]:].any()

    ctx.cache_infer(t)
    ctx.render(cam, st, out, w, h)
    torch.cuda.synchronize()
    check()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.render(cam, st, out, w, h)
    for _ in range(2):
        ctx.cache_infer(t)
        enc = ctx.cache_params(4).reshape(-1, 64)[::97].astype(np.float64)
        assert np.allclose(enc, O.cache_encode(O.CacheGeom(lo, hi), grid, s[::97]), rtol=4e-3, atol=2e-3)
        g.replay()
        torch.cuda.synchronize()
        check()
