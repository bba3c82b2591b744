"""GPU: frames are the same bits whether the lengths of the vertex normals take the short
or the general root (test_gpu_exact_math.py holds each function against its general
form), and so do the two register layouts of ReSTIR's
spatial pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(ctx, scale):
    """A small room; the vertex normals are unit normals times `scale`."""
    from helpers import ArrayScene
    s = ArrayScene()
    s.quad([-1, 0, -1], [0, 0, 2], [2, 0, 0], [0.7, 0.6, 0.5], 0, roughness=0.4)
    s.quad([-1, 0, -1], [2, 0, 0], [0, 2, 0], [0.3, 0.7, 0.4], 0, roughness=0.02, metallic=1.0)
    s.quad([-1, 0, -1], [0, 2, 0], [0, 0, 2], [0.6, 0.3, 0.3], 2)
    s.quad([-0.3, 1.9, -0.3], [0.6, 0, 0], [0, 0, 0.6], [6.0, 6.0, 5.0], 1)
    s.nrm = [n * np.float32(scale) for n in s.nrm]
    s.load_into(ctx)


def _frames(ctx, mode, w, h, n=2, **kw):
    import snkpt
    import torch
    cam = snkpt.SceneData(1).camera(0, w, h)
    out = torch.zeros(h, w, 4, device="cuda")
    got = []
    for f in range(n):
        ctx.render(cam, snkpt.default_settings(mode=mode, frame=f, seed=7, **kw), out, w, h)
        got.append(out.cpu().numpy().copy())
    return np.stack(got)


# squared lengths 2^-60 and 2^64 take the short form, 2^104 and 2^120 the general one;
# every step of the normalisation scales by a power of two, so the images are equal
@pytest.mark.parametrize("exponent", [-30, 32, 52, 60])
@pytest.mark.parametrize("mode,depth", [("MODE_PT", 4), ("MODE_RESTIR", 2)])
def test_length_of_vertex_normals_changes_nothing(gpu, exponent, mode, depth):
    import snkpt
    got = []
    for scale in (1.0, 2.0 ** exponent):
        ctx = snkpt.Context(0)
        _box(ctx, scale)
        got.append(_frames(ctx, getattr(snkpt, mode), 97, 53, max_depth=depth, num_spatial_resamples=3))
    assert np.isfinite(got[0]).all() and got[0].max() > 0.0
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


# within 0.4 pixels every neighbour is the pixel itself and is dropped: one input, whose
# sample is always taken, so the count of neighbours asked for changes nothing
@pytest.mark.parametrize("w,h", [(1, 1), (17, 15), (130, 67)])
def test_spatial_layouts_agree_without_neighbours(gpu, w, h):
    import snkpt
    got = []
    for k in (1, 5, 6, 8):
        ctx = snkpt.Context(0)
        _box(ctx, 1.0)
        got.append(_frames(ctx, snkpt.MODE_RESTIR, w, h, max_depth=1, num_spatial_resamples=k, restir_radius=0.4))
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))
