"""GPU: paths run to their ends by the path kernels (a group of eight lanes per path, a
thread per path, or lanes in stages, chosen by the frame's size and the tree's depth) give the frame
and the ray counts of the launch-per-bounce wavefront bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config,rr", [(1, 0), (5, 2)])
@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (160, 120), (256, 140), (256, 141), (256, 160), (256, 161),
                                 (258, 255), (420, 301), (640, 512), (641, 512)])
def test_path_kernels_match_wavefront(gpu, config, rr, w, h):
    import snkpt
    import torch
    from helpers import make_ctx
    scene = snkpt.SceneData(config, 1 if config == 5 else 0)
    ctx = make_ctx(scene)
    cam = scene.camera(0, w, h)
    got = []
    for tail in (6, 1, 2, 0):  # never, from bounce 1, from bounce 2, the context's own choice
        out = torch.zeros(h, w, 4, device="cuda")
        s = snkpt.default_settings(max_depth=6, rr_start=rr, seed=3, frame=2, tail_bounce=tail)
        ctx.render(cam, s, out, w, h)
        st = ctx.frame_stats()
        got.append((out.cpu().numpy(), st.extension_rays, st.shadow_rays))
    assert np.isfinite(got[0][0]).all()
    for g in got[1:]:
        assert np.array_equal(g[0].view(np.uint32), got[0][0].view(np.uint32))
        assert g[1:] == got[0][1:]


@pytest.mark.parametrize("w,h", [(64, 48), (257, 161), (700, 500)])
def test_path_kernels_after_restir(gpu, w, h):
    """The bounces after ReSTIR's primary vertex, by the same kernels."""
    import snkpt
    import torch
    from helpers import make_ctx
    scene = snkpt.SceneData(1)
    cam = scene.camera(0, w, h)
    got = []
    for tail in (5, 1, 0):
        ctx = make_ctx(scene)  # no history
        out = torch.zeros(h, w, 4, device="cuda")
        s = snkpt.default_settings(mode=snkpt.MODE_RESTIR, max_depth=5, seed=3, tail_bounce=tail)
        ctx.render(cam, s, out, w, h)
        st = ctx.frame_stats()
        got.append((out.cpu().numpy(), st.extension_rays, st.shadow_rays))
    for g in got[1:]:
        assert np.array_equal(g[0].view(np.uint32), got[0][0].view(np.uint32))
        assert g[1:] == got[0][1:]
