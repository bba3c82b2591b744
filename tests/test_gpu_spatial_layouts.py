"""GPU: ReSTIR's spatial pass gives the same reservoirs bit for bit whichever register
layout it is compiled for, with neighbours accepted and rejected."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "native", "libspatial_check.so")


def _inputs(w, h, rng):
    """A wavy floor under 300 emitters: most neighbours pass the normal and distance tests."""
    n = w * h
    y, x = np.mgrid[0:h, 0:w].reshape(2, -1)
    g = np.zeros((5, n, 4), np.float32)
    g[0, :, 0], g[0, :, 2] = x / 20.0, y / 20.0
    g[0, :, 1] = 0.05 * np.sin(x / 7.0)
    g[0, :, 3] = np.where(rng.random(n) < 0.1, 0.0, 1e-4)  # no surface
    nrm = np.stack([0.4 * np.sin(x / 9.0 + y / 5.0), np.ones(n), 0.3 * rng.normal(size=n) * (rng.random(n) < 0.2)], 1)
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    g[1, :, :3] = g[2, :, :3] = nrm
    g[1, :, 3] = np.where(rng.random(n) < 0.2, 0.0, rng.uniform(0, 1, n))  # mirrors among them
    g[2, :, 3] = rng.integers(0, 2, n)
    g[3, :, :3] = rng.uniform(0.1, 0.9, (n, 3))
    g[3, :, 3] = np.where(rng.random(n) < 0.3, 2, 0).astype(np.uint32).view(np.float32)  # Lambert or GGX
    wo = np.stack([rng.normal(size=n) * 0.5, np.ones(n), rng.normal(size=n) * 0.5], 1)
    g[4, :, :3] = wo / np.linalg.norm(wo, axis=1, keepdims=True)
    g[4, :, 3] = rng.uniform(3.0, 3.5, n)
    ne = 300
    e = np.zeros((ne, 4, 4), np.float32)
    c = np.stack([rng.uniform(-1, w / 20 + 1, ne), rng.uniform(0.5, 2, ne), rng.uniform(-1, h / 20 + 1, ne)], 1)
    for v in range(3):
        e[:, v, :3] = c + rng.normal(size=(ne, 3)) * 0.1
    e[::50, 1] = e[::50, 0]  # triangles of no area
    e[:, 2, 3] = 1.0 / ne
    e[:, 3, :3] = rng.uniform(0, 5, (ne, 3))
    e[:, 3, 3] = 0.02
    r = np.zeros((n, 4), np.float32)
    idx = rng.integers(0, ne, n).astype(np.uint32)
    idx[rng.random(n) < 0.1] = 0xFFFFFFFF
    r[:, 0] = idx.view(np.float32)
    u = np.sort(rng.random((n, 2)), axis=1)
    r[:, 1], r[:, 2] = u[:, 0], 1 - u[:, 1]
    r[:, 3] = np.where(rng.random(n) < 0.1, 0.0, rng.uniform(0.1, 3, n))
    m = rng.integers(1, 21, n).astype(np.float32)
    return g, r, m, e


@pytest.mark.parametrize("w,h", [(1, 1), (37, 23), (130, 67)])
def test_layouts_agree(gpu, w, h):
    import torch
    if not os.path.exists(LIB):
        subprocess.run(["make", "-C", os.path.join(ROOT, "snake-vk_amd", "csrc"), "check"], check=True)
    lib = ctypes.CDLL(LIB)
    P, U = ctypes.c_void_p, ctypes.c_uint32
    lib.check_spatial.argtypes = [U, P, P, P, P, U, U, U, U, ctypes.c_float, ctypes.c_uint64, P, P]
    g, r, m, e = _inputs(w, h, np.random.default_rng(w))
    d = [torch.from_numpy(a).cuda() for a in (g, r, m, e)]

    def run(layout, k, radius):
        out_r, out_m = torch.zeros(w * h, 4, device="cuda"), torch.zeros(w * h, device="cuda")
        torch.cuda.synchronize()
        assert lib.check_spatial(layout, *[P(t.data_ptr()) for t in d], len(e), w, h, k, radius, 0x1234,
                                 P(out_r.data_ptr()), P(out_m.data_ptr())) == 0
        return out_r.cpu().numpy().view(np.uint32), out_m.cpu().numpy()

    for radius in (2.5, 30.0):
        for k in range(1, 9):
            got = [run(lay, k, radius) for lay in (5, 8, 10) if k <= lay]
            for o in got[1:]:
                assert np.array_equal(o[0], got[0][0]) and np.array_equal(o[1], got[0][1]), (k, radius)
            if w > 1 and k == 8:  # not in vain: a neighbour was taken for many pixels, and its sample for some
                assert (got[0][1] > m).mean() > 0.25
                assert (got[0][0][:, 0] != r[:, 0].view(np.uint32)).mean() > 0.02
