"""GPU: the short square root, reciprocal and quotient against IEEE arithmetic (numpy
on the CPU) over all mantissas and over random and nearly half-way quotients up to
the ends of the stated ranges; and the shading functions, which choose between short
and general forms, against the same formulas in general forms, for materials,
normals and directions on both sides of every line between the two."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tests", "native", "libshading_check.so")


@pytest.fixture(scope="module")
def check(gpu):
    if not os.path.exists(LIB):
        subprocess.run(["make", "-C", os.path.join(ROOT, "snake-vk_amd", "csrc"), "check"], check=True)
    lib = ctypes.CDLL(LIB)
    P, U = ctypes.c_void_p, ctypes.c_uint32
    lib.check_unary.argtypes = [ctypes.c_int, P, P, U]
    lib.check_quotient.argtypes = [P, P, P, P, U]
    lib.check_shading.argtypes = [P, P, P, U]
    return lib


def _call(fn, args, outs):
    """fn(device copies of args, device buffers of the shapes outs, count) -> the buffers."""
    import torch
    n = len(args[-1])
    dev = [torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda() for a in args]
    buf = [torch.zeros(s, device="cuda") for s in outs]
    torch.cuda.synchronize()
    assert fn(*[ctypes.c_void_p(t.data_ptr()) for t in dev + buf], n) == 0
    return [b.cpu().numpy() for b in buf]


def _same(got, want, what):
    g, w = got.view(np.uint32), want.view(np.uint32)
    bad = np.nonzero((g != w) & ~(np.isnan(got) & np.isnan(want)))[0]
    assert bad.size == 0, f"{what}: {bad.size} differ, first {bad[:3]}: {got[bad[:3]]} for {want[bad[:3]]}"


@pytest.mark.parametrize("op", ["rcp", "sqrt"])
@pytest.mark.parametrize("exponent", [-100, -61, -1, 0, 1, 60, 99])
def test_all_mantissas(check, op, exponent):
    a = (np.arange(1 << 23, dtype=np.uint32) | np.uint32((127 + exponent) << 23)).view(np.float32)
    got, = _call(lambda p, q, n: check.check_unary(0 if op == "rcp" else 1, p, q, n), [a], [a.size])
    _same(got, np.float32(1) / a if op == "rcp" else np.sqrt(a), f"{op}, exponent {exponent}")


@pytest.mark.parametrize("xe,de", [((-60, 59), (-60, 59)), ((-100, -60), (-100, 24)), ((-74, 49), (-50, 49)),
                                   ((0, 0), (0, 0)), ((-100, -100), (-25, 24))])
def test_quotients(check, xe, de):
    rng = np.random.default_rng(abs(xe[0] * 1000 + de[1]))
    n = 1 << 22
    m = rng.integers(0, 1 << 23, (2, n), dtype=np.uint32)
    d = (m[0] | ((127 + rng.integers(de[0], de[1] + 1, n)) << 23).astype(np.uint32)).view(np.float32)
    x = (m[1] | ((127 + rng.integers(xe[0], xe[1] + 1, n)) << 23).astype(np.uint32)).view(np.float32)
    # half of them next to the middle of two neighbouring quotients: (2^24 + odd) 2^-24 d, rounded
    half = (((1 << 24) + 2 * rng.integers(0, 1 << 23, n // 2) + 1).astype(np.float64)
            * np.exp2(-24.0) * d[:n // 2].astype(np.float64)).astype(np.float32)
    e = np.clip(np.frexp(half)[1] - 1, xe[0], xe[1])
    x[:n // 2] = np.ldexp(np.frexp(half)[0], e + 1)
    x *= np.where(rng.random(n) < 0.5, np.float32(1), np.float32(-1))
    x[-16:] = np.float32([0.0, -0.0] * 8)
    with np.errstate(over="ignore", under="ignore"):
        want, q = x / d, np.abs(x.astype(np.float64) / d)
    ok = (x == 0) | ((q >= 2.0 ** -125) & (q < 2.0 ** 125))
    assert ok.mean() > 0.5
    got, sgn = _call(check.check_quotient, [x, d], [n, n])
    z = ok & (x != 0)
    _same(got[z], want[z], "quotient")
    assert not got[x == 0].view(np.uint32).any()  # a zero gives +0
    _same(sgn[ok], want[ok], "signed quotient")


def _unit(v):
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def _cases(kind, n, rng):
    c = np.zeros((n, 20))
    c[:, 0:3] = _unit(rng.normal(size=(n, 3)))
    for k in (3, 6):
        v = _unit(rng.normal(size=(n, 3)))
        c[:, k:k + 3] = v * np.where((v * c[:, 0:3]).sum(1, keepdims=True) < 0, -1.0, 1.0)
    c[:, 9:12] = rng.uniform(0, 1, (n, 3))
    c[:, 12] = rng.uniform(0, 1, n)
    c[:, 13] = np.where(rng.random(n) < 0.5, rng.integers(0, 2, n), rng.uniform(0, 1, n))
    c[:, 14:17] = rng.integers(0, 1 << 24, (n, 3)) / 2.0 ** 24
    c[:, 17:19] = np.exp2(rng.uniform(-8, 8, (n, 2)))
    if kind == "roughness":  # smooth to far beyond 1, and negative
        c[:, 12] = np.exp2(rng.uniform(-40, 40, n)) * np.where(rng.random(n) < 0.1, -1, 1)
        c[::7, 12] = 0.0
        c[1::31, 12] = np.inf
    elif kind == "grazing":  # cosines down to the smallest and exact zeros
        t = np.stack([c[:, 1], -c[:, 0], np.zeros(n)], 1)
        e = np.exp2(rng.uniform(-70, -1, (n, 2, 1)))
        e[::5] = 0.0
        t = _unit(t)
        for j, k in enumerate((3, 6)):
            c[:, k:k + 3] = _unit(t * (1 - 2 * j * (rng.random((n, 1)) < 0.5)) + e[:, j] * c[:, 0:3])
    elif kind == "mirror":  # the lobe's centre, and its neighbours
        d = 2 * (c[:, 0:3] * c[:, 3:6]).sum(1, keepdims=True) * c[:, 0:3] - c[:, 3:6]
        c[:, 6:9] = d + np.exp2(rng.uniform(-40, -5, (n, 1))) * rng.normal(size=(n, 3))
        c[:, 12] = np.exp2(rng.uniform(-20, 0, n))
    elif kind == "normals":  # of any length, some axis aligned, some with tiny components
        c[:, 0:3] *= np.exp2(rng.uniform(-70, 70, (n, 1)))
        c[::3, 0:3] *= np.where(rng.random((len(c[::3]), 3)) < 0.5, 0.0, 1.0)
        c[1::3, 0:3] *= np.exp2(rng.uniform(-90, 0, (len(c[1::3]), 3)))
    elif kind == "pdfs":
        c[:, 17:19] = np.exp2(rng.uniform(-70, 70, (n, 2)))
        c[::9, 17] = 0.0
        c[::11, 18] = 0.0
    elif kind == "lambert":
        c[:, 19] = 1.0
    with np.errstate(over="ignore", invalid="ignore"):
        return c.astype(np.float32)


@pytest.mark.parametrize("kind", ["usual", "roughness", "grazing", "mirror", "normals", "pdfs", "lambert"])
def test_shading_equals_general_forms(check, kind):
    n = 1 << 19
    c = _cases(kind, n, np.random.default_rng(len(kind)))
    got, want = _call(check.check_shading, [c], [(n, 15), (n, 15)])
    for k, name in enumerate(["normalize x", "normalize y", "normalize z", "f r", "f g", "f b", "pdf", "heuristic",
                              "wi x", "wi y", "wi z", "above", "short f r", "short f g", "short f b"]):
        _same(np.ascontiguousarray(got[:, k]), np.ascontiguousarray(want[:, k]), f"{kind}, {name}")
