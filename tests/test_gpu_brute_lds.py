"""Frames without a tree whose shapes fit LDS: primitives tested four at a time, shapes and lights read from LDS up to
their limits (256 primitives, 64 shapes, 32 lights).  Colours and seeds equal the oracle's brute force bit for bit
(RadianceGPU with ACCELSTR 0, rendering_kernel.cl:495-753), pixels within its powf's one step, and all three equal the
launch that counts tests, which reads one primitive at a time.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
import pyoracle as O
from ptgpu_pc_amd import scenes
from ptgpu_pc_amd.layout import default_seeds

from test_gpu_parity import SPHERE, image_checks, render_oracle, say

pytestmark = pytest.mark.gpu
F32 = np.float32


def _scene(kind, n, lights, w, h):
    s = scenes.soup(max(n, 4), seed=n)[0][-n:].copy()
    rng = np.random.default_rng(n)
    k = np.arange(n)
    sph = {"spheres": k >= 0, "triangles": k < 0, "mixed": (k % 5 < 2) | (k // 4 % 2 == 0)}[kind]
    c = rng.random((n, 3)).astype(F32)
    rad = (0.05 + 0.1 * rng.random(n)).astype(F32)
    for i in np.flatnonzero(sph):
        s["type"][i] = SPHERE
        s["rad"][i] = rad[i]
        s["p"][i] = c[i]
        s["area"][i] = F32(4 * np.pi) * rad[i] * rad[i]
    s["refl"] = np.where(k % 7 == 3, 1, np.where(k % 7 == 5, 2, 0))
    s["c"] = F32(0.75)
    s["e"] = 0
    for i in range(min(lights, n)):
        s["e"][i * n // max(lights, 1)] = (3, 2, 1)
    _, _, cam = scenes.soup(16, seed=1, width=w, height=h)
    pt.update_camera(cam)
    return s, min(lights, n), cam


def _frame(ctx, s, lc, cam, w, h, spp, depth, stats=None):
    col = ctx.alloc(w * h * 12, F32).zero()
    seeds = ctx.to_device(default_seeds(w, h))
    pix = ctx.alloc(w * h * 4, np.uint32)
    pt.render(ctx, None, None, colors=col, seeds=seeds, camera=ctx.to_device(cam), shapes=ctx.to_device(s), shapeCnt=len(s),
              lightCnt=lc, width=w, height=h, spp=spp, max_depth=depth, pixels=pix, trav_stats=stats)
    ctx.synchronize()
    return col.download(F32), seeds.download(np.uint32), pix.download(np.uint32)


@pytest.mark.parametrize("n,lights", [(1, 1), (2, 1), (4, 1), (5, 2), (9, 1), (63, 3), (64, 31), (65, 32), (255, 33),
                                      (256, 2), (257, 2)])
@pytest.mark.parametrize("kind", ["spheres", "triangles", "mixed"])
def test_brute_frame(ctx, kind, n, lights):
    say("case brute", kind, n, lights)
    w, h = 37, 22
    s, lc, cam = _scene(kind, n, lights, w, h)
    got = _frame(ctx, s, lc, cam, w, h, 2, 4)
    image_checks(*got, *render_oracle(s, lc, cam, w, h, 2, 4, O.accel_none()))
    ref = _frame(ctx, s, lc, cam, w, h, 2, 4, ctx.alloc(16, np.uint64).zero())
    for a, b in zip(got, ref):
        assert a.tobytes() == b.tobytes()


@pytest.mark.parametrize("what", ["tangent", "zero radius", "huge radius", "far", "nan centre", "inf camera", "nan camera"])
def test_brute_odd_spheres(ctx, what):
    """Determinants of zero, at the ends of the exponent range, and not finite."""
    say("case brute odd", what)
    w, h = 33, 17
    s, lc, cam = _scene("spheres", 9, 1, w, h)
    if what == "tangent":      # axis rays along a sphere's side: the determinant is exactly zero
        cam["x"][0] = 0
        cam["y"][0] = 0
        cam["dir"][0] = (0, 0, -1)
        cam["orig"][0] = (0.5, 0.5, 2.5)
        s["p"][4] = (0.25, 0.5, 0.5)
        s["rad"][4] = 0.25
    elif what == "zero radius":
        s["rad"][::2] = 0
    elif what == "huge radius":
        s["rad"][3] = F32(1e20)
        s["p"][3] = (0, 0, F32(2e20))
    elif what == "far":
        cam["orig"][0] = (0.5, 0.5, 1e19)
    elif what == "nan centre":
        s["p"][2] = np.nan
    else:
        cam["orig"][0] = np.inf if what == "inf camera" else np.nan
    got = _frame(ctx, s, lc, cam, w, h, 1, 3)
    ref = _frame(ctx, s, lc, cam, w, h, 1, 3, ctx.alloc(16, np.uint64).zero())
    for a, b in zip(got, ref):
        assert a.tobytes() == b.tobytes()
