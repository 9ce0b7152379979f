"""Sparse waves and the bounce's shared shading pass.

A small frame gives each wave only 1, 2, 4 or 8 pixels and the other lanes help their queries (groups of 4
to 64 lanes per query, several stack entries per step), by a rule on the frame's pixels; a full wave goes
through the same phases as its lanes run out.  Shadow rays of a bounce are drawn two at a time with the next
direction.  Neither changes a bit: each frame equals the same frame with 64 pixels per wave and one lane per
query, and the oracle's (RadianceGPU, rendering_kernel.cl:969-1150).
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
import pyoracle as O
from ptgpu_pc_amd import scenes
from ptgpu_pc_amd.layout import default_seeds

from test_gpu_parity import image_checks, render_oracle, say

pytestmark = pytest.mark.gpu
F32 = np.float32


def _frame(ctx, bvh, d_sh, n, lc, d_cam, w, h, spp, depth):
    col = ctx.alloc(w * h * 12, F32).zero()
    seeds = ctx.to_device(default_seeds(w, h))
    pix = ctx.alloc(w * h * 4, np.uint32)
    pt.render(ctx, bvh, None, colors=col, seeds=seeds, camera=d_cam, shapes=d_sh, shapeCnt=n, lightCnt=lc, width=w,
              height=h, spp=spp, max_depth=depth, pixels=pix)
    ctx.synchronize()
    return col.download(F32), seeds.download(np.uint32), pix.download(np.uint32)


def _scene(kind, w, h):
    if kind == "soup":
        s, lc, cam = scenes.soup(3000, seed=6, width=w, height=h)
    elif kind == "lights":   # five emitters, two of them spheres: more than one pass draws at a time
        s, lc, cam = scenes.soup(400, seed=8, width=w, height=h)
        s["e"][[7, 90, 203]] = ((3, 2, 1), (1, 4, 2), (2, 2, 5))
        for k in (90, 203):
            p = s["p1"][k].copy()
            s["type"][k] = 0
            s["rad"][k] = F32(0.03)
            s["p"][k] = p
            s["area"][k] = F32(4 * np.pi * 0.03 ** 2)
        lc = 5
    else:
        s, lc, cam = scenes.icosphere_in_box(2, seed=3, width=w, height=h)
    pt.update_camera(cam)
    return s, lc, cam


# 1 pixel; around 4096, 8192, 16384 and 32768 pixels, where the rule's pixels per wave change (1, 2, 4, 8, 64)
@pytest.mark.parametrize("w,h", [(1, 1), (64, 64), (241, 17), (90, 91), (91, 91), (129, 128), (181, 181), (182, 181)])
@pytest.mark.parametrize("kind", ["soup", "mesh", "lights"])
def test_pixels_per_wave(kind, w, h):
    say("case pixels per wave", kind, w, h)
    s, lc, cam = _scene(kind, w, h)
    with pt.Context(0) as ctx:
        d_sh, d_cam = ctx.to_device(s), ctx.to_device(cam)
        bvh = pt.CLBVH(ctx, d_sh)
        bvh.buildRadixTree()
        bvh.buildBVHTree()
        got = _frame(ctx, bvh, d_sh, len(s), lc, d_cam, w, h, 2, 5)
        ctx.set_tuning("blocks_per_cu", 2)   # 64 pixels per wave
        ctx.set_tuning("quad", 0)            # one lane per query
        ref = _frame(ctx, bvh, d_sh, len(s), lc, d_cam, w, h, 2, 5)
        ctx.set_tuning("wide", 0)            # binary nodes
        ref2 = _frame(ctx, bvh, d_sh, len(s), lc, d_cam, w, h, 2, 5)
        bvh.close()
    for a, b, c in zip(got, ref, ref2):
        assert a.tobytes() == b.tobytes()
        assert a.tobytes() == c.tobytes()
    if w * h <= 4096:
        _, _, btn, btl = O.build_lbvh(s)
        image_checks(*got, *render_oracle(s, lc, cam, w, h, 2, 5, O.accel_bvh(btn, btl)))


def test_camera_inside_and_outside():
    """More than two pixels per lane slot of two workgroups per CU: a camera inside the scene's box keeps all four
    workgroups of a CU, one outside two.  The same bits either way."""
    w, h = 700, 560
    for kind in ("soup", "mesh"):
        say("case camera", kind)
        s, lc, cam = _scene(kind, w, h)
        with pt.Context(0) as ctx:
            d_sh, d_cam = ctx.to_device(s), ctx.to_device(cam)
            bvh = pt.CLBVH(ctx, d_sh)
            bvh.buildRadixTree()
            bvh.buildBVHTree()
            got = _frame(ctx, bvh, d_sh, len(s), lc, d_cam, w, h, 1, 4)
            ctx.set_tuning("blocks_per_cu", 1)
            ref = _frame(ctx, bvh, d_sh, len(s), lc, d_cam, w, h, 1, 4)
            bvh.close()
        for a, b in zip(got, ref):
            assert a.tobytes() == b.tobytes()


def test_axis_rays_and_far_origins(ctx):
    """The binary16 slab test's ends: directions with zero and denormal components, origins far outside; hits
    equal the binary walk's (which forms (bound - origin) / direction) on every ray."""
    s, lc, cam = scenes.soup(3000, seed=9)
    d_sh = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d_sh)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    # a camera ray through every pixel of a frame whose camera looks exactly along -z, from far away
    w, h = 64, 48
    out = []
    for wide, orig in ((2, 2.5), (0, 2.5), (2, 3e5), (0, 3e5)):
        _, _, cam = scenes.soup(16, seed=1, width=w, height=h)
        cam["orig"][0] = (0.5, 0.5, orig)
        pt.update_camera(cam)
        cam["x"][0] = (0.0, 0.0, 0.0)        # every ray has the exact direction (0, 0, -1)
        cam["y"][0] = (0.0, 1e-39, 0.0)      # or a denormal y component
        ctx.set_tuning("wide", wide)
        try:
            out.append(_frame(ctx, bvh, d_sh, len(s), lc, ctx.to_device(cam), w, h, 1, 3))
        finally:
            ctx.set_tuning("wide", 2)
    bvh.close()
    for a, b in ((out[0], out[1]), (out[2], out[3])):
        for x, y in zip(a, b):
            assert x.tobytes() == y.tobytes()


@pytest.mark.parametrize("orig", [(np.nan,) * 3, (np.inf, np.inf, np.inf), (-np.inf, np.inf, 0.5), (np.nan, 0.5, 0.5)])
def test_camera_not_finite(orig):
    """Rays that pass every box test reach the unused slots of nodes too: they end, and the image is the binary
    walk's."""
    say("case camera not finite", orig)
    s, lc, cam = _scene("soup", 65, 33)
    cam["orig"][0] = orig
    out = []
    with pt.Context(0) as ctx:
        d_sh, d_cam = ctx.to_device(s), ctx.to_device(cam)
        bvh = pt.CLBVH(ctx, d_sh)
        bvh.buildRadixTree()
        bvh.buildBVHTree()
        for quad, wide in ((8, 2), (0, 2), (0, 0)):
            ctx.set_tuning("quad", quad)
            ctx.set_tuning("wide", wide)
            out.append(_frame(ctx, bvh, d_sh, len(s), lc, d_cam, 65, 33, 1, 3))
        bvh.close()
    for a, b, c in zip(*out):
        assert a.tobytes() == b.tobytes()
        assert a.tobytes() == c.tobytes()
