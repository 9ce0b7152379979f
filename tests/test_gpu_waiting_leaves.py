"""KD trees in the binary16 walk: leaves wait until enough lanes of a wave have one, or lanes can do nothing else.  Frames
and queries equal the binary-node walk's bit for bit, whatever the number of lanes at work (one pixel or ray, sparse
waves with and without shared queries, full waves) and in each stack class.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
from ptgpu_pc_amd import scenes
from ptgpu_pc_amd.layout import default_seeds

from test_gpu_parity import random_rays, say
from test_gpu_query_walk import _both_walks, _maxt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf", [1, 4, 16])
@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (64, 65), (300, 200)])
@pytest.mark.parametrize("stack", [0, 48, 64])
def test_kd_frames(stack, w, h, leaf):
    say("case waiting leaves", stack, w, h, leaf)
    s, lc, cam = scenes.soup(3000, seed=12, width=w, height=h)
    pt.update_camera(cam)
    out = []
    with pt.Context(0) as ctx:
        d_sh, d_cam = ctx.to_device(s), ctx.to_device(cam)
        kd = pt.KDTree(ctx, s, sah=True, max_depth=24, max_leaf=leaf)
        ctx.set_tuning("stack", stack)
        for quad, wide in ((16, 2), (0, 2), (0, 0)):
            ctx.set_tuning("quad", quad)
            ctx.set_tuning("wide", wide)
            col = ctx.alloc(w * h * 12, np.float32).zero()
            seeds = ctx.to_device(default_seeds(w, h))
            pix = ctx.alloc(w * h * 4, np.uint32)
            pt.render(ctx, None, kd, colors=col, seeds=seeds, camera=d_cam, shapes=d_sh, shapeCnt=len(s), lightCnt=lc,
                      width=w, height=h, spp=2, max_depth=4, pixels=pix)
            ctx.synchronize()
            out.append((col.download(np.float32), seeds.download(np.uint32), pix.download(np.uint32)))
    for a, b, c in zip(*out):
        assert a.tobytes() == b.tobytes()
        assert a.tobytes() == c.tobytes()


@pytest.mark.parametrize("leaf", [1, 16])
@pytest.mark.parametrize("n", [1, 40, 4097, 70001])
def test_kd_queries(ctx, n, leaf):
    say("case waiting leaves, queries", n, leaf)
    s = scenes.soup(3000, seed=13)[0]
    kd = pt.KDTree(ctx, s, sah=True, max_depth=24, max_leaf=leaf)
    rays = random_rays(n, n)
    _both_walks(ctx, None, kd, ctx.to_device(s), len(s), rays, _maxt(rays, n))
