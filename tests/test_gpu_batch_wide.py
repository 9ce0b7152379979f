"""A batch derives the four-wide nodes of its trees together, up to 32 a launch: batches of 1, 32, 33 and 70 jobs over
freshly built trees, some of them listed twice and some restructured, equal each job's own render bit for bit.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
from ptgpu_pc_amd import scenes
from ptgpu_pc_amd.layout import default_seeds

from test_gpu_batch import _run
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("njobs", [1, 32, 33, 70])
def test_trees_of_a_batch(ctx, njobs):
    say("case trees of a batch", njobs)
    jobs, d_all = [], []
    for k in range(njobs):
        w, h = 8 + k % 5, 6 + k % 3
        s, lc, cam = scenes.soup(2 + 17 * k, seed=k + 1, width=w, height=h)
        pt.update_camera(cam)
        d_all.append(ctx.to_device(s))
        jobs.append(dict(bvh=None, kd=None, shapes=d_all[-1], shapeCnt=len(s), lightCnt=lc, width=w, height=h, spp=1,
                         currentSample=0, max_depth=3, camera=ctx.to_device(cam),
                         colors0=np.zeros(w * h * 3, np.float32), seeds0=default_seeds(w, h)))
    handles = pt.CLBVH.create_batch(ctx, d_all)   # built, not walked
    for k, (j, h) in enumerate(zip(jobs, handles)):
        j["bvh"] = h
        if k % 11 == 5:
            h.optimize(5)
    jobs += [dict(jobs[0]), dict(jobs[njobs // 2])]   # listed twice
    got = _run(ctx, jobs, True)
    ref = _run(ctx, jobs, False)
    for a, b in zip(got, ref):
        for x, y in zip(a, b):
            assert x.tobytes() == y.tobytes()
    for h in handles:
        h.close()
