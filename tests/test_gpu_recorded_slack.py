"""A frame recorded right after its tree's build, when the height is not known to the host, shares its queries as the same
calls issued one by one do: the kernel reads the height it was built with.
"""
import time

import numpy as np
import pytest

import ptgpu_pc_amd as pt
from ptgpu_pc_amd import scenes
from ptgpu_pc_amd.layout import default_seeds

from test_gpu_parity import say

pytestmark = pytest.mark.gpu
F32 = np.float32


# the 48-entry class (on the short stack), the 32-entry one, and the 48-entry one without the short stack
@pytest.mark.parametrize("n,short", [(65536, 1), (2000, 1), (65536, 0)])
def test_recorded_step(n, short):
    w, h = 97, 61
    say("case recorded step", n, short)
    s, lc, cam = scenes.soup(n, seed=1, width=w, height=h)
    pt.update_camera(cam)
    with pt.Context(0) as ctx:
        ctx.set_tuning("short_stack", short)
        d_sh = ctx.to_device(s)
        bvh = pt.CLBVH(ctx, d_sh)
        sd0, sd = ctx.to_device(default_seeds(w, h)), ctx.alloc(w * h * 8, np.uint32)
        col, pix = ctx.alloc(w * h * 12, F32).zero(), ctx.alloc(w * h * 4, np.uint32)
        d_cam = ctx.to_device(cam)

        def step():
            bvh.reset()
            bvh.buildRadixTree()
            bvh.buildBVHTree()
            ctx.memcpy_async(sd, sd0, w * h * 8)
            pt.render(ctx, bvh, None, colors=col, seeds=sd, camera=d_cam, shapes=d_sh, shapeCnt=len(s), lightCnt=lc,
                      width=w, height=h, spp=1, max_depth=5, pixels=pix)

        def ms(fn):
            best = 1e9
            for _ in range(5):
                t = time.perf_counter()
                for _ in range(10):
                    fn()
                    ctx.synchronize()
                best = min(best, (time.perf_counter() - t) / 10)
            return 1e3 * best

        step()
        ctx.synchronize()
        want = [x.download(np.uint32).tobytes() for x in (col, sd, pix)]
        eager = ms(step)
        ctx.graph_begin()
        try:
            step()
        finally:
            g = ctx.graph_end()
        for _ in range(3):
            col.zero()
            g.launch()
            ctx.synchronize()
            assert [x.download(np.uint32).tobytes() for x in (col, sd, pix)] == want
        recorded = ms(g.launch)
        say(f"  eager {eager:.4f} ms, recorded {recorded:.4f} ms")
        g.close()
        bvh.close()
    assert recorded < 1.08 * eager
