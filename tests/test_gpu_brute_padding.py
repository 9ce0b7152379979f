"""Brute-force frames whose primitives are no multiple of four: the last group's empty places cost no more than
primitives there would (they used to send all four to the general intersection).
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
from ptgpu_pc_amd import scenes
from ptgpu_pc_amd.layout import concat_shapes, default_seeds

from test_gpu_parity import say

pytestmark = pytest.mark.gpu
F32 = np.float32


def _ms(ctx, n, w=256, h=256):
    """The nine Cornell spheres and n - 9 more, far away and small, before them."""
    s, lc, cam = scenes.cornell(w, h)
    pt.update_camera(cam)
    far = s[[6] * (n - 9)].copy()
    far["p"] = (1e4, 1e4, 1e4)
    far["rad"] = 1.0
    s = concat_shapes([far, s]) if n > 9 else s
    s["index"] = np.arange(n)
    args = dict(colors=ctx.alloc(w * h * 12, F32).zero(), seeds=ctx.alloc(w * h * 8, np.uint32), camera=ctx.to_device(cam),
                shapes=ctx.to_device(s), shapeCnt=n, lightCnt=lc, width=w, height=h, spp=4, max_depth=5)
    seeds0 = ctx.to_device(default_seeds(w, h))
    best = 1e9
    for _ in range(12):
        args["seeds"].copy_from(seeds0)
        ctx.record(0)
        pt.render(ctx, None, None, **args)
        ctx.record(1)
        best = min(best, ctx.elapsed_ms(0, 1))
    return best, args["colors"].download(F32)


@pytest.mark.parametrize("n,full", [(9, 12), (10, 12), (13, 16), (14, 16)])
def test_empty_places(ctx, n, full):
    """10 spheres 0.206 ms and 12 spheres 0.178, before; 0.178 both now."""
    say("case empty places", n, full)
    (a, image), (b, other) = _ms(ctx, n), _ms(ctx, full)
    say(f"  {n} spheres {a:.4f} ms, {full} spheres {b:.4f} ms")
    assert image.tobytes() == other.tobytes()
    if n % 4 == 2:
        assert a < 1.07 * b
