"""Launch shapes of small frames: how many lanes of a wave take pixels and how many workgroups work follows from the
frame's pixels, the tree's height and, on the device, from where the camera is; the waves' first pixels follow from their
number, the others from a counter.  Every shape gives the bits of the fixed one (tuning blocks_per_cu 2, quad 0), and a
frame that is spread costs little where there is nothing to walk, and leaves room for frames in flight beside it.
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


def _scene(kind, w, h):
    """"mesh" and "deep" are seen from inside (32- and 48-entry stack classes), "soup" from outside, "far" from so far
    that the frame is background."""
    if kind in ("mesh", "deep"):
        s, lc, cam = scenes.icosphere_in_box(2 if kind == "mesh" else 5, seed=3, width=w, height=h)
    else:
        s, lc, cam = scenes.soup(3000, seed=6, width=w, height=h)
        if kind == "far":
            cam["orig"][0] = (0.5, 0.5, 30.5)
    pt.update_camera(cam)
    return s, lc, cam


class _Frames:
    def __init__(self, kind, w, h, contexts=1):
        s, lc, cam = _scene(kind, w, h)
        self.all = []
        for _ in range(contexts):
            ctx = pt.Context(0)
            d_sh = ctx.to_device(s)
            bvh = pt.CLBVH(ctx, d_sh)
            bvh.buildRadixTree()
            bvh.buildBVHTree()
            args = dict(colors=ctx.alloc(w * h * 12, F32).zero(), seeds=ctx.alloc(w * h * 8, np.uint32),
                        pixels=ctx.alloc(w * h * 4, np.uint32).zero(), camera=ctx.to_device(cam), shapes=d_sh,
                        shapeCnt=len(s), lightCnt=lc, width=w, height=h, spp=1, max_depth=5)
            self.all.append((ctx, bvh, ctx.to_device(default_seeds(w, h)), args))

    def tune(self, name, value):
        for ctx, *_ in self.all:
            ctx.set_tuning(name, value)

    def run(self, n):
        for k in range(n):
            ctx, bvh, seeds0, args = self.all[k % len(self.all)]
            ctx.synchronize()
            args["seeds"].copy_from(seeds0)
            pt.render(ctx, bvh, None, **args)
        for ctx, *_ in self.all:
            ctx.synchronize()

    def ms(self, n=30):
        self.run(2 * len(self.all))
        best = 1e9
        for _ in range(4):
            t = time.perf_counter()
            self.run(n)
            best = min(best, (time.perf_counter() - t) / n)
        return 1e3 * best

    def result(self):
        args = self.all[0][3]
        return [args[k].download(np.uint32) for k in ("colors", "seeds", "pixels")]

    def close(self):
        for ctx, bvh, *_ in self.all:
            bvh.close()
            ctx.close()


# around the limits of each share on 256 CUs: 4096, 8192, 16384 and 32768 pixels, inside 12288 and 20480 for "mesh"
@pytest.mark.parametrize("w,h", [(1, 3), (64, 48), (439, 7), (64, 64), (241, 17), (96, 64), (1229, 5), (2731, 3), (3277, 5), (96, 128), (4097, 3),
                                 (192, 128), (3511, 7), (182, 180), (331, 99), (128, 64), (128, 128), (160, 128),
                                 (10241, 2), (256, 128)])
@pytest.mark.parametrize("kind", ["mesh", "deep", "soup"])
def test_shapes_same_bits(kind, w, h):
    say("case frame shapes", kind, w, h)
    f = _Frames(kind, w, h)
    f.run(1)
    got = f.result()
    f.tune("blocks_per_cu", 2)
    f.tune("quad", 0)
    f.run(1)
    for a, b in zip(got, f.result()):
        assert a.tobytes() == b.tobytes()
    f.close()


@pytest.mark.parametrize("kind,w,h,contexts", [("far", 64, 64, 1), ("far", 128, 64, 3), ("mesh", 256, 128, 3),
                                               ("mesh", 180, 180, 3)])
def test_spread_leaves_room(kind, w, h, contexts):
    """Against 64 pixels a wave: background took up to twice as long (117 / 60 us alone, 92 / 43 in flight), a closed
    mesh with three frames in flight 265 / 147 us a frame."""
    say("case spread", kind, w, h, contexts)
    f = _Frames(kind, w, h, contexts)
    default = f.ms()
    f.tune("blocks_per_cu", 2)
    fixed = f.ms()
    say(f"  default {default:.4f} ms, 64 pixels a wave {fixed:.4f} ms")
    f.close()
    assert default < 1.3 * fixed


@pytest.mark.parametrize("accel,most", [("kd", 0.75), ("kd_sah", 0.9), ("index", 0.9)])
@pytest.mark.parametrize("w,h", [(64, 112), (129, 64), (128, 112), (260, 75), (182, 180), (331, 99)])
def test_long_walks_share(accel, most, w, h):
    """KD trees and index-keyed ones, seen from inside: shared up to 32,768 pixels, with the bits of 64 pixels a wave (their
    times, 22,500 pixels of the 5,132-shape mesh: 379 against 719 us, SAH 356 / 494, index-keyed 496 / 644)."""
    say("case long walks", accel, w, h)
    s, lc, cam = scenes.icosphere_in_box(4, seed=3, width=w, height=h)
    pt.update_camera(cam)
    with pt.Context(0) as ctx:
        d_sh = ctx.to_device(s)
        bvh = kd = None
        if accel == "index":
            bvh = pt.CLBVH(ctx, d_sh, traversal="reference")
            bvh.buildRadixTree()
            bvh.buildBVHTree()
        else:
            kd = pt.KDTree(ctx, s, sah=accel == "kd_sah", max_depth=24, max_leaf=4) if accel == "kd_sah" else pt.KDTree(ctx, s)
        seeds = ctx.to_device(default_seeds(w, h))
        col, sd = ctx.alloc(w * h * 12, F32).zero(), ctx.alloc(w * h * 8, np.uint32)
        args = dict(colors=col, seeds=sd, camera=ctx.to_device(cam), shapes=d_sh, shapeCnt=len(s), lightCnt=lc, width=w,
                    height=h, spp=1, max_depth=5)

        def best():
            ms = []
            for _ in range(12):
                sd.copy_from(seeds)
                ctx.record(0)
                pt.render(ctx, bvh, kd, **args)
                ctx.record(1)
                ms.append(ctx.elapsed_ms(0, 1))
            return min(ms[2:]), col.download(np.uint32).tobytes() + sd.download(np.uint32).tobytes()

        default, bits = best()
        ctx.set_tuning("blocks_per_cu", 4)
        fixed, same = best()
        say(f"  default {default:.4f} ms, 64 pixels a wave {fixed:.4f} ms")
        assert bits == same
        assert default < (most if w * h <= 32768 else 1.05) * fixed
