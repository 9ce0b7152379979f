"""Batch queries over binary16 four-wide nodes: how many lanes of a wave take rays (1, 2, 4, 8 or all) follows the
number of rays, waves own runs of them, and trees that binary16 bounds blur are walked over their binary nodes.
Every answer equals the binary-node walk's of the same tree bit for bit (the closest hit is the least t, then the
higher id, whatever the order), and the oracle's brute force (Intersect / IntersectP, rendering_kernel.cl:486-560).
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
import pyoracle as O
from ptgpu_pc_amd import scenes

from test_gpu_parity import assert_closest_parity, gpu_trace, random_rays, say

pytestmark = pytest.mark.gpu
F32 = np.float32


def _moved(shapes, offset):
    """The scene moved by `offset` along each axis (triangles and bounds; the scenes used here have no spheres)."""
    s = shapes.copy()
    assert (s["type"] != 0).all()
    for f in ("p1", "p2", "p3"):
        s[f] = s[f] + F32(offset)
    s["b"] = np.concatenate([np.minimum(np.minimum(s["p1"], s["p2"]), s["p3"]),
                             np.maximum(np.maximum(s["p1"], s["p2"]), s["p3"])], axis=1)
    return s


def _both_walks(ctx, bvh, kd, d_sh, n, rays, maxt):
    out = []
    for wide in (2, 0):
        ctx.set_tuning("wide", wide)
        try:
            out.append((*gpu_trace(ctx, bvh, kd, d_sh, n, rays), gpu_trace(ctx, bvh, kd, d_sh, n, rays, maxt)))
        finally:
            ctx.set_tuning("wide", 2)
    for a, b in zip(*out):
        assert a.tobytes() == b.tobytes()
    return out[0]


def _maxt(rays, seed):
    m = np.random.default_rng(seed).random(len(rays)).astype(F32)
    m[::7] = 0.0
    m[1::7] = 1e20
    return m


# one ray; a wave and its neighbours; around 4096, 8192, 16384 and 32768 rays, where 1, 2, 4, 8 and 64 lanes of a wave
# take them; more than one ray per lane of the launch
@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 1027, 4096, 4097, 8193, 16385, 32768, 32769, 300007])
@pytest.mark.parametrize("accel", ["bvh", "kd_sah"])
def test_ray_counts(ctx, accel, n):
    say("case ray counts", accel, n)
    s = scenes.soup(3000, seed=31)[0]
    rays = random_rays(n, n)
    d_sh = ctx.to_device(s)
    bvh = kd = None
    if accel == "bvh":
        bvh = pt.CLBVH(ctx, d_sh)
        bvh.buildRadixTree()
        bvh.buildBVHTree()
    else:
        kd = pt.KDTree(ctx, s, sah=True, max_depth=24, max_leaf=4)
    maxt = _maxt(rays, n)
    t, ids, hit = _both_walks(ctx, bvh, kd, d_sh, len(s), rays, maxt)
    if n <= 1027:
        t_o, id_o = O.trace_closest(s, O.accel_none(), rays)
        if n >= 64:
            assert_closest_parity(t, ids, t_o, id_o)
            assert (hit == O.trace_any(s, rays, maxt)).mean() >= 0.9999
        else:
            assert (ids == id_o).all()


# every stack class
@pytest.mark.parametrize("key,value", [("stack", 48), ("stack", 64), ("short_stack", 0),
                                       ("quad", 0)])
def test_stack_classes(key, value):
    say("case stack classes", key, value)
    s = scenes.soup(3000, seed=32)[0]
    rays = random_rays(5001, 4)
    with pt.Context(0) as ctx:
        d_sh = ctx.to_device(s)
        bvh = pt.CLBVH(ctx, d_sh)
        bvh.buildRadixTree()
        bvh.buildBVHTree()
        if key == "short_stack":
            ctx.set_tuning("stack", 48)
        ctx.set_tuning(key, value)
        _both_walks(ctx, bvh, None, d_sh, len(s), rays, _maxt(rays, 5))
        bvh.close()


@pytest.mark.parametrize("n", [1, 2, 3, 5])
def test_smallest_trees(ctx, n):
    say("case smallest trees", n)
    s = scenes.soup(64, seed=33)[0][-n:].copy()
    s["index"] = np.arange(n)
    d_sh = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d_sh)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    rays = random_rays(777, n)
    c = s["b"][:, :3][np.arange(777) % n] * F32(0.5) + s["b"][:, 3:][np.arange(777) % n] * F32(0.5)
    d = c - rays["o"]
    rays["d"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(F32)   # towards the shapes
    _both_walks(ctx, bvh, None, d_sh, n, rays, _maxt(rays, n))


def test_unusual_rays(ctx):
    """Zero, denormal, huge, infinite and NaN components; origins on box planes and far away; limits of 0, below 0,
    infinite and NaN."""
    say("case unusual rays")
    s = scenes.soup(3000, seed=34)[0]
    d_sh = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d_sh)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    rays = random_rays(4200, 6)
    odd = np.array([0.0, -0.0, 1e-39, -1e-39, 1e-30, 1e30, -1e30, 3e38, np.inf, -np.inf, np.nan, 1e-7], F32)
    for k in range(3):
        rays["d"][k * 400:(k + 1) * 400, k] = odd[np.arange(400) % 12]
        rays["o"][1200 + k * 300:1200 + (k + 1) * 300, k] = odd[np.arange(300) % 12]
        rays["o"][2100 + k * 300:2100 + (k + 1) * 300, k] = s["b"][np.arange(300) * 7, k]
        rays["d"][2100 + k * 300:2100 + (k + 1) * 300, (k + 1) % 3] = 0.0
    rays["o"][3000:3300] -= rays["d"][3000:3300] * F32(1e4)
    rays["d"][3300:3400] = 0.0
    rays["d"][3400:3500] *= F32(1e3)
    rays["d"][3500:3600] *= F32(1e-3)
    maxt = _maxt(rays, 8)
    maxt[3600:3700] = np.inf
    maxt[3700:3800] = np.nan
    maxt[3800:3900] = -1.0
    _both_walks(ctx, bvh, None, d_sh, len(s), rays, maxt)


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_rays_in_box_planes(ctx, axis):
    """Rays with zero direction components from planes that boxes on both sides share, at zero and elsewhere: both
    sides' boxes are walked.  Three layers of a grid of triangles on multiples of 1/8, where every test is exact: a
    ray through an edge or a corner hits all its triangles at one t, and the answer is the highest of their ids.
    (Not compared with the binary nodes' walk, whose test drops a box that has the origin on its bound.)"""
    say("case rays in box planes", axis)
    i, j, k = (v.ravel() for v in np.meshgrid(np.arange(-8, 8), np.arange(-8, 8), np.arange(3), indexing="ij"))
    lo = np.stack([i, j, -k], axis=1) / 8.0
    corner = lambda dx, dy: np.roll(lo + np.array([dx, dy, 0.0]) / 8.0, axis, axis=1).astype(F32)
    s = scenes.soup(2 * len(lo), seed=1)[0][-2 * len(lo):].copy()
    s["p1"], s["p2"], s["p3"] = (np.concatenate(v) for v in ((corner(0, 0), corner(1, 1)), (corner(1, 0), corner(0, 1)),
                                                             (corner(0, 1), corner(1, 0))))
    s["b"] = _moved(s, 0.0)["b"]
    s, _ = O.clbvh_construct(s)
    x, y = (v.ravel() for v in np.meshgrid(np.arange(-17, 18), np.arange(-17, 18), indexing="ij"))
    rays = random_rays(2 * len(x), 1)
    o = np.stack([x / 16.0, y / 16.0, np.ones(len(x))], axis=1)
    rays["o"] = np.roll(np.concatenate([o, o]), axis, axis=1).astype(F32)
    d = np.concatenate([np.tile([0.0, 0.0, -1.0], (len(x), 1)), np.tile([-0.0, -0.0, -1.0], (len(x), 1))])
    rays["d"] = np.roll(d, axis, axis=1).astype(F32)
    d_sh = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d_sh)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    t, ids = gpu_trace(ctx, bvh, None, d_sh, len(s), rays)
    t_o, id_o = O.trace_closest(s, O.accel_none(), rays)
    assert (id_o >= 0).sum() > 1000
    np.testing.assert_array_equal(ids, id_o)
    np.testing.assert_array_equal(t[id_o >= 0], t_o[id_o >= 0])


# binary16 bounds are absolute: from offsets of some tens of the scene's size on they blur its shapes
@pytest.mark.parametrize("offset", [0.0, 8.0, 40.0, 1000.0, 60000.0, 70000.0])
def test_far_scenes(ctx, offset):
    say("case far scenes", offset)
    s = _moved(scenes.soup(3000, seed=35)[0][2:], offset)
    d_sh = ctx.to_device(s)
    rays = random_rays(9001, 7)
    rays["o"] += F32(offset)
    maxt = _maxt(rays, 9)
    bvh = pt.CLBVH(ctx, d_sh)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    _both_walks(ctx, bvh, None, d_sh, len(s), rays, maxt)
    kd = pt.KDTree(ctx, s, sah=True, max_depth=24, max_leaf=4)
    _both_walks(ctx, None, kd, d_sh, len(s), rays, maxt)
