"""Batch queries along directions of any length.  A ray in an axis plane has an infinite reciprocal on that axis, which
the binary16 slab test holds to a finite one; beside a direction that is short altogether its box would seem
to end before the others begin.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
import pyoracle as O
from ptgpu_pc_amd import scenes

from test_gpu_parity import gpu_trace, random_rays, say

pytestmark = pytest.mark.gpu
F32 = np.float32


# length 1; the shortest whose farthest hit stays below the limit of closest hits (1e20); one between
@pytest.mark.parametrize("exponent", [0, -40, -63])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_short_directions_in_planes(ctx, axis, exponent):
    """Three layers of a grid of triangles on multiples of 1/8, looked at along an axis from points on and between
    its lines, and from 2^-70 beside the lines at zero (inside the boxes on one side only): the brute force's hits."""
    say("case short directions", axis, exponent)
    i, j, k = (v.ravel() for v in np.meshgrid(np.arange(-8, 8), np.arange(-8, 8), np.arange(3), indexing="ij"))
    lo = np.stack([i, j, -k], axis=1) / 8.0
    corner = lambda dx, dy: np.roll(lo + np.array([dx, dy, 0.0]) / 8.0, axis, axis=1).astype(F32)
    s = scenes.soup(2 * len(lo), seed=1)[0][-2 * len(lo):].copy()
    s["p1"], s["p2"], s["p3"] = (np.concatenate(v) for v in ((corner(0, 0), corner(1, 1)), (corner(1, 0), corner(0, 1)),
                                                             (corner(0, 1), corner(1, 0))))
    p = np.stack([s["p1"], s["p2"], s["p3"]], axis=1)
    s["b"] = np.concatenate([p.min(axis=1), p.max(axis=1)], axis=1)
    s, _ = O.clbvh_construct(s)
    x, y = (v.ravel() for v in np.meshgrid(np.arange(-17, 18), np.arange(-17, 18), indexing="ij"))
    rays = random_rays(3 * len(x), 1)
    o = np.concatenate([np.stack([x / 16.0 + e, y / 16.0 + e, np.ones(len(x))], axis=1) for e in (0.0, -2.0 ** -70, 2.0 ** -70)])
    d = np.tile([0.0, 0.0, -(2.0 ** exponent)], (len(o), 1))
    rays["o"] = np.roll(o, axis, axis=1).astype(F32)
    rays["d"] = np.roll(d, axis, axis=1).astype(F32)
    d_sh = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d_sh)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    t, ids = gpu_trace(ctx, bvh, None, d_sh, len(s), rays)
    t_o, id_o = O.trace_closest(s, O.accel_none(), rays)
    assert (id_o >= 0).sum() > 1500
    np.testing.assert_array_equal(ids, id_o)
    np.testing.assert_array_equal(t[id_o >= 0], t_o[id_o >= 0])
    maxt = np.full(len(rays), 1e20, F32)
    np.testing.assert_array_equal(gpu_trace(ctx, bvh, None, d_sh, len(s), rays, maxt), O.trace_any(s, rays, maxt))
    bvh.close()
