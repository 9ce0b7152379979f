"""Builds of at most one sort tile (4,096 shapes) sort in one workgroup: order, codes and trees at its edges equal the
oracle's (a stable sort by descending code, CLBVH.cpp:166-211), for spread, few and equal codes and both digit widths.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
import pyoracle as O
from ptgpu_pc_amd.layout import SHAPE_DTYPE

from test_gpu_morton_tree import _spheres
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1025, 4095, 4096, 4097])
@pytest.mark.parametrize("kind", ["spread", "repeated", "equal"])
def test_small_sort(ctx, kind, n, bits):
    say("case small sort", kind, n, bits)
    s = _spheres(kind, n)
    ref_s, ref_sorted, ref_btn, ref_btl = O.build_lbvh(s)
    d = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d, digit_bits=bits)
    for _ in range(2):   # a rebuild finds the counters of the build before it
        bvh.reset()
        bvh.buildRadixTree()
        bvh.buildBVHTree()
    np.testing.assert_array_equal(bvh.sorted_indices(), ref_sorted)
    np.testing.assert_array_equal(d.download(SHAPE_DTYPE)["morton_code"], ref_s["morton_code"])
    btn, btl = bvh.getTrees()
    if n > 1:
        np.testing.assert_array_equal(btn.view(np.uint8), ref_btn.view(np.uint8))
        assert bvh.export_traversal()[2] >= 1
    np.testing.assert_array_equal(btl.view(np.uint8), ref_btl.view(np.uint8))
    bvh.close()
