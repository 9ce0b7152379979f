"""The Morton-keyed traversal tree, built bottom-up over lists of 128 leaves and then over sixteen lists' leftovers
at a time: topology, node numbering, boxes and height equal the radix tree's over the sorted codes, at the edges
of a list and of each level, for codes that are spread, repeated, all equal and of few bits (the most leftovers).
Whole numbers and boxes are compared exactly.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
from ptgpu_pc_amd.layout import SHAPE_DTYPE

from test_gpu_parity import SPHERE, check_traversal_tree, say

pytestmark = pytest.mark.gpu
F32 = np.float32


def _spheres(kind, n):
    s = np.zeros(n, dtype=SHAPE_DTYPE)
    s["type"] = SPHERE
    s["rad"] = 0.01
    rng = np.random.default_rng(n)
    if kind == "spread":
        p = rng.random((n, 3))
    elif kind == "repeated":
        p = np.round(rng.random((n, 3)) * 3) / 3
    elif kind == "equal":
        p = np.full((n, 3), 0.25)
        p[0] = 0.0
        p[-1] = 1.0
    else:   # few bits: every cell coordinate a power of two of 1024
        p = 2.0 ** rng.integers(-10, 1, (n, 3))
        p[0] = 0.0
        p[-1] = 1.0
    s["p"] = p.astype(F32)
    return s


def _radix_tree(codes):
    """(left, right, first, last) per internal node and the height, by the definition: a range splits where its
    adjacent prefix is shortest; a left child is numbered by its last leaf, any other node by its first."""
    n = len(codes)
    keys = (~codes.astype(np.int64)) & 0x3FFFFFFF
    assert (np.diff(keys) >= 0).all()
    pre = np.empty(n - 1, np.int64)   # prefix length of leaves k and k + 1
    for k in range(n - 1):
        x = int(keys[k] ^ keys[k + 1])
        pre[k] = 32 - x.bit_length() if x else 64 - (k ^ (k + 1)).bit_length()
    # the tree of least prefixes over the splits, by a stack; then ranges from the root down
    left, right, stack = [-1] * (n - 1), [-1] * (n - 1), []
    for k in range(n - 1):
        last = -1
        while stack and pre[stack[-1]] > pre[k]:
            last = stack.pop()
        left[k] = last
        if stack:
            right[stack[-1]] = k
        stack.append(k)
    refs = np.zeros((n - 1, 4), np.int64)
    depth_max, todo = 0, [(stack[0], 0, n - 1, 0, 1)]   # split, first, last, number, depth
    while todo:
        k, lo, hi, num, depth = todo.pop()
        depth_max = max(depth_max, depth)
        refs[num] = (~k if lo == k else k, ~hi if hi == k + 1 else k + 1, lo, hi)
        if lo < k:
            todo.append((left[k], lo, k, k, depth + 1))
        if k + 1 < hi:
            todo.append((right[k], k + 1, hi, k + 1, depth + 1))
    return refs, depth_max


@pytest.mark.parametrize("n", [2, 3, 64, 127, 128, 129, 257, 2048, 2049, 32768, 32769])
@pytest.mark.parametrize("kind", ["spread", "repeated", "equal", "few bits"])
def test_tree_equals_definition(ctx, kind, n):
    say("case morton tree", kind, n)
    s = _spheres(kind, n)
    d = ctx.to_device(s)
    bvh = pt.CLBVH(ctx, d)
    bvh.buildRadixTree()
    bvh.buildBVHTree()
    out = d.download(SHAPE_DTYPE)
    refs, _, height = bvh.export_traversal()
    ref, ref_height = _radix_tree(out["morton_code"][bvh.sorted_indices()])
    np.testing.assert_array_equal(np.asarray(refs).reshape(-1, 4), ref)
    assert height == ref_height
    if n <= 2049:
        check_traversal_tree(bvh, out)
    bvh.close()
