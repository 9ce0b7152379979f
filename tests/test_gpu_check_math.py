"""The render kernels' reciprocal, root and RGBA8 byte against the compiler's division, sqrtf and powf-based form (toInt,
vec.h:60), for every binary32 bit pattern: every image's bits rest on their being equal.
"""
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 1, 2], ids=["reciprocal", "root", "byte"])
def test_every_pattern(ctx, which):
    for first in range(0, 1 << 32, 1 << 30):
        say("case check math", which, hex(first))
        assert ctx.check_math(which, first, 1 << 30) == 0


# across the ends of the fast forms' ranges, where a wave holds both kinds of values: 2^-125 and 2^125, 2^-96 and 2^126,
# and around zero, the negatives and the NaN
@pytest.mark.parametrize("which,edges", [(0, (0x01000000, 0x7E000000, 0x81000000, 0xFE000000, 0, 0x7F800000)),
                                         (1, (0x0F800000, 0x7E800000, 0, 0x80000000, 0x7F800000)),
                                         (2, (0, 0x3F800000, 0x80000000, 0x7F800000))])
def test_ends_of_the_ranges(ctx, which, edges):
    for e in edges:
        for shift in range(0, 64, 7):
            assert ctx.check_math(which, (e - 192 + shift) & 0xFFFFFFFF, 384) == 0


def test_counts(ctx):
    assert ctx.check_math(0, 0, 0) == 0 and ctx.check_math(2, 123, 1) == 0
