"""The light list of a frame without a handle: built per call over chunks of 4096 shapes, its length left on the device.
Emitters at the edges of chunks, and lists shorter and longer than the stated number of lights, against the oracle
(SampleLights, rendering_kernel.cl:415-490): colours and seeds bit for bit.
"""
import numpy as np
import pytest

import ptgpu_pc_amd as pt
import pyoracle as O
from ptgpu_pc_amd import scenes

from test_gpu_brute_lds import _frame
from test_gpu_parity import image_checks, render_oracle, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,emitters", [(1, [0]), (255, [254]), (257, [0, 255, 256]), (4096, [0, 4095]), (4097, [4095, 4096]),
                                        (8193, [1, 4096, 8191, 8192])])
@pytest.mark.parametrize("stated", [0, 1, 3, 7])
def test_light_list(ctx, n, emitters, stated):
    say("case light list", n, stated)
    w, h = 9, 7
    s = scenes.soup(max(n, 4), seed=n)[0][-n:].copy()
    s["e"] = 0
    for k in emitters:
        s["e"][k] = (2, 3, 1)
    _, _, cam = scenes.soup(16, seed=1, width=w, height=h)
    pt.update_camera(cam)
    got = _frame(ctx, s, stated, cam, w, h, 1, 3)
    image_checks(*got, *render_oracle(s, stated, cam, w, h, 1, 3, O.accel_none()))
