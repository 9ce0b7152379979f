"""Runs after the other tests: the session's context still has the default launch settings, so they ran them."""
import pytest

import ptgpu_pc_amd as pt

pytestmark = pytest.mark.gpu


def test_session_context_has_the_defaults(ctx):
    with pt.Context(0) as fresh:
        for name in ("regroup", "blocks_per_cu", "wide", "quad", "stack", "short_stack", "batch_regroup",
                     "batch_blocks_per_cu"):
            assert ctx.get_tuning(name) == fresh.get_tuning(name), name
