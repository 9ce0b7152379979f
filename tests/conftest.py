import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
for p in (str(ROOT), str(ROOT / "oracle")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) device; runs through libptgpu.so")
    config.addinivalue_line("markers", "slow: long-running CPU test")


@pytest.fixture(scope="session")
def ctx():
    """One device context for the whole GPU session (fails loudly without a device)."""
    import ptgpu_pc_amd as pt
    c = pt.Context(0)
    yield c
    c.close()


_TUNING = ("regroup", "blocks_per_cu", "wide", "quad", "stack", "short_stack", "batch_regroup", "batch_blocks_per_cu")


@pytest.fixture(autouse=True)
def session_tuning(request):
    """The session's context leaves each test with the launch settings it came with (some tests restore numbers of their
    own, and those after them would run those settings instead of the defaults)."""
    if "ctx" not in request.fixturenames:
        yield
        return
    c = request.getfixturevalue("ctx")
    saved = {k: c.get_tuning(k) for k in _TUNING}
    yield
    for k, v in saved.items():
        c.set_tuning(k, v)
