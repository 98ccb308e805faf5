import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


def gpu_available() -> bool:
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle as O
    O.build()
    return O


@pytest.fixture(autouse=True)
def default_launch_state(request):
    """The library's launch settings are process-wide: whatever a GPU test pins is
    back at the choice by size for the next one."""
    yield
    if request.node.get_closest_marker("gpu"):
        from cochlearmodel_amd import _lib
        if os.path.exists(_lib.LIB_PATH):
            L = _lib.lib()
            L.cm_set_bm_order(None, 0)
            L.cm_reset_bm_launch()
            L.cm_reset_bm_jacobi_unroll()
            L.cm_reset_bm_sections_per_lane()
