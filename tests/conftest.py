import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def orc():
    import oracle
    oracle.lib()
    return oracle


@pytest.fixture(scope="session")
def rt():
    from vpux_plugin_amd import runtime
    runtime.lib()
    return runtime


@pytest.fixture
def without_nce_direct(rt):
    """Layers that are over before a tile is staged run nce_direct; without it they run the kernel that serves their family at
    larger sizes, which is what a test that names one is about."""
    rt.set_tuning("VPX_NCE_DIRECT", "off")
    yield
    rt.set_tuning("VPX_NCE_DIRECT", None)


@pytest.fixture(scope="session")
def dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")
