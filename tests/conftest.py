import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


@pytest.fixture(scope="session")
def lbmoe():
    """The loaded C-ABI library; built in-tree first when hipcc is present and it or the host
    extension is missing."""
    from layerbatch_amd import _lib, build
    if not (os.path.exists(_lib.LIB_PATH) and os.path.exists(build.HOST)):
        build.build()
    return _lib.lib()


@pytest.fixture(scope="session")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible")
    return torch.device("cuda:0")
