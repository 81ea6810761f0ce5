import os
import sys

import pytest

# The few tests that run torch's own convolutions on the GPU (the VAE decoder's library path) would otherwise spend
# most of a minute in the convolution library's exhaustive algorithm search, and log every missing solver.
os.environ.setdefault("MIOPEN_FIND_MODE", "2")
os.environ.setdefault("MIOPEN_LOG_LEVEL", "1")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


def _has_gpu():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


def pytest_collection_modifyitems(config, items):
    if _has_gpu():
        return
    skip = pytest.mark.skip(reason="no GPU in this environment")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(autouse=True)
def _nothing_kept_for_backwards(request):
    """Whether a Monarch forward under autograd leaves its intermediates follows what became of earlier ones: every GPU test starts
    as a program does, whatever ran before it."""
    if "gpu" in request.keywords:
        import self_forcing_amd as sfa
        sfa.monarch_attn._KEPT.clear()
    yield
