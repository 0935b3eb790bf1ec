import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def device():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.fixture(params=["64x64", "128x128"])
def direct_tile(request, monkeypatch):
    """Both tiles of the direct kernel for the small results of a test: 64 x 64 by the library's rule, and the 128 x 128 of larger results."""
    if request.param == "128x128":
        monkeypatch.setenv("KERMAC_AMD_DIRECT_SMALL_MAX_TILES", "0")
    return request.param


@pytest.fixture(params=["by the rule", "256x128"])
def product_tile(request, monkeypatch):
    """Both tiles of the workspace route's product kernel for the small results of a test: 128 x 128 by the library's rule, and 256 x 128."""
    if request.param == "256x128":
        monkeypatch.setenv("KERMAC_AMD_WIDE_LARGE_TILE_MIN_TILES", "1")
    return request.param
