"""The launch-time models by which L1 gradients below the library's rule take the fp16 route or stay on the fp32 kernels: calls that were timed on both (us in the comments)."""
import importlib

import pytest
import torch

grad_module = importlib.import_module("kermac_amd.cdist_grad")       # the package attribute of that name is the function


def _route(L, M, N, O, K, p=1.0):
    batch = (L,) if L > 1 else ()
    a, b, c, d = (torch.empty(*batch, *shape) for shape in ((K, M), (N, K), (O, K), (N, M)))
    return grad_module._route_of_any_size(grad_module._plan_cdist_grad(a, b, c, d, None, p, require_device=False))


@pytest.fixture(autouse=True)
def no_switches(monkeypatch):
    for name in ("KERMAC_AMD_GRADIENT_WORKSPACE", "KERMAC_AMD_GRADIENT_F16_MIN_TERMS", "KERMAC_AMD_NO_CUT"):
        monkeypatch.delenv(name, raising=False)


def test_calls_that_the_route_makes_slower_stay():
    for shape in ((1, 8808, 37, 16, 174),        # fp32 44, route 53
                  (1, 5205, 9, 1, 256),          # 32, 35
                  (1, 10304, 675, 1, 175)):      # 117, 227
        assert _route(*shape) is None


def test_calls_that_the_route_makes_faster_take_it():
    for shape in ((2, 768, 28, 1, 1651),         # 191, 56
                  (1, 192, 22, 32, 1088),        # 118, 39
                  (1, 428, 18, 4, 256),          # 40, 23
                  (1, 1009, 254, 1, 1044)):      # 74, 48
        assert _route(*shape) is not None
        assert _route(*shape, p=2.0) is None     # the L2 gradient's pieces are not as exact as the fp32 kernels below the library's rule
