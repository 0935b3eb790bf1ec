"""Calls that take a route through fp16 pieces although the library's own rule does not ask for it: on heavy-tailed values, values offset from the origin and features
of very different scales their error against float64 is no larger than that of the kernels that run without a workspace.

Tolerances, in units of the error of those kernels: 1.05 for the 2-norm (0.08 .. 1.02 measured over 240 calls of squared differences and their products, 0.2 .. 0.8 over 60 L1
gradients) and 1.5 for the largest error of a value (at most 1.21 and 0.8)."""
import importlib

import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu

grad_module = importlib.import_module("kermac_amd.cdist_grad")       # the package attribute of that name is the function
GAUSSIAN = kermac.KernelDescriptor(kermac.InnerOperator.DIFF, kermac.PowerType.SQUARE, kermac.PowerType.NOOP, kermac.KernelType.GAUSSIAN)
KINDS = ["normal", "heavy", "offset", "scaled"]


def _values(kind, shape, device, g):
    x = torch.randn(*shape, device=device, generator=g)
    if kind == "heavy":
        x = x / torch.rand(*shape, device=device, generator=g).clamp_min(1e-3)
    return x + 30.0 if kind == "offset" else x


def _scales(kind, K, device, g, decades=6.0):
    return 10.0 ** (decades * (torch.rand(K, device=device, generator=g) - 0.5)) if kind == "scaled" else torch.ones(K, device=device)


def _points(kind, L, rows, scales, k_contiguous, device, g):
    x = _values(kind, (L, rows, len(scales)), device, g) * scales
    return x if k_contiguous else x.transpose(-1, -2).contiguous().transpose(-1, -2)


def _squares(a, b):
    return torch.stack([torch.cdist(x, y, compute_mode="donot_use_mm_for_euclid_dist") for x, y in zip(a.double(), b.double())]) ** 2


def _no_worse(got, before, want):
    error, error_before = ((x.double().reshape(want.shape) - want).abs() for x in (got, before))
    assert float(error.norm()) <= 1.05 * float(error_before.norm())
    assert float(error.max()) <= 1.5 * float(error_before.max())


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("L,M,N,K,k_contiguous", [(1, 600, 3000, 250, True), (2, 448, 1420, 2048, False), (4, 900, 1900, 70, True), (1, 1950, 3100, 213, False),
                                                  (4, 257, 385, 1440, True)])
def test_squared_differences(device, monkeypatch, kind, L, M, N, K, k_contiguous):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    scales = _scales(kind, K, device, g)
    a, b = (_points(kind, L, rows, scales, k_contiguous, device, g) for rows in (M, N))
    call = lambda: kermac.cdist(a, b, p=2.0)
    assert any("gram_f16_wide" in name for name in kernels_of(call))
    got = call()
    monkeypatch.setenv("KERMAC_AMD_L2_WORKSPACE", "0")
    assert not any("gram_f16_wide" in name for name in kernels_of(call))
    _no_worse(got, call(), _squares(a, b).sqrt())


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("L,M,N,K,O", [(1, 303, 1500, 200, 10), (2, 640, 900, 1100, 32), (1, 3001, 2960, 97, 1), (4, 400, 500, 384, 3)])
def test_products_with_coefficients(device, monkeypatch, kind, L, M, N, K, O):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    scales = _scales(kind, K, device, g)
    a, b = (_points(kind, L, rows, scales, True, device, g) for rows in (M, N))
    coef = torch.randn(L, N, O, device=device, generator=g)
    squares = _squares(a, b)
    bandwidth = float(squares.median()) ** 0.5
    call = lambda: kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=bandwidth)
    assert any("gram_f16_wide" in name for name in kernels_of(call))
    got = call()
    monkeypatch.setenv("KERMAC_AMD_L2_WORKSPACE", "0")
    assert not any("gram_f16_wide" in name for name in kernels_of(call))
    _no_worse(got, call(), torch.exp(-squares / (2 * bandwidth ** 2)) @ coef.double())


# rows of a scaled over 8 decades, those of c by the inverse: the pieces are of their products
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("L,M,N,O,K", [(1, 428, 18, 4, 256), (1, 201, 33, 1, 471), (2, 64, 11, 1, 1301), (1, 1045, 24, 10, 5706), (1, 192, 22, 33, 1088)])
def test_l1_gradient(device, monkeypatch, kind, L, M, N, O, K):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    batch = (L,) if L > 1 else ()
    scales = _scales(kind, K, device, g, 8.0)
    a, b, c, d = (_values(kind, (*batch, *shape), device, g) for shape in ((K, M), (N, K), (O, K), (N, M)))
    a, c = a * scales[:, None], c / scales
    call = lambda: kermac.cdist_grad(a, b, c, d, p=1.0)
    assert grad_module._route_of_any_size(grad_module._plan_cdist_grad(a, b, c, d, None, 1.0)) is not None
    got = call()
    monkeypatch.setenv("KERMAC_AMD_GRADIENT_WORKSPACE", "0")
    a3, b3, c3, d3 = (x.double().reshape(L, *x.shape[-2:]) for x in (a, b, c, d))
    want = torch.stack([c3 @ (a3 * torch.where(d3[:, n, None, :] >= b3[:, n, :, None], 1.0, -1.0)) for n in range(N)], 2)          # [L, O, N, M]
    _no_worse(got, call(), want)
