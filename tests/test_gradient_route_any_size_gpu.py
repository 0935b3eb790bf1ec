"""L1 gradients below the library's rule for the fp16 route: the route that the launch-time models choose
against float64 and against the kernels it takes the place of, in every form the calls come in."""
import importlib

import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu

grad_module = importlib.import_module("kermac_amd.cdist_grad")       # the package attribute of that name is the function
ROUTE = "norm_gradient_l1_f16"


def _operands(device, L, M, N, O, K):
    g = torch.Generator(device=device).manual_seed(M + N + O + K)
    batch = (L,) if L > 1 else ()

    def normal(*shape):
        return torch.randn(*batch, *shape, device=device, generator=g)

    return normal(K, M), normal(N, K), normal(O, K), normal(N, M)


def _errors(got, a, b, c, d, p):
    """The 2-norm of the error against float64 in units of the 2-norm of sum_k |c a g(d - b)|, and its largest multiple of that sum."""
    a, b, c, d = (x.double() for x in (a, b, c, d))
    worst, error, scale = 0.0, 0.0, 0.0
    for n in range(b.shape[-2]):
        g = d[..., n, None, :] - b[..., n, :, None]
        if p == 1.0:
            g = torch.where(g >= 0, 1.0, -1.0).double()
        want, size = c @ (a * g), c.abs() @ (a * g).abs()
        off = (got[..., :, n, :].double().reshape(want.shape) - want).abs()
        worst = max(worst, float((off / size).max()))
        error, scale = error + float(off.square().sum()), scale + float(size.square().sum())
    return (error / scale) ** 0.5, worst


# uncut and cut over k, with a rest (9 x 512 + 424) and without, odd sizes, one output and more than a tile of them, batches
@pytest.mark.parametrize("p,L,M,N,O,K", [(1.0, 1, 428, 18, 4, 256), (1.0, 1, 201, 33, 1, 471), (1.0, 2, 64, 11, 1, 1301), (1.0, 1, 1045, 24, 10, 5706),
                                         (1.0, 1, 192, 22, 33, 1088)])
def test_gradient_on_the_route_of_any_size(device, monkeypatch, p, L, M, N, O, K):
    operands = _operands(device, L, M, N, O, K)
    plan = grad_module._plan_cdist_grad(*operands, None, p)
    route = grad_module._route_of_any_size(plan)
    assert route is not None and _backend.norm_gradient_workspace_bytes(plan.params) == 0
    assert any(ROUTE in name for name in kernels_of(lambda: kermac.cdist_grad(*operands, p=p)))
    got = kermac.cdist_grad(*operands, p=p)
    # an `out` with gaps, and the last operand misaligned and padded: the planes of `out` form no matrix
    wide = torch.full((L, O, N, M + 3), -7.0, device=device)
    a, b, c, d = operands
    padded = torch.zeros(*d.shape[:-1], M + 5, device=device)
    padded[..., 1:M + 1] = d
    result = kermac.cdist_grad(a, b, c, padded[..., 1:M + 1], out=wide[..., :M], p=p)
    assert torch.equal(result, got) and torch.all(wide[..., M:] == -7.0)
    # three pieces' products per term are off by 3 * 2^-22 of it, and the sums round like those of the fp32 kernels: at most their error and that
    monkeypatch.setenv("KERMAC_AMD_GRADIENT_WORKSPACE", "0")
    fp32 = kermac.cdist_grad(*operands, p=p)
    on_route, on_fp32 = _errors(got, *operands, p), _errors(fp32, *operands, p)
    assert on_route[0] <= 1.05 * on_fp32[0] and on_route[1] <= on_fp32[1] + 3 * 2.0 ** -22


@pytest.mark.parametrize("p", [1.0, 2.0])
def test_gradient_without_memory_for_the_route_runs_as_before(device, monkeypatch, p):
    operands = _operands(device, 1, 256, 62, 4, 832)
    kermac.set_max_scratch_bytes(300000)
    try:
        got = kermac.cdist_grad(*operands, p=p)
    finally:
        kermac.set_max_scratch_bytes(None)
    monkeypatch.setenv("KERMAC_AMD_GRADIENT_WORKSPACE", "0")
    kermac.set_max_scratch_bytes(300000)
    try:
        assert torch.equal(got, kermac.cdist_grad(*operands, p=p))
    finally:
        kermac.set_max_scratch_bytes(None)
