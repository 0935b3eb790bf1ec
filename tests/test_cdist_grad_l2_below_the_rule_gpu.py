"""L2 gradients below the library's rule for the route through fp16 pieces: they stay on the fp32 kernels, whose error is bounded by the sum of the terms'
magnitudes alone.  Pieces are scaled by the largest magnitude of a row of a or of c (b - s); what lies far below it is held to fewer bits, which is too few where
the other factor is large just there.

Tolerance: a term c a (d - b) rounds three times by 2^-24 of itself, a sum of K of them by at most K 2^-24 of their magnitudes."""
import importlib

import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu

grad_module = importlib.import_module("kermac_amd.cdist_grad")       # the package attribute of that name is the function


def _worst(got, a, b, c, d):
    """The largest error against float64 in units of sum_k |c a (d - b)|."""
    a, b, c, d = (x.double() for x in (a, b, c, d))
    worst = 0.0
    for n in range(b.shape[-2]):
        terms = a * (d[..., n, None, :] - b[..., n, :, None])
        want, size = c @ terms, c.abs() @ terms.abs()
        worst = max(worst, float(((got[..., :, n, :].double().reshape(want.shape) - want).abs() / size).max()))
    return worst


# one problem, cut over k or not, and batches, which are not cut
@pytest.mark.parametrize("L,M,N,O,K", [(1, 256, 62, 4, 832), (2, 576, 22, 2, 2048), (1, 2513, 17, 10, 5032), (1, 1479, 23, 32, 633), (2, 65, 37, 1, 3001),
                                       (2, 717, 52, 16, 390)])
@pytest.mark.parametrize("decades", [0, 6, 8, 10])
def test_rows_of_opposite_scales(device, L, M, N, O, K, decades):
    g = torch.Generator(device=device).manual_seed(M + N + O + K)
    batch = (L,) if L > 1 else ()

    def normal(*shape):
        return torch.randn(*batch, *shape, device=device, generator=g)

    scales = 10.0 ** (decades * (torch.rand(K, device=device, generator=g) - 0.5))
    a, b, c, d = normal(K, M) * scales[:, None], normal(N, K), normal(O, K) / scales, normal(N, M)
    call = lambda: kermac.cdist_grad(a, b, c, d, p=2.0)
    assert _worst(call(), a, b, c, d) <= (K + 3) * 2.0 ** -24
    assert not any("gram_f16_wide" in name for name in kernels_of(call))


@pytest.mark.parametrize("L,M,N,O,K", [(1, 256, 62, 4, 832), (2, 65, 37, 1, 3001)])
def test_a_caller_of_the_library_may_ask_for_the_route(device, L, M, N, O, K):
    """KMC_FLAG_GRAM_WORKSPACE_ANY_SIZE in the flags of the C entry: the route at its own bound, 3 * 2^-22 sum_k |c a (b - s)| and the rounding of its sums."""
    g = torch.Generator(device=device).manual_seed(K)
    batch = (L,) if L > 1 else ()
    a, b, c, d = (torch.randn(*batch, *shape, device=device, generator=g) for shape in ((K, M), (N, K), (O, K), (N, M)))
    plan = grad_module._plan_cdist_grad(a, b, c, d, None, 2.0)
    assert _backend.norm_gradient_workspace_bytes(plan.params) == 0
    assert grad_module._launch(plan, a.device, False, True, any_size=True)
    assert _worst(plan.out, a, b, c, d) <= 2e-6 + K * 2.0 ** -24
