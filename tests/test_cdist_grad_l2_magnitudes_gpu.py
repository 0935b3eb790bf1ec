"""GPU tests of the scales of a on the L2 gradient's route through a workspace: the largest magnitude of every column of a comes from the
kernel that makes g, in ranges of k and teams of waves.  Every column has one value far above its others, at another k each: a range, a team, a
tail or a lane that is left out would overflow fp16.  A column of that kind has its error bounded by its largest products:
2^-21 sum_k |c a (b - s)| from the pieces (3 * 2^-22), sums of K <= 1537 products in fp32 and the same for (d - s) g: 4e-6 of the sum of both."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def l2_route(monkeypatch):
    monkeypatch.setenv("KERMAC_AMD_GRADIENT_L2_MIN_TERMS", "1")


def check(a, b, c, d):
    got = kermac.cdist_grad(a, b, c, d, p=2.0).double()
    a, b, c, d = (t.double() if t.dim() == 3 else t.double()[None] for t in (a, b, c, d))
    s = b.mean(-1, keepdim=True)

    def both(a, b, c, d, sign):
        # sum_k c a (d - b), the two terms apart
        g = c @ a                                                              # [L, O, M]
        p = (c[:, :, None, :] * b[:, None, :, :]).flatten(1, 2) @ a           # [L, O N, M]
        return g[:, :, None, :] * d[:, None, :, :] + sign * p.reshape(got.shape[0], c.size(1), b.size(1), -1)

    L = got.size(0)
    a, b, c, d, s = (t.expand(L, -1, -1).contiguous() for t in (a, b, c, d, s))
    truth = both(a, b - s, c, d - s, -1.0)
    size = both(a.abs(), (b - s).abs(), c.abs(), (d - s).abs(), 1.0)
    assert torch.all((got - truth).abs() <= 4e-6 * size + 1e-30)


@pytest.mark.parametrize("M,K", [(1, 1), (4, 7), (5, 8), (127, 9), (128, 64), (129, 65), (256, 1023), (257, 1024), (300, 1025), (260, 1537), (513, 513)])
@pytest.mark.parametrize("N,O", [(3, 1), (40, 16), (9, 33)])
@pytest.mark.parametrize("padding", [0, 1, 4])
def test_one_large_value_per_column(device, M, N, O, K, padding):
    g = torch.Generator().manual_seed(M + N + O + K + padding)
    ld = -(-M // 4) * 4 + padding          # 1: rows of a that cannot be read 16 bytes at a time, which take the other way
    a = torch.rand(K, ld, generator=g).to(device)[:, :M]
    at = (torch.arange(M) * 7 + 3) % K
    a[at.to(device), torch.arange(M, device=device)] = 3e5
    b, c, d = (torch.randn(*shape, generator=g).to(device) for shape in ((N, K), (O, K), (N, M)))
    names = kernels_of(lambda: kermac.cdist_grad(a, b, c, d, p=2.0))
    assert any(f"matrix_times_coefficients_rows4" in name and "true" in name for name in names) == (padding != 1)
    check(a, b, c, d)


@pytest.mark.parametrize("shared", [False, True])
def test_batches(device, shared):
    g = torch.Generator().manual_seed(3)
    a = torch.rand(1 if shared else 3, 300, 200, generator=g).to(device)
    a[:, (torch.arange(200) * 11) % 300, torch.arange(200)] = 1e5
    a = a * (1.0 if shared else torch.tensor([1.0, 1e-3, 1e4]).reshape(3, 1, 1).to(device))
    b, c, d = (torch.randn(3, *shape, generator=g).to(device) for shape in ((20, 300), (10, 300), (20, 200)))
    check(a, b, c, d)


def test_columns_that_are_not_numbers(device):
    g = torch.Generator().manual_seed(4)
    a, b, c, d = (torch.rand(*shape, generator=g).to(device) for shape in ((300, 200), (20, 300), (10, 300), (20, 200)))
    a[299, 3], a[0, 77], a[150, 199] = float("nan"), float("inf"), float("-inf")
    got = kermac.cdist_grad(a, b, c, d, p=2.0)
    good = torch.ones(200, dtype=torch.bool, device=device)
    good[[3, 77, 199]] = False
    assert not torch.isfinite(got[..., ~good]).any()
    a = torch.where(torch.isfinite(a), a, torch.zeros_like(a))
    assert torch.equal(got[..., good], kermac.cdist_grad(a, b, c, d, p=2.0)[..., good])
