"""The direct kernel in tiles of 64 x 64 (results of few tiles): its bits are those of the 128 x 128 tile, over every storage, remainder and
epilogue.  The larger tile is reached with the same points inside a batch that has too many tiles for the small one."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu

COPIES = 257        # batch entries of at least one tile of 128 x 128 each: more than the small tile takes


def _stored(x, form):
    if form == "panel":
        return x.transpose(-1, -2).contiguous().transpose(-1, -2)
    if form == "misaligned":
        return torch.nn.functional.pad(x, (1, 0))[..., 1:]
    if form == "misaligned_panel":
        return torch.nn.functional.pad(x.transpose(-1, -2), (1, 0))[..., 1:].transpose(-1, -2)
    return x


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (63, 65, 15), (64, 64, 32), (65, 127, 33), (130, 61, 16), (129, 200, 47), (200, 70, 100)])
@pytest.mark.parametrize("form_a,form_b", [("rows", "rows"), ("panel", "panel"), ("misaligned", "panel"), ("misaligned_panel", "misaligned"),
                                           ("rows", "misaligned_panel")])
@pytest.mark.parametrize("p", [1.0, 2.0, 1.3, 3.0])
def test_the_bits_of_the_large_tile(device, M, N, K, form_a, form_b, p):
    gen = torch.Generator(device=device).manual_seed(M + N + K)
    a, b = (torch.randn(rows, K, device=device, generator=gen) for rows in (M, N))
    a_many, b_many = (_stored(x.expand(COPIES, *x.shape).contiguous(), f) for x, f in ((a, form_a), (b, form_b)))
    a, b = _stored(a, form_a), _stored(b, form_b)
    with kermac.l2_mode("direct"):
        small, large = kermac.cdist(a, b, p=p), kermac.cdist(a_many, b_many, p=p)
        assert torch.equal(small.reshape(M, N), large[COPIES - 1])
        laplace = [kermac.run_kernel(kermac.kernel_descriptor_laplace_l2, x, y, bandwidth=3.0, regularization=0.5)
                   for x, y in ((a, b), (a_many, b_many))]
        assert torch.equal(laplace[0].reshape(M, N), laplace[1][COPIES - 1])
    truth = torch.cdist(a.double().cpu(), b.double().cpu(), p=p)
    # fp32 sums of K terms, each term and root a few units in the last place
    assert ((small.reshape(M, N).double().cpu() - truth).abs() <= (1e-4 if p == 1.3 else 1e-5) * truth).all()


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (63, 65, 15), (65, 127, 33), (130, 61, 16), (129, 200, 47)])
@pytest.mark.parametrize("form_a,form_b", [("rows", "rows"), ("panel", "panel"), ("misaligned", "panel"), ("misaligned_panel", "misaligned")])
@pytest.mark.parametrize("operator", ["signed differences", "products"])
def test_the_bits_of_the_large_tile_where_no_power_is_taken(device, M, N, K, form_a, form_b, operator):
    gen = torch.Generator(device=device).manual_seed(M + N + K)
    a, b = (torch.randn(rows, K, device=device, generator=gen) for rows in (M, N))
    a_many, b_many = (_stored(x.expand(COPIES, *x.shape).contiguous(), f) for x, f in ((a, form_a), (b, form_b)))
    inner = kermac.InnerOperator.DIFF if operator == "signed differences" else kermac.InnerOperator.DOT
    descriptor = kermac.KernelDescriptor(inner, kermac.PowerType.NOOP, kermac.PowerType.NOOP, kermac.KernelType.NONE)
    results = []
    with kermac.l2_mode("direct"):
        for x, y, kernel in ((_stored(a, form_a), _stored(b, form_b), True), (a_many, b_many, False)):
            kept = []
            ran = [name for name in kernels_of(lambda: kept.append(kermac.run_kernel(descriptor, x, y))) if "build_kernel" in name]
            assert len(ran) == 1 and ("build_kernel_small<" in ran[0]) == kernel
            results.append(kept[0])
    assert torch.equal(results[0].reshape(M, N), results[1][COPIES - 1])
    x, y = a.double(), b.double()
    if operator == "products":
        truth, scale = x @ y.t().contiguous(), x.abs() @ y.abs().t().contiguous()
    else:
        truth, scale = (x[:, None] - y[None]).sum(-1), (x[:, None] - y[None]).abs().sum(-1)
    assert ((results[0].reshape(M, N).double() - truth).abs() <= 1e-5 * scale).all()         # fp32 sums of K terms


@pytest.mark.parametrize("M,K", [(65, 20), (300, 6), (129, 64)])
def test_a_set_against_itself(device, M, K):
    gen = torch.Generator(device=device).manual_seed(M)
    a = torch.randn(M, K, device=device, generator=gen)
    a[M // 2, 0] = float("nan")
    got = kermac.cdist(a, a, p=1.0)[0]
    other = kermac.cdist(a, a.clone(), p=1.0)[0]
    same = (got == other) | (torch.isnan(got) & torch.isnan(other))
    assert same.all() and ((got == got.t()) | torch.isnan(got)).all()


@pytest.mark.parametrize("p,most", [(1.0, 256), (3.0, 256), (1.3, 192), (0.5, 192), (1.5, 192)])
def test_up_to_how_many_tiles(device, p, most):
    """Fractional powers lose on a fourth workgroup per CU, the others do not."""
    x = torch.randn(most + 1, 40, 5, device=device, generator=torch.Generator(device=device).manual_seed(1))
    ran = [[name for name in kernels_of(lambda: kermac.cdist(x[:tiles], x[:tiles] + 1.0, p=p)) if "build_kernel" in name] for tiles in (most, most + 1)]
    assert ["build_kernel_small<" in name for names in ran for name in names] == [True, False]
