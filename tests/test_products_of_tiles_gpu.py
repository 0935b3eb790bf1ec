"""GPU tests of the kernel matrix x coefficients contracted where the route through a workspace makes the matrix (KMC_FLAG_PRODUCT_PIECES):
in both tiles of the product kernel that contract (the fixture sends the small results to the tile of the larger ones), at the edges of tiles, column blocks and panels, with tiles that the repair launch makes again.

Tolerance: 1e-5 of every kernel value (the route's) under the sum, sum_n 1e-5 |C(m, n) coef[n, o]|, and N 2^-24 of the same sum for the fp32 additions."""
import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend
from tests.helpers import kernels_of, make_operand

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("product_tile")]

GAUSSIAN = kermac.KernelDescriptor(kermac.InnerOperator.DIFF, kermac.PowerType.SQUARE, kermac.PowerType.NOOP, kermac.KernelType.GAUSSIAN)
INSIDE = "contracted where they are made"


@pytest.fixture(autouse=True)
def route(monkeypatch):
    monkeypatch.setenv("KERMAC_AMD_WIDE_MIN_TILES", "1")
    with kermac.l2_mode("gram_bf16", min_k=0):
        yield


def check(got, matrix, coef, what):
    """matrix [L, M, N] in float64"""
    coef = coef.double()
    if coef.dim() == 2:
        coef = coef[None]
    truth, size = matrix @ coef, matrix.abs() @ coef.abs()
    bound = (1e-5 + matrix.size(-1) * 2.0 ** -24) * size + 1e-30
    error = (got.double() - truth).abs()
    assert not torch.isnan(got).any() and torch.all(error <= bound), f"{what}: {(error / bound).max().item():.3g} of the bound"


def gaussian(a, b, bandwidth):
    return torch.exp(-torch.cdist(a.double(), b.double()) ** 2 / (2 * bandwidth ** 2))


@pytest.mark.parametrize("M,N,K,O", [(1, 1, 1, 1), (127, 129, 16, 3), (128, 128, 33, 4), (129, 127, 40, 15), (300, 520, 64, 16), (257, 400, 70, 17),
                                     (513, 130, 20, 31), (64, 1000, 30, 32), (1000, 257, 100, 10), (260, 8200, 17, 5), (1000, 8700, 32, 10)])
@pytest.mark.parametrize("layout", ["rr", "cc"])
def test_shapes(device, capsys, M, N, K, O, layout):
    g = torch.Generator().manual_seed(M + N + K + O)
    a, b = (make_operand(1, rows, K, layout[0] == "c", device, g) for rows in (M, N))
    coef = torch.randn(N, O + 2, generator=g).to(device)[:, 1:O + 1]
    store = torch.full((1, M, O + 1), 7.0, device=device)
    for descriptor, matrix, kw in ((GAUSSIAN, gaussian(a, b, K ** 0.5), dict(bandwidth=K ** 0.5)),
                                   (kermac.kernel_descriptor_l2_norm, torch.cdist(a.double(), b.double()), {})):
        got = kermac.run_kernel(descriptor, a, b, out=store[..., :O], coefficients=coef, debug=True, **kw)
        assert INSIDE in capsys.readouterr().out
        check(got, matrix, coef, f"{descriptor!r}")
        assert torch.all(store[..., O] == 7.0), "wrote outside the result"
        assert torch.equal(got, kermac.run_kernel(descriptor, a, b, coefficients=coef, **kw)), "another run, another storage"


@pytest.mark.parametrize("O", [1, 10, 32, 33])
def test_sums_of_products(device, capsys, O):
    g = torch.Generator().manual_seed(O)
    a, b, coef = (torch.randn(*shape, generator=g).to(device) for shape in ((2, 300, 70), (2, 700, 70), (2, 700, O)))
    cubed = kermac.KernelDescriptor(kermac.InnerOperator.DOT, kermac.PowerType.NOOP, kermac.PowerType.SQUARE, kermac.KernelType.NONE)
    got = kermac.run_kernel(cubed, a, b, coefficients=coef, debug=True)
    assert (INSIDE in capsys.readouterr().out) == (O <= 32)
    products = a.double() @ b.double().transpose(-1, -2)
    size = (2 * (a.double().abs() @ b.double().abs().transpose(-1, -2)) * products.abs()) @ coef.double().abs()
    # the error of a.b is below 1e-6 sum |a b|, that of its square twice that times |a.b|
    assert torch.all((got.double() - products ** 2 @ coef.double()).abs() <= 1e-6 * size + 700 * 2.0 ** -24 * (products ** 2 @ coef.double().abs()))


def test_panels_and_batches_with_a_regularised_diagonal(device, monkeypatch, capsys):
    """Panels are added to the result; the split of the rows is kept for them; one bandwidth and one set of points per entry."""
    g = torch.Generator().manual_seed(5)
    L, M, N, K, O = 3, 700, 1300, 40, 10
    monkeypatch.setenv("KERMAC_AMD_COEFFICIENT_PANEL_BYTES", "4096")
    a, b, coef = (torch.randn(*shape, generator=g).to(device) for shape in ((L, M, K), (N, K), (L, N, O)))
    a, b = a + 20.0, b + 20.0
    bandwidth = torch.tensor([4.0, 6.0, 9.0], device=device)
    got = kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=bandwidth, regularization=0.5, regularization_offset_x=2, debug=True)
    assert "6 panels of 256 centres" in capsys.readouterr().out
    matrix = gaussian(a, b.expand(L, N, K), bandwidth.double().reshape(L, 1, 1))
    m, n = torch.arange(M, device=device)[:, None], torch.arange(N, device=device)[None]
    check(got, torch.where(2 + n == m, torch.full_like(matrix, 1.5), matrix), coef, "panels")


def test_tiles_that_are_made_again(device):
    """Near-duplicates far from the origin: in a few tiles, and in nearly all of them (the sample then leaves everything to the other kernel)."""
    g = torch.Generator().manual_seed(6)
    base = torch.randn(64, 48, generator=g) * 5
    for shuffled in (False, True):
        a, b = (base.repeat_interleave(n, 0) + 1e-3 * torch.randn(64 * n, 48, generator=g) for n in (10, 30))
        if shuffled:
            a, b = a[torch.randperm(640, generator=g)], b[torch.randperm(1920, generator=g)]
        a, b, coef = a.to(device), b.to(device), torch.randn(1920, 20, generator=g).to(device)
        check(kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=3.0), gaussian(a, b, 3.0)[None], coef, f"shuffled {shuffled}")
        assert "kernel_times_coefficients" in " ".join(kernels_of(lambda: kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=3.0)))
    # a set against rows of its own: the distances on the diagonal are zero
    x = torch.randn(900, 60, generator=g).to(device)
    check(kermac.run_kernel(GAUSSIAN, x, x[100:500], coefficients=coef[:400], bandwidth=7.0), gaussian(x, x[100:500], 7.0)[None], coef[:400], "own rows")


def test_values_without_a_number_stay_in_their_rows(device):
    """A row of a that is not a number spoils its own row of the result only; a function that has no value where no column is, none."""
    g = torch.Generator().manual_seed(8)
    a, b, coef = (torch.randn(*shape, generator=g).to(device) for shape in ((300, 40), (200, 40), (200, 10)))
    a[17, 3] = float("nan")
    got = kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=6.0)
    assert torch.isnan(got[0, 17]).all()
    keep = torch.arange(300, device=device) != 17
    check(got[:, keep], gaussian(a[keep], b, 6.0)[None], coef, "the other rows")
    a[17] = 0.0          # at distance zero from the zeros that pad b: 1 / d has no value there
    inverse = kermac.KernelDescriptor(kermac.InnerOperator.DIFF, kermac.PowerType.SQUARE, kermac.PowerType.POW, kermac.KernelType.NONE)
    got = kermac.run_kernel(inverse, a, b, coefficients=coef, outer_p=-0.5)
    check(got, 1.0 / torch.cdist(a.double(), b.double())[None], coef, "1 / d")


def test_without_its_workspace_the_fused_kernel_runs(device, monkeypatch):
    g = torch.Generator().manual_seed(9)
    a, b, coef = (torch.randn(*shape, generator=g).to(device) for shape in ((300, 70), (400, 70), (400, 10)))
    from kermac_amd import kernel_coefficients as module
    plan = module._plan_run_kernel_coefficients(GAUSSIAN, a, b, coef, None, None, None, None, 8.0, None, None, 0, 0)
    stream = torch.cuda.current_stream().cuda_stream
    _backend.kernel_times_coefficients(plan.params, stream)
    fused = plan.out.clone()
    plan.params.kernel.flags |= _backend.FLAG_PRODUCT_PIECES
    needed = _backend.kernel_coefficients_workspace_bytes(plan.params)
    assert needed > 0
    workspace = torch.empty(needed, dtype=torch.uint8, device=device)
    for pointer, size in ((0, 0), (workspace.data_ptr(), needed - 1), (workspace.data_ptr() + 16, needed)):
        plan.out.fill_(-1.0)
        plan.params.kernel.gram_workspace, plan.params.kernel.gram_workspace_bytes = pointer, size
        _backend.kernel_times_coefficients(plan.params, stream)
        assert torch.equal(plan.out, fused)
        plan.params.kernel.flags |= _backend.FLAG_PRODUCT_ACCUMULATE
        with pytest.raises(_backend.BackendError, match="ACCUMULATE"):
            _backend.kernel_times_coefficients(plan.params, stream)
        plan.params.kernel.flags &= ~_backend.FLAG_PRODUCT_ACCUMULATE
    plan.params.kernel.gram_workspace, plan.params.kernel.gram_workspace_bytes = workspace.data_ptr(), needed
    _backend.kernel_times_coefficients(plan.params, stream)
    check(plan.out, gaussian(a, b, 8.0)[None], coef, "with the workspace")
    wide = torch.randn(400, 33, generator=g).to(device)
    plan = module._plan_run_kernel_coefficients(GAUSSIAN, a, b, wide, None, None, None, None, 8.0, None, None, 0, 0)
    plan.params.kernel.flags |= _backend.FLAG_PRODUCT_PIECES
    assert _backend.kernel_coefficients_workspace_bytes(plan.params) == 0          # 33 columns


def test_graph_replays(device):
    g = torch.Generator().manual_seed(10)
    a, b, coef = (torch.randn(*shape, generator=g).to(device) for shape in ((300, 70), (700, 70), (700, 10)))
    out = torch.empty(1, 300, 10, device=device)
    scratch = torch.empty(1 << 24, dtype=torch.uint8, device=device)

    def call():
        with kermac.scratch(scratch):
            kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=8.0, out=out)
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(4):
        a.copy_(torch.randn(300, 70, generator=g))
        out.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        out.fill_(-1.0)
        call()
        torch.cuda.synchronize()
        assert torch.equal(out, replayed)
