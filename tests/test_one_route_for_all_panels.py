"""A product in several panels takes its route for all of them: the library's rule for the route through a workspace, which looks at the size of a
matrix, would refuse a last panel much shorter than the others.  No switch of the environment sets that rule aside here.

Tolerance on the GPU: 1e-5 of every kernel value (the route's) under the sum, sum_n 1e-5 |C(m, n) coef[n, o]|, and N 2^-24 of the same sum for the fp32
additions."""
import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend, _scratch
from kermac_amd import kernel_coefficients as module

GAUSSIAN = kermac.KernelDescriptor(kermac.InnerOperator.DIFF, kermac.PowerType.SQUARE, kermac.PowerType.NOOP, kermac.KernelType.GAUSSIAN)
LINEAR = kermac.KernelDescriptor(kermac.InnerOperator.DOT, kermac.PowerType.NOOP, kermac.PowerType.NOOP, kermac.KernelType.NONE)


@pytest.fixture(autouse=True)
def the_rule_alone(monkeypatch):
    for name in ("KERMAC_AMD_WIDE_MIN_TILES", "KERMAC_AMD_COEFFICIENT_PANEL_BYTES", "KERMAC_AMD_PRODUCTS_OF_TILES", "KERMAC_AMD_L2_WORKSPACE"):
        monkeypatch.delenv(name, raising=False)


class Somewhere:
    """Stands in for device memory of any size: only its address is looked at."""

    def data_ptr(self):
        return 1 << 40


@pytest.mark.parametrize("descriptor,L,M,N,K,O,k_contiguous", [
    (GAUSSIAN, 1, 100000, 100000, 256, 10, False), (GAUSSIAN, 1, 121491, 129213, 241, 10, False), (GAUSSIAN, 4, 25470, 31302, 411, 10, False),
    (GAUSSIAN, 4, 63328, 1189, 318, 32, False), (GAUSSIAN, 4, 12973, 133678, 167, 10, True), (LINEAR, 1, 188653, 29567, 196, 10, False),
    (LINEAR, 4, 47035, 3099, 133, 10, True), (GAUSSIAN, 1, 100000, 100000, 256, 40, False), (LINEAR, 4, 47035, 3099, 133, 40, True)])
def test_every_panel_gets_the_workspace_of_the_first(monkeypatch, descriptor, L, M, N, K, O, k_contiguous):
    def points(rows):
        return torch.empty(L, rows, K) if k_contiguous else torch.empty(L, K, rows).transpose(1, 2)

    bandwidth = 2.0 if descriptor is GAUSSIAN else None
    plan = module._plan_run_kernel_coefficients(descriptor, points(M), points(N), torch.empty(L, N, O), torch.empty(L, M, O), None, None, None,
                                                bandwidth, None, None, 0, 0, require_device=False)
    shape = module._panel_shape(plan, _backend.FLAG_L2_GRAM_BF16 if descriptor is GAUSSIAN else _backend.FLAG_DOT_PIECES)
    assert shape is not None and shape[1] > 1, "the case is of several panels"
    launched = []

    def product(params, stream):
        launched.append((params.kernel.n, _backend.kernel_coefficients_workspace_bytes(params), params.kernel.gram_workspace_bytes))

    def matrix(params, stream):
        launched.append((params.n, _backend.gram_workspace_bytes(params), params.gram_workspace_bytes))

    monkeypatch.setattr(_backend, "kernel_times_coefficients", product)
    monkeypatch.setattr(_backend, "build_kernel", matrix)
    monkeypatch.setattr(_backend, "matrix_times_coefficients", lambda params, stream: None)
    monkeypatch.setattr(module, "_sum_partials", lambda buffers, out: None)
    monkeypatch.setattr(_scratch, "allocate", lambda nbytes, device: Somewhere())
    monkeypatch.setattr(_scratch, "allocate_floats", lambda shape, device: Somewhere())
    monkeypatch.setattr(module, "_partial_products", lambda parts, plan, device: (Somewhere(), None))
    assert module._run_in_panels(plan, shape, 0, torch.device("cpu"), False)
    assert sum(n for n, _, _ in launched) == N and len(launched) == shape[1]
    for n, wanted, given in launched:
        assert 0 < wanted <= given, f"a panel of {n} centres: the library wants {wanted} bytes for its route, {given} are there"


@pytest.mark.parametrize("limit,runs", [(None, 2), (300 << 20, 7), (100 << 20, 27), (10 << 20, None)])
def test_the_memory_of_a_run_of_centres_is_bounded(monkeypatch, limit, runs):
    """Few rows against many centres: the pieces of the centres, 512 bytes each here, are most of what a run takes."""
    L, M, N, K, O = 1, 200, 3000000, 100, 10
    plan = module._plan_run_kernel_coefficients(GAUSSIAN, torch.empty(M, K), torch.empty(N, K), torch.empty(N, O), torch.empty(L, M, O), None, None, None, 10.0, None, None, 0, 0,
                                                require_device=False)
    assert module._auto_products_of_tiles(plan) and module._panel_shape(plan, _backend.FLAG_L2_GRAM_BF16) is None
    taken, launched = [], []

    def allocate(nbytes, device):
        if limit is not None and nbytes > limit:
            return None
        taken.append(nbytes)
        return Somewhere()

    monkeypatch.setattr(_scratch, "allocate", allocate)
    monkeypatch.setattr(_backend, "kernel_times_coefficients", lambda params, stream: launched.append((params.kernel.n, params.kernel.b - plan.params.kernel.b)))
    assert module._products_of_tiles_at_any_size(plan, 0, torch.device("cpu"), False) == (runs is not None)
    assert len(launched) == (runs or 0)
    if runs is not None:
        assert len(taken) == 1 and taken[0] <= 1 << 30
        assert sum(n for n, _ in launched) == N and [b for _, b in launched] == [4 * K * launched[0][0] * i for i in range(runs)]


@pytest.mark.gpu
@pytest.mark.parametrize("limit,runs", [(None, 1), (12 << 20, 4), (1 << 20, 0)])
def test_fewer_centres_at_once_where_the_memory_is_refused(device, monkeypatch, capsys, limit, runs):
    M, N, K, O = 200, 60000, 100, 10
    monkeypatch.setenv("KERMAC_AMD_COEFFICIENT_PANEL_BYTES", str(40 << 20))
    g = torch.Generator().manual_seed(3)
    a, b, coef = (torch.randn(*shape, generator=g).to(device) for shape in ((M, K), (N, K), (N, O)))
    kermac.set_max_scratch_bytes(limit)
    try:
        got = kermac.run_kernel(GAUSSIAN, a, b, coefficients=coef, bandwidth=10.0, debug=True)
    finally:
        kermac.set_max_scratch_bytes(None)
    said = capsys.readouterr().out
    rows = -(-N // max(runs, 1) // 256) * 256 if runs != 1 else N
    assert (f"tile by tile, {rows} centres at once" in said) == (runs > 0), said
    matrix = torch.exp(-torch.cdist(a.double(), b.double()) ** 2 / 200)
    error, size = (got.double()[0] - matrix @ coef.double()).abs(), (1e-5 + N * 2.0 ** -24) * matrix @ coef.double().abs()
    assert torch.all(error <= size), f"{(error / size).max().item():.3g} of the bound"


@pytest.mark.gpu
@pytest.mark.parametrize("O", [10, 40])
@pytest.mark.parametrize("descriptor,M", [(GAUSSIAN, 3072), (LINEAR, 4096)])
def test_a_short_last_panel(device, monkeypatch, descriptor, M, O):
    """Panels of 1024 centres, the last of 100, on points far from the origin, which only a centre keeps from the repair launch."""
    K, N = 784, 3 * 1024 + 100
    monkeypatch.setenv("KERMAC_AMD_COEFFICIENT_PANEL_BYTES", str(4 * M * 1024))
    g = torch.Generator().manual_seed(O)
    offset = 30.0 if descriptor is GAUSSIAN else 0.0
    a, b, coef = ((torch.randn(*shape, generator=g) + shift).to(device) for shape, shift in (((M, K), offset), ((N, K), offset), ((N, O), 0.0)))
    kw = dict(bandwidth=K ** 0.5) if descriptor is GAUSSIAN else {}
    plan = module._plan_run_kernel_coefficients(descriptor, a, b, coef, None, None, None, None, kw.get("bandwidth"), None, None, 0, 0)
    route = _backend.FLAG_L2_GRAM_BF16 if descriptor is GAUSSIAN else _backend.FLAG_DOT_PIECES
    shape = module._panel_shape(plan, route)
    assert shape[:2] == (1024, 4) and shape[4] == route, "the library's rule takes the first panel"
    block = _backend.BuildKernelParams.from_buffer_copy(plan.params.kernel)
    block.flags, block.n, block.c_ld = block.flags | route, 100, M
    assert _backend.gram_workspace_bytes(block) == 0, "and not the last one"
    got = kermac.run_kernel(descriptor, a, b, coefficients=coef, **kw)
    a, b, coef = a.double(), b.double(), coef.double()
    if descriptor is GAUSSIAN:
        matrix = torch.exp(-torch.cdist(a, b) ** 2 / (2 * K))
        size = (1e-5 + N * 2.0 ** -24) * matrix @ coef.abs()
    else:
        matrix = a @ b.T
        size = 1e-5 * (a.abs() @ b.abs().T) @ coef.abs() + N * 2.0 ** -24 * matrix.abs() @ coef.abs()
    error = (got.double()[0] - matrix @ coef).abs()
    assert torch.all(error <= size), f"{(error / size).max().item():.3g} of the bound"
