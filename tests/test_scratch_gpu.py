"""What the operators allocate beside `out`, and the two controls over it (kermac_amd/_scratch.py): with the limit
at 0 a call allocates nothing -- the reference's contract (README.md:69,135: "aside from `out` ... does not allocate")
-- and inside `kermac.scratch(buffer)` it takes its buffers from the caller's memory and allocates nothing either.
Allocations are counted by torch's allocator statistics around the call.
"""
import contextlib
import importlib

import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend
from tests.helpers import assert_close_to_truth, kernels_of, l1_distances_float64

grad_module = importlib.import_module("kermac_amd.cdist_grad")      # the package attribute of that name is the operator

pytestmark = pytest.mark.gpu


def allocations(device):
    return torch.cuda.memory_stats(device)["allocation.all.allocated"]


def counted(device, fn):
    torch.cuda.synchronize(device)
    before = allocations(device)
    result = fn()
    torch.cuda.synchronize(device)
    return result, allocations(device) - before


@pytest.fixture
def cases(device):
    """Three default-mode calls that take a workspace route when they are given the memory: squared distances,
    the L1 gradient, a Gaussian kernel matrix times coefficients (panels)."""
    g = torch.Generator().manual_seed(31)
    a = torch.randn(512, 4096, generator=g).to(device).t()
    b = torch.randn(512, 4096, generator=g).to(device).t()
    out = torch.empty(4096, 4096, device=device).t()
    kernel = torch.rand(2048, 2048, generator=g).to(device)
    x = (torch.randn(512, 2048, generator=g) / 512 ** 0.5).to(device)
    coefs = torch.randn(16, 2048, generator=g).to(device)
    z = (torch.randn(512, 2048, generator=g) / 512 ** 0.5).to(device)
    grad = torch.empty(1, 16, 512, 2048, device=device)
    coefficients = torch.randn(4096, 32, generator=g).to(device)
    product = torch.empty(4096, 32, device=device)
    gaussian = kermac.KernelDescriptor(kermac.InnerOperator.DIFF, kermac.PowerType.SQUARE, kermac.PowerType.NOOP,
                                       kermac.KernelType.GAUSSIAN)
    calls = {
        "cdist p=2": lambda: kermac.cdist(a, b, out=out, p=2.0),
        "cdist_grad p=1": lambda: kermac.cdist_grad(kernel, x, coefs, z, out=grad, p=1.0),
        "gaussian x coefficients": lambda: kermac.run_kernel(gaussian, a, b, out=product, bandwidth=30.0, coefficients=coefficients),
    }
    for call in calls.values():
        call()                      # kernels loaded, allocator warm
    return calls


def test_default_calls_do_allocate(device, cases):
    for name, call in cases.items():
        _, count = counted(device, call)
        assert count > 0, f"{name}: the default route was expected to take a workspace"


def test_limit_zero_allocates_nothing(device, cases):
    reference = {name: call().clone() for name, call in cases.items()}
    kermac.set_max_scratch_bytes(0)
    try:
        assert kermac.get_max_scratch_bytes() == 0
        for name, call in cases.items():
            result, count = counted(device, call)
            assert count == 0, f"{name}: {count} allocations with the limit at 0"
            # another route (no workspace), the same tolerance: close to the default route's result
            scale = reference[name].abs().mean().item()
            assert (result - reference[name]).abs().max().item() <= 2e-5 * max(scale, 1e-30) * (50 if "grad" in name or "coeff" in name else 1), name
    finally:
        kermac.set_max_scratch_bytes(None)
    assert kermac.get_max_scratch_bytes() is None


def test_supplied_buffer_allocates_nothing_and_takes_the_same_routes(device, cases):
    reference = {name: call().clone() for name, call in cases.items()}
    buffer = torch.empty(3 << 30, dtype=torch.uint8, device=device)
    with kermac.scratch(buffer):
        for name, call in cases.items():
            result, count = counted(device, call)
            assert count == 0, f"{name}: {count} allocations inside scratch(buffer)"
            assert torch.equal(result, reference[name]), f"{name}: the route with the caller's buffer gives other bits"
    # a buffer that is too small for anything: the calls do without, still without allocating
    tiny = torch.empty(1024, dtype=torch.uint8, device=device)
    with kermac.scratch(tiny):
        for name, call in cases.items():
            _, count = counted(device, call)
            assert count == 0, name
    with pytest.raises(TypeError):
        with kermac.scratch(torch.empty(16, device=device)):
            pass


def test_fixed_point_route_and_cut_launches_respect_the_limit(device):
    g = torch.Generator().manual_seed(32)
    a = torch.randn(2048, 700, generator=g).to(device)          # 6 x 6 tiles over k = 2048: cut over k by default
    b = torch.randn(2048, 650, generator=g).to(device)
    a, b = a.t(), b.t()
    out = torch.empty(650, 700, device=device).t()
    kermac.cdist(a, b, out=out, p=1.0)
    _, count = counted(device, lambda: kermac.cdist(a, b, out=out, p=1.0))
    assert count > 0
    kermac.set_max_scratch_bytes(0)
    try:
        _, count = counted(device, lambda: kermac.cdist(a, b, out=out, p=1.0))
        assert count == 0
        assert_close_to_truth(out, l1_distances_float64(a, b), rtol=1e-5, what="uncut launch")
        with kermac.l1_mode("fixed"):
            _, count = counted(device, lambda: kermac.cdist(a, b, out=out, p=1.0))
            assert count == 0
    finally:
        kermac.set_max_scratch_bytes(None)


def _gradient(device, M, N, O, K):
    g = torch.Generator(device=device).manual_seed(M + N)
    a, b, c, d = (torch.randn(rows, columns, device=device, generator=g) for rows, columns in ((K, M), (N, K), (O, K), (N, M)))
    return lambda: kermac.cdist_grad(a, b, c, d, p=1.0), grad_module._plan_cdist_grad(a, b, c, d, None, 1.0)


def _bytes_of(plan, cut):
    """Partial results and workspace of a call that is cut over k, each at a multiple of 256 bytes as in a supplied buffer."""
    slices, depth, leftover, needs_workspace = cut
    partial = -(-4 * (slices + (leftover > 0)) * plan.O * plan.N * plan.M // 256) * 256
    params = type(plan.params).from_buffer_copy(plan.params)
    params.k, params.l, params.d_bs = depth, slices, 0
    params.a_bs, params.b_bs, params.c_bs = depth * params.a_ld, depth, depth
    return partial + (_backend.norm_gradient_workspace_bytes(params) if needs_workspace else 0)


@contextlib.contextmanager
def _at_most(nbytes, how, device):
    if how == "buffer":
        with kermac.scratch(torch.empty(nbytes, dtype=torch.uint8, device=device)):
            yield
    else:
        kermac.set_max_scratch_bytes(nbytes)
        try:
            yield
        finally:
            kermac.set_max_scratch_bytes(None)


# f16 slices wanted: several, fewer than the fp32 kernels, none
@pytest.mark.parametrize("M,N,O,K", [(2000, 24, 16, 9000), (4000, 100, 16, 10000), (8192, 128, 16, 8192)])
@pytest.mark.parametrize("how", ["limit", "buffer"])
def test_l1_gradient_without_its_workspace_is_cut_for_the_kernels_that_run(device, monkeypatch, how, M, N, O, K):
    """A limit that holds the partial results of the fp32 kernels' slices, but not the workspace of the fp16 route: the bits of a
    process without that route."""
    call, plan = _gradient(device, M, N, O, K)
    *on_f16, on_fp32 = grad_module._cuts_over_contraction(plan)
    assert on_f16 and all(cut[3] for cut in on_f16) and not on_fp32[3]
    enough = _bytes_of(plan, on_fp32)
    assert all(_bytes_of(plan, cut) > enough + 4096 for cut in on_f16 if cut[0] > 1)
    with _at_most(enough + 4096, how, device):
        if on_f16[0][0] == 1:
            assert _backend.norm_gradient_workspace_bytes(plan.params) > enough + 4096
        got = call()
    monkeypatch.setenv("KERMAC_AMD_GRADIENT_WORKSPACE", "0")
    assert torch.equal(got, call())


@pytest.mark.parametrize("how", ["limit", "buffer"])
def test_l1_gradient_takes_fewer_slices_where_more_do_not_fit(device, how):
    call, plan = _gradient(device, 1408, 128, 32, 9522)
    more, fewer, _ = grad_module._cuts_over_contraction(plan)
    assert more[0] > fewer[0] > 1 and _bytes_of(plan, more) > _bytes_of(plan, fewer) + 4096
    with _at_most(_bytes_of(plan, fewer) + 4096, how, device):
        assert any("norm_gradient_l1_f16" in name for name in kernels_of(call))


@pytest.mark.parametrize("how", ["limit", "buffer"])
def test_l2_gradient_asks_for_its_pieces_and_no_more(device, how):
    """Two fp16 pieces per value of a and of the products c (b - s), 4 bytes, are what the route cannot do without: a tenth more holds it."""
    M, N, O, K = 4096, 512, 16, 2048
    a, b, c, d = (torch.randn(rows, columns, device=device) for rows, columns in ((K, M), (N, K), (O, K), (N, M)))
    with _at_most(int(1.1 * 4 * (M + O * N) * K), how, device):
        assert any("gram_f16_wide" in name for name in kernels_of(lambda: kermac.cdist_grad(a, b, c, d, p=2.0)))
