"""GPU tests of the direct kernel for contractions of few terms (csrc/kernels/build_kernel_short.hpp): the bits of the ordinary
direct kernel over operand storages, alignments of the result, ragged sizes, batches and kernel functions.
KERMAC_AMD_DIRECT_SHORT_MAX_K chooses between the two."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu

DIFF, DOT = kermac.InnerOperator.DIFF, kermac.InnerOperator.DOT
POW = kermac.PowerType


def descriptor(inner, power, outer=POW.NOOP, kind=kermac.KernelType.NONE):
    return kermac.KernelDescriptor(inner, power, outer, kind)


DESCRIPTORS = {
    "l1": descriptor(DIFF, POW.ABS),
    "l2": descriptor(DIFF, POW.SQUARE, POW.SQRT),
    "signed": descriptor(DIFF, POW.NOOP),
    "dot": descriptor(DOT, POW.NOOP, POW.SQUARE),
    "laplace": descriptor(DIFF, POW.ABS, POW.NOOP, kermac.KernelType.LAPLACE),
    "gaussian": descriptor(DIFF, POW.SQUARE, POW.NOOP, kermac.KernelType.GAUSSIAN),
    "cubes": descriptor(DIFF, POW.POW),
    "fourth powers": descriptor(DIFF, POW.POW, POW.SQRT),
}


def launches_short(call):
    return any("build_kernel_short" in name for name in kernels_of(call))


def both(monkeypatch, call):
    monkeypatch.setenv("KERMAC_AMD_DIRECT_SHORT_MAX_K", "24")
    assert launches_short(call)
    short = call()
    monkeypatch.setenv("KERMAC_AMD_DIRECT_SHORT_MAX_K", "0")
    assert not launches_short(call)
    return short, call()


@pytest.mark.parametrize("K", [1, 4, 5, 8, 9, 13, 16, 20, 21, 24])
@pytest.mark.parametrize("kind", sorted(DESCRIPTORS))
def test_the_bits_of_the_ordinary_kernel(device, monkeypatch, K, kind):
    g = torch.Generator().manual_seed(K)
    M, N = 531, 277
    options = dict(bandwidth=1.7, regularization=0.25, regularization_offset_x=3, regularization_offset_y=1) if kind in ("laplace", "gaussian") else {}
    if kind in ("cubes", "fourth powers"):
        options["inner_p"] = 3.0 if kind == "cubes" else 4.0
    a, b = torch.randn(M, K, generator=g).to(device), torch.randn(N, K, generator=g).to(device)
    for a_used in (a, a.t().contiguous().t()):
        for b_used in (b, b.t().contiguous().t()):
            short, ordinary = both(monkeypatch, lambda: kermac.run_kernel(DESCRIPTORS[kind], a_used, b_used, **options))
            assert torch.equal(short, ordinary)


@pytest.mark.parametrize("ld", [256, 288, 300, 310, 257, 528])
@pytest.mark.parametrize("offset", [0, 1, 2, 4, 31])
def test_every_place_in_a_line(device, monkeypatch, ld, offset):
    """Results whose columns start anywhere in a line of 128 bytes, batch entries included; nothing beside them is written."""
    g = torch.Generator().manual_seed(ld + offset)
    L, M, N, K = 2, 251, 300, 6
    a, b = torch.randn(L, K, M, generator=g).to(device).transpose(1, 2), torch.randn(L, K, N, generator=g).to(device).transpose(1, 2)

    def call():
        store = torch.full((L * N * ld + 64 + 7 * L,), -5.0, device=device)
        out = store[offset:].as_strided((L, M, N), (N * ld + 7, 1, ld))
        kermac.cdist(a, b, out=out, p=1.0)
        return store
    short, ordinary = both(monkeypatch, call)
    assert torch.equal(short, ordinary)


@pytest.mark.parametrize("M,N", [(1, 1), (1, 1000), (1000, 1), (255, 15), (256, 16), (257, 17), (225, 129), (512, 40), (4000, 2100)])
def test_edges(device, monkeypatch, M, N):
    g = torch.Generator().manual_seed(M + N)
    a, b = torch.randn(M, 11, generator=g).to(device), torch.randn(N, 11, generator=g).to(device)
    short, ordinary = both(monkeypatch, lambda: kermac.cdist(a, b, p=2.0))
    assert torch.equal(short, ordinary)
    # sums of 11 squares and a root, 1 ulp each: 7 * 2^-24 relative to the distance
    truth = torch.cdist(a.double(), b.double())
    assert torch.allclose(short[0].double() if short.dim() == 3 else short.double(), truth, rtol=7 * 2.0 ** -24, atol=1e-30)


def test_not_a_number_and_infinities(device, monkeypatch):
    g = torch.Generator().manual_seed(3)
    a, b = torch.randn(300, 7, generator=g), torch.randn(200, 7, generator=g)
    a[5, 2], a[9, 0], b[3, 6], b[8, 1] = float("nan"), float("inf"), float("-inf"), float("nan")
    a, b = a.to(device), b.to(device)
    for p in (1.0, 2.0):
        short, ordinary = both(monkeypatch, lambda: kermac.cdist(a, b, p=p))
        assert torch.equal(short.view(torch.int32), ordinary.view(torch.int32)) or torch.allclose(short, ordinary, rtol=0, atol=0, equal_nan=True)


def test_a_set_against_itself(device, monkeypatch):
    g = torch.Generator().manual_seed(4)
    x = torch.randn(3, 400, 6, generator=g).to(device)
    short, ordinary = both(monkeypatch, lambda: kermac.run_kernel(DESCRIPTORS["gaussian"], x, x, bandwidth=2.0, regularization=1e-3))
    assert torch.equal(short, ordinary) and torch.equal(short, short.transpose(1, 2))


@pytest.mark.parametrize("M", [2 ** 31 - 1, 2 ** 31 - 1 - 200])
@pytest.mark.parametrize("k_contiguous", [False, True])
def test_a_result_of_nearly_2_to_the_31_rows(device, monkeypatch, M, k_contiguous):
    """The last tiles' row numbers, which end at M, do not fit 32 bits once a tile is added.  K = 2 with k contiguous would be 16 GB: K = 1 there."""
    monkeypatch.setenv("KERMAC_AMD_DIRECT_SHORT_MAX_K", "24")
    x = torch.empty(M, 1, device=device) if k_contiguous else torch.empty(1, M, device=device).t()
    x.copy_(torch.arange(M, dtype=torch.int32, device=device)[:, None] % 4093)
    point = torch.full((1, 1), 17.0, device=device)
    guard = torch.full((M + 64,), -5.0, device=device)
    out = guard[33:33 + M].as_strided((M, 1), (1, M))
    kermac.cdist(x, point, out=out, p=1.0)
    assert bool((guard[:33] == -5.0).all()) and bool((guard[33 + M:] == -5.0).all())
    x.sub_(17.0).abs_()
    assert torch.equal(out, x)


# (M, N, K): rows of the result contiguous.  More than 256 tiles of 128 x 128; above 8 terms 1024 columns; 13 .. 16 terms of unaligned rows only;
# 17 .. 24 from 1024 tiles on; and rows that fill the tiles of 256, more of them for more terms and for a kernel function
@pytest.mark.parametrize("M,N,K,distance,gaussian", [
    (2100, 2100, 8, True, True), (2048, 2048, 8, False, False), (30001, 150, 8, True, True), (5000, 1024, 9, True, True), (5000, 1023, 9, False, False),
    (5000, 1024, 12, True, True), (5000, 1024, 13, False, False), (5001, 1024, 13, True, True), (5001, 1024, 16, True, True), (5000, 3300, 17, True, True),
    (5000, 3200, 17, False, False), (5000, 3300, 24, True, True), (5000, 3300, 25, False, False),
    (100, 60000, 4, True, False), (100, 60000, 8, True, False), (100, 60000, 12, False, False), (256, 20000, 12, True, True), (300, 30000, 8, True, True),
    (300, 30000, 12, False, False), (504, 12000, 12, True, False), (504, 40000, 20, False, False), (1012, 20000, 20, True, True), (756, 26000, 20, False, False),
    (17, 60000, 4, True, False), (17, 60000, 5, False, False), (127, 40000, 8, True, True), (127, 40000, 12, True, False), (301, 30000, 12, True, True),
    (257, 30000, 15, True, False), (257, 60000, 20, True, False), (129, 90000, 20, True, True)])
def test_the_rule(device, M, N, K, distance, gaussian):
    a, b = torch.zeros(K, M, device=device).t(), torch.zeros(K, N, device=device).t()
    out = torch.empty(N, M, device=device).t()
    assert launches_short(lambda: kermac.cdist(a, b, out=out, p=1.0)) == distance
    with kermac.l2_mode("direct"):
        assert launches_short(lambda: kermac.run_kernel(DESCRIPTORS["gaussian"], a, b, out=out, bandwidth=1.0)) == gaussian


@pytest.mark.parametrize("K,expected", [(8, True), (9, False)])
def test_the_rule_for_a_set_against_itself(device, K, expected):
    x = torch.zeros(2100, K, device=device)
    assert launches_short(lambda: kermac.cdist(x, x, p=1.0)) == expected
