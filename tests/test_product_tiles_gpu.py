"""The product kernel of the workspace route in both of its tiles (128 x 128, and 256 x 128 where those are many): edges of
tiles and of steps of 32 k, one row and one column, sets against themselves, against float64 on a part of the batch."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu

# L x ceil(M / 256) x ceil(N / 128) says which tile runs: below 4096 the small one
SHAPES = [
    (1, 1, 1, 1), (1, 128, 128, 32), (1, 129, 127, 33), (3, 255, 257, 31), (2, 384, 130, 64), (1, 513, 640, 96),
    (4100, 17, 9, 40), (1100, 300, 140, 33), (1030, 257, 256, 32), (2050, 1, 129, 65), (1030, 512, 129, 95),
]


def _truth(a, b, entries):
    return torch.stack([torch.cdist(a[e].double().cpu(), b[e].double().cpu(), p=2.0, compute_mode="donot_use_mm_for_euclid_dist")
                        for e in entries]).to(a.device)


@pytest.fixture(autouse=True)
def any_size(monkeypatch):
    monkeypatch.setenv("KERMAC_AMD_WIDE_MIN_TILES", "1")


@pytest.mark.parametrize("L,M,N,K", SHAPES)
@pytest.mark.parametrize("panel", [False, True])
def test_distances_and_products(device, L, M, N, K, panel):
    gen = torch.Generator(device=device).manual_seed(L + M + N + K)
    a, b = (torch.randn(L, rows, K, device=device, generator=gen) for rows in (M, N))
    if panel:
        a, b = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (a, b))
    entries = sorted({0, L // 2, L - 1})
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(a, b, p=2.0)
        dot = kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)
    truth = _truth(a, b, entries)
    assert ((got[entries].double() - truth).abs() <= 1e-5 * truth).all()        # the route's stated tolerance
    # error of the three products of pieces: below 3 * 2^-22 sum |a b|, beside the fp32 sum of K terms
    exact = torch.matmul(a[entries].double(), b[entries].double().transpose(1, 2).contiguous())
    scale = torch.matmul(a[entries].double().abs(), b[entries].double().abs().transpose(1, 2).contiguous())
    assert ((dot[entries].double() - exact).abs() <= 1e-6 * scale).all()


@pytest.mark.parametrize("L,M,N,K,tile", [(192, 256, 256, 48, "128, 128"), (193, 256, 256, 48, "256, 128"), (224, 256, 256, 48, "256, 128"),
                                          (225, 256, 256, 48, "128, 128"), (225, 256, 256, 2033, "256, 128"), (256, 256, 256, 2048, "256, 128"),
                                          (257, 256, 256, 2048, "128, 128"), (769, 128, 128, 48, "128, 128"), (56, 600, 300, 48, "256, 128"),
                                          (86, 300, 600, 48, "128, 128"), (2, 2816, 2810, 2048, "256, 128")])
@pytest.mark.parametrize("same", [False, True])
def test_which_tile_runs(device, L, M, N, K, tile, same):
    """A round of the chip is 768 tiles of 128 x 128 or 512 of 256 x 128: the large ones where they are one round and the small ones are a
    little more (up to 896) or K is long, but not for a set against itself."""
    gen = torch.Generator(device=device).manual_seed(L)
    # rows contiguous, the result too: M is the kernel's m
    a, b = (torch.randn(L, K, rows, device=device, generator=gen).transpose(1, 2) for rows in (M, N))
    b = a if same else b
    out = torch.empty(L, b.size(1), M, device=device).transpose(1, 2)
    with kermac.l2_mode("gram_bf16", min_k=1):
        names = kernels_of(lambda: kermac.cdist(a, b, out=out, p=2.0))
    ran = [name.split("WideTile<")[1].split(">")[0] for name in names if "gram_f16_wide<" in name]
    assert ran == ["128, 128" if same else tile]
    rows, columns = (sorted({min(at, n - 1) for at in (0, 1, 127, 128, 255, 256, n // 2, n - 129, n - 1)}) for n in (M, b.size(1)))
    truth = _truth(a[:, rows], b[:, columns], [0, L - 1])
    assert ((out[[0, L - 1]][:, rows][:, :, columns].double() - truth).abs() <= 1e-5 * truth).all()


@pytest.mark.parametrize("L,M,N,K", [(7, 130, 129, 40), (8, 130, 257, 33), (9, 300, 140, 32), (23, 65, 129, 20), (8, 1024, 2048, 16), (8, 1024, 2049, 16),
                                     (4100, 17, 9, 40), (4100, 129, 128, 8)])
@pytest.mark.parametrize("same", [False, True])
def test_every_entry_of_a_batch(device, L, M, N, K, same):
    """Eight entries at a time have an XCD each, up to 128 tiles per entry; the entries behind the last eight, and larger ones, are spread over all."""
    if same and M == 1024:
        M = N = 1408 if N == 2048 else 1409             # 121 and 144 tiles
    gen = torch.Generator(device=device).manual_seed(L + M)
    a, b = (torch.randn(L, rows, K, device=device, generator=gen) for rows in (M, N))
    b = a if same else b
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(a, b, p=2.0)
        dot = kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)
    for entry in range(0, L, 1 if L < 100 else 53):
        x, y = a[entry].double(), b[entry].double()
        exact, scale = x @ y.t().contiguous(), x.abs() @ y.abs().t().contiguous()
        truth = ((x * x).sum(1)[:, None] + (y * y).sum(1)[None] - 2 * exact).clamp_min(0).sqrt()
        if same:
            truth.fill_diagonal_(0)
        assert ((got[entry].double() - truth).abs() <= 1e-5 * truth).all()
        assert ((dot[entry].double() - exact).abs() <= 1e-6 * scale).all()        # as above


@pytest.mark.parametrize("L,M,K", [(1, 1, 5), (2, 130, 33), (1, 385, 64), (1400, 257, 40), (4200, 140, 32)])
def test_a_set_against_itself(device, L, M, K):
    gen = torch.Generator(device=device).manual_seed(M)
    a = torch.randn(L, M, K, device=device, generator=gen)
    entries = sorted({0, L // 2, L - 1})
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(a, a, p=2.0)
    truth = _truth(a, a, entries)
    assert ((got[entries].double() - truth).abs() <= 1e-5 * truth).all()
    assert torch.equal(got, got.transpose(1, 2))
    assert (torch.diagonal(got, dim1=1, dim2=2) == 0).all()


@pytest.mark.parametrize("L,M,K", [(1, 1, 130), (1, 129, 128), (2, 257, 140), (1, 385, 200), (3, 128, 33)])
@pytest.mark.parametrize("panel", [False, True])
def test_a_set_against_itself_in_one_step(device, monkeypatch, L, M, K, panel):
    """The split kernel without a workspace: zero on the diagonal, symmetric bit for bit, also where the tile is recomputed
    (a pair of near-duplicates, a row that is not a number), and a set against a run of its own rows."""
    monkeypatch.setenv("KERMAC_AMD_L2_WORKSPACE", "0")
    gen = torch.Generator(device=device).manual_seed(M + K)
    a = torch.randn(L, M, K, device=device, generator=gen)
    if M > 200:
        a[0, 150] = a[0, 3] + 1e-3
        a[-1, 200, 5] = float("nan")
    if panel:
        a = a.transpose(1, 2).contiguous().transpose(1, 2)
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(a, a, p=2.0)
        run = kermac.cdist(a[:, M // 3:], a, p=2.0)
    truth = _truth(a, a, list(range(L)))
    finite = torch.isfinite(truth)
    assert torch.equal(torch.isfinite(got), finite)
    assert ((got.double() - truth).abs() <= 1e-5 * truth)[finite].all()
    clean = torch.where(finite, got, torch.zeros_like(got))
    assert torch.equal(clean, clean.transpose(1, 2)) and (torch.diagonal(clean, dim1=1, dim2=2) == 0).all()
    part = truth[:, M // 3:]
    assert ((run.double() - part).abs() <= 1e-5 * part)[torch.isfinite(part)].all()


@pytest.mark.parametrize("K", [20, 300])
@pytest.mark.parametrize("panel", [False, True])
def test_distrusted_parts_of_a_large_tile(device, monkeypatch, panel, K):
    """A tile of 256 x 128 is two parts to the repair launch: a near-duplicate in one of them, in the other, in both, a row that is not a
    number; of a set against itself also with twins on the diagonal and in the part above it inside a tile."""
    monkeypatch.setenv("KERMAC_AMD_WIDE_LARGE_TILE_MIN_TILES", "1")
    monkeypatch.setenv("KERMAC_AMD_L2_PROBE", "0")
    gen = torch.Generator(device=device).manual_seed(K)
    a, b = torch.randn(700, K, device=device, generator=gen), torch.randn(515, K, device=device, generator=gen)
    b[5], b[130], b[300], b[301] = a[3] + 1e-3, a[140] + 1e-3, a[400] + 1e-3, a[513] + 1e-3
    own = a.clone()
    own[100], own[300], own[500] = own[20] + 1e-3, own[140] + 1e-3, own[390] + 1e-3      # one part, across parts, above the diagonal
    a[650, K // 2], own[690, 0] = float("nan"), float("inf")

    def stored(x):
        return x.t().contiguous().t() if panel else x

    a, b, own = stored(a), stored(b), stored(own)
    calls = []
    for x, y in ((a, b), (own, own)):
        out = torch.empty(y.size(0), x.size(0), device=device).t()
        with kermac.l2_mode("gram_bf16", min_k=1):
            calls += [name for name in kernels_of(lambda: kermac.cdist(x, y, out=out, p=2.0)) if "gram_f16_wide<" in name]
        truth = _truth(x[None], y[None], [0])[0]
        finite = torch.isfinite(truth)
        assert (torch.isfinite(out) == finite).all()
        assert ((out.double() - truth).abs() <= 1e-5 * truth)[finite].all()
        if y is x:
            clean = torch.where(finite, out, torch.zeros_like(out))
            assert torch.equal(clean, clean.t()) and (torch.diagonal(clean) == 0).all()
    assert len(calls) == 2 and all("WideTile<256, 128>" in name for name in calls)


@pytest.mark.parametrize("K", [3, 255, 256, 257, 260, 511, 512, 513, 1000, 1023, 1024, 1025])
@pytest.mark.parametrize("form", ["rows", "misaligned", "a_panel", "b_panel", "offset"])
def test_rows_of_any_length(device, K, form):
    """Pieces made in one pass (k contiguous, K up to 1024) and in two, in every mixture, with and without a centre."""
    L, M, N = 2, 131, 47
    gen = torch.Generator(device=device).manual_seed(K)
    a, b = (torch.randn(L, rows, K, device=device, generator=gen) for rows in (M, N))
    if form == "misaligned":
        a, b = (torch.nn.functional.pad(x, (1, 0))[:, :, 1:] for x in (a, b))
    elif form == "a_panel":
        a = a.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "b_panel":
        b = b.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "offset":
        a, b = a + 30.0, b + 30.0
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(a, b, p=2.0)
        alone = kermac.cdist(a, a, p=2.0)
    # the rounding of the offset operands themselves is in both sides
    truth, truth_alone = _truth(a, b, [0, 1]), _truth(a, a, [0, 1])
    assert ((got.double() - truth).abs() <= 1e-5 * truth).all()
    assert ((alone.double() - truth_alone).abs() <= 1e-5 * truth_alone).all()


def test_rows_that_are_not_numbers(device):
    gen = torch.Generator(device=device).manual_seed(3)
    a, b = (torch.randn(rows, 300, device=device, generator=gen) for rows in (200, 150))
    a[5, 7], b[9, 299] = float("nan"), float("inf")
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(a, b, p=2.0)[0]
    truth = _truth(a[None], b[None], [0])[0]
    assert torch.equal(torch.isnan(got), torch.isnan(truth)) and torch.equal(torch.isinf(got), torch.isinf(truth))
    finite = torch.isfinite(truth)
    assert ((got.double() - truth).abs() <= 1e-5 * truth)[finite].all()


def _variants(x, y):
    """Whether the one-step split kernel that a call runs is the one that looks for equal points (its last template argument)."""
    with kermac.l2_mode("gram_bf16", min_k=1):
        return [name.split("gram_bf16_l2_kernel<")[1].split(">")[0].split(",")[-1].strip()
                for name in kernels_of(lambda: kermac.cdist(x, y, p=2.0)) if "gram_bf16_l2_kernel<" in name]


@pytest.mark.parametrize("panel", [False, True])
def test_only_a_set_against_itself_looks_for_equal_points(device, monkeypatch, panel):
    """The comparisons of the variant cost any other call up to a tenth."""
    monkeypatch.setenv("KERMAC_AMD_L2_WORKSPACE", "0")
    gen = torch.Generator(device=device).manual_seed(5)
    a, b = torch.randn(300, 256, device=device, generator=gen), torch.randn(260, 260, device=device, generator=gen)[:, :256]
    if panel:
        a, b = (x.t().contiguous().t() for x in (a, b))
    assert _variants(a, b) == ["false"]
    assert _variants(a, a) == ["true"]
    assert _variants(a[30:], a) == ["true"] and _variants(a, a[30:]) == ["true"]
    assert _variants(a[:100], a[:100]) == ["false"]        # one tile is left to the repair launch


@pytest.mark.parametrize("panel", [False, True])
def test_parts_of_one_set_that_share_no_point(device, monkeypatch, panel):
    monkeypatch.setenv("KERMAC_AMD_L2_WORKSPACE", "0")
    gen = torch.Generator(device=device).manual_seed(6)
    x = torch.randn(700, 256, device=device, generator=gen)
    x = x.t().contiguous().t() if panel else x
    for first, second in ((x[:300], x[300:]), (x[300:], x[:300]), (x[:150], x[400:])):
        assert _variants(first, second) == ["false"]
    assert _variants(x[:301], x[300:]) == ["true"] and _variants(x[300:], x[:301]) == ["true"]      # one point on both sides
    with kermac.l2_mode("gram_bf16", min_k=1):
        got = kermac.cdist(x[:301], x[300:], p=2.0)[0]
    truth = _truth(x[None, :301], x[None, 300:], [0])[0]
    assert got[300, 0] == 0 and ((got.double() - truth).abs() <= 1e-5 * truth).all()


def _points(distribution, M, K, device):
    gen = torch.Generator(device=device).manual_seed(M + K)
    normal = lambda *shape: torch.randn(*shape, device=device, generator=gen)
    if distribution == "uniform":
        return torch.rand(M, K, device=device, generator=gen)
    if distribution == "heavy tails":
        return normal(M, K) * torch.exp(1.5 * normal(M, K))
    if distribution == "mostly zeros":
        return (normal(M, K) - 0.8).clamp_min(0)
    if distribution == "clusters":                      # squared distances from about a quarter of the norms on, where trust ends
        return normal(40, K)[torch.randint(0, 40, (M,), device=device, generator=gen)] + 0.75 * normal(M, K)
    if distribution == "scaled rows":
        return normal(M, K) * torch.exp(2.0 * normal(M, 1))
    return normal(M, K)


# the workspace route and the one-step split kernel, two storage orders
@pytest.mark.parametrize("M,K,panel", [(1400, 400, False), (2000, 256, False), (2000, 1024, False), (1000, 200, True), (1500, 200, True), (2400, 1024, True)])
@pytest.mark.parametrize("distribution", ["normal", "uniform", "heavy tails", "mostly zeros", "clusters", "scaled rows"])
def test_the_error_of_a_set_against_itself_is_no_larger_than_the_direct_kernels(device, monkeypatch, M, K, panel, distribution):
    """Sets against themselves multiply pieces of their values by default.  The direct kernel subtracts in fp32 and rounds once per term; the
    pieces hold 22 or 24 bits, and the products round once per 16 or 32 terms, which leaves the error (2-norm, against float64) below the direct
    kernel's, of the whole result and of the parts on its diagonal."""
    x = _points(distribution, M, K, device)
    stored = x.t().contiguous().t() if panel else x
    centred = x.double() - x.double().mean(0)
    squares = (centred * centred).sum(1)
    truth = (squares[:, None] + squares[None] - 2 * (centred @ centred.t().contiguous())).clamp_min(0).sqrt().fill_diagonal_(0)
    got = kermac.cdist(stored, stored, p=2.0)[0].double()
    monkeypatch.setenv("KERMAC_AMD_NO_CUT", "1")
    with kermac.l2_mode("direct"):
        direct = kermac.cdist(stored, stored, p=2.0)[0].double()
    diagonal = torch.block_diag(*[torch.ones(min(128, M - at), min(128, M - at), device=device, dtype=torch.bool) for at in range(0, M, 128)]).bool()
    for part in (torch.ones_like(diagonal), diagonal):
        assert (got - truth)[part].norm() <= (direct - truth)[part].norm()


@pytest.mark.parametrize("M,K", [(1300, 512), (1400, 784), (1664, 1030), (1300, 4096)])
@pytest.mark.parametrize("distribution", ["normal", "clusters"])
def test_a_small_set_against_itself_keeps_the_short_sums_of_the_direct_path(device, M, K, distribution):
    """Where the direct path is cut over k (512 terms and more, fewer than 192 tiles) its error is below that of the pieces."""
    x = _points(distribution, M, K, device)
    got = kermac.cdist(x, x, p=2.0)
    with kermac.l2_mode("direct"):
        assert torch.equal(got, kermac.cdist(x, x, p=2.0))
