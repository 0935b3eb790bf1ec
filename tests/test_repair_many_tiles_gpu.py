"""The repair launch of a matrix-core result of more tiles than the chip holds workgroups: every distrusted part is found and recomputed, wherever it lies."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu


def _stored(x, k_contiguous):
    return x if k_contiguous else x.transpose(-1, -2).contiguous().transpose(-1, -2)


# tiles of 128 x 128: 65 x 65, 3 x 38 x 38, 17 x 245 with remainders on both sides, a triangle of 92
@pytest.mark.parametrize("L,M,N,K,own", [(1, 8320, 8320, 64, False), (3, 4800, 4810, 72, False), (1, 2050, 31300, 96, False), (1, 11700, 11700, 64, True)])
@pytest.mark.parametrize("k_contiguous", [True, False])
def test_every_near_duplicate_is_found(device, L, M, N, K, own, k_contiguous):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    a = torch.randn(L, M, K, device=device, generator=g)
    b = a if own else torch.randn(L, N, K, device=device, generator=g)
    # the corners, and 60 pairs anywhere, a thousandth apart: |a|^2 + |b|^2 - 2 a.b says nothing about their distance
    anywhere = [torch.randperm(rows - 4, device=device, generator=g)[:60] + 2 for rows in (M, N)]
    rows = torch.cat([torch.tensor([0, 1, M - 1, M - 2], device=device), anywhere[0]])
    columns = torch.cat([torch.tensor([0, N - 1, 1, N - 2], device=device), anywhere[1]])
    if own:
        keep = ~torch.isin(columns, rows)
        rows, columns = rows[keep], columns[keep]
    assert len(rows) > 50
    b[:, columns] = a[:, rows] + 1e-3 * torch.randn(L, len(rows), K, device=device, generator=g)
    a, b = _stored(a, k_contiguous), None if own else _stored(b, k_contiguous)
    b = a if own else b
    call = lambda: kermac.cdist(a, b, p=2.0)
    names = kernels_of(call)
    assert any("gram_f16_wide" in name for name in names) and any("build_kernel_repair" in name for name in names)
    want = (a[:, rows].double() - b[:, columns].double()).norm(dim=-1)
    for _ in range(2):
        got = call()[:, rows, columns].double()
        # the direct kernel: a difference is off by 2^-24 of itself, a sum of K squares by K 2^-24 at most, the root by half of that
        assert float(((got - want) / want).abs().max()) < (K / 2 + 3) * 2.0 ** -24


@pytest.mark.parametrize("probe", [True, False])
@pytest.mark.parametrize("k_contiguous", [True, False])
def test_a_result_that_is_all_marked(device, monkeypatch, probe, k_contiguous):
    """Points in 64 places, so that every tile has pairs below the threshold: the direct kernel's bits everywhere, with the sample and without it."""
    if not probe:
        monkeypatch.setenv("KERMAC_AMD_L2_PROBE", "0")
    g = torch.Generator(device=device).manual_seed(5)
    places = torch.randn(64, 64, device=device, generator=g)
    a, b = (_stored(places[torch.randint(0, 64, (rows,), device=device, generator=g)] + 1e-3 * torch.randn(rows, 64, device=device, generator=g), k_contiguous)
            for rows in (8448, 8576))
    assert any("gram_f16_wide" in name for name in kernels_of(lambda: kermac.cdist(a, b, p=2.0)))
    got = kermac.cdist(a, b, p=2.0)
    with kermac.l2_mode("direct"):
        assert torch.equal(got, kermac.cdist(a, b, p=2.0))


def _in_places(rows, K, places, device, g):
    """Points stored place by place: their near-duplicates fill blocks of neighbouring tiles on the diagonal."""
    labels = torch.randint(0, len(places), (rows,), device=device, generator=g).sort().values
    return places[labels] + 1e-3 * torch.randn(rows, K, device=device, generator=g), labels


@pytest.mark.parametrize("M,N,K,places,own", [(9000, 8900, 72, 5, False), (8330, 8330, 64, 2, False), (11700, 11700, 64, 9, True)])
@pytest.mark.parametrize("k_contiguous", [True, False])
def test_marked_tiles_that_lie_together(device, M, N, K, places, own, k_contiguous):
    """Blocks of hundreds of marked tiles, of two places half of all: the direct kernel's bits where two points share a place."""
    g = torch.Generator(device=device).manual_seed(M + K)
    centres = 10.0 * torch.randn(places, K, device=device, generator=g)
    a, label_a = _in_places(M, K, centres, device, g)
    b, label_b = (a, label_a) if own else _in_places(N, K, centres, device, g)
    a, b = _stored(a, k_contiguous), None if own else _stored(b, k_contiguous)
    b = a if own else b
    names = kernels_of(lambda: kermac.cdist(a, b, p=2.0))
    assert any("gram_f16_wide" in name for name in names)
    scan, repair = (next((i for i, name in enumerate(names) if what in name), None) for what in ("repair_scan", "build_kernel_repair"))
    assert scan is not None and repair == scan + 1, names
    out = torch.empty(1, M, N, device=device)
    graph = torch.cuda.CUDAGraph()
    scratch = torch.empty(1 << 25, dtype=torch.uint8, device=device)
    with kermac.scratch(scratch):
        with torch.cuda.graph(graph):
            kermac.cdist(a, b, p=2.0, out=out)
        with kermac.l2_mode("direct"):
            want = kermac.cdist(a, b, p=2.0)[0]
    same = label_a[:, None] == label_b[None]
    for replay in range(3):                    # the counters are cleared on every one
        out.fill_(-1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0][same], want[same])
        far = ~same
        assert not far.any() or float(((out[0][far] - want[far]).double() / want[far]).abs().max()) < 1e-5


def test_marked_tiles_that_lie_together_are_shared_out(device):
    """64 places of 12000 x 9000 points, 1 tile in 64 marked.  With all marked tiles of a run of 32 in one workgroup the call took 3.2 times as long as one
    without any, shared out 1.4 times."""
    g = torch.Generator(device=device).manual_seed(1)
    M, N, K = 12000, 9000, 512
    centres = 10.0 * torch.randn(64, K, device=device, generator=g)
    packed = tuple(_in_places(rows, K, centres, device, g)[0] for rows in (M, N))
    spread = tuple(torch.randn(rows, K, device=device, generator=g) for rows in (M, N))

    def least(a, b):
        times = []
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            kermac.cdist(a, b, p=2.0)
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    assert least(*packed) < 2.0 * least(*spread)
