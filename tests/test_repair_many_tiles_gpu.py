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
