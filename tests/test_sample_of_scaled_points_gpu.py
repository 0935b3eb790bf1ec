"""The sample in front of a matrix-core launch looks at up to 128 of the k.  Where a few k hold most of every distance, pairs look like near-duplicates on the
others; that is no reason to leave a call to the direct kernel, which is slower and, uncut over a long contraction, less exact.

Tolerance: 1e-5 of every distance (the route's), and a 2-norm error of at most 1.25 times that of the same call without a sample."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu


def _points(kind, L, rows, K, k_contiguous, device, g, centres=None):
    x = torch.randn(L, rows, K, device=device, generator=g)
    if kind == "heavy":
        x = x / torch.rand(L, rows, K, device=device, generator=g).clamp_min(1e-3)
    elif kind == "scaled":
        h = torch.Generator(device=device).manual_seed(K)
        x = x * 10.0 ** (6.0 * (torch.rand(K, device=device, generator=h) - 0.5))
    elif kind == "places":
        x = centres[torch.randint(0, len(centres), (L, rows), device=device, generator=g)] + 1e-3 * x
    return x if k_contiguous else x.transpose(-1, -2).contiguous().transpose(-1, -2)


@pytest.mark.parametrize("kind,L,M,N,K,k_contiguous", [("heavy", 2, 701, 256, 3648, False), ("scaled", 2, 448, 1420, 2048, False), ("scaled", 4, 324, 499, 670, False),
                                                       ("scaled", 2, 390, 448, 1552, True), ("scaled", 1, 2500, 2500, 1030, True), ("scaled", 1, 2000, 3000, 2304, True)])
def test_calls_of_scaled_points_stay_on_the_matrix_cores(device, monkeypatch, kind, L, M, N, K, k_contiguous):
    g = torch.Generator(device=device).manual_seed(M + N + K)
    a, b = (_points(kind, L, rows, K, k_contiguous, device, g) for rows in (M, N))
    got = kermac.cdist(a, b, p=2.0)
    assert any("gram_f16_wide" in name for name in kernels_of(lambda: kermac.cdist(a, b, p=2.0)))
    want = torch.stack([torch.cdist(x, y, compute_mode="donot_use_mm_for_euclid_dist") for x, y in zip(a.double(), b.double())])
    error = (got.double() - want).abs()
    assert torch.all(error <= 1e-5 * want)
    monkeypatch.setenv("KERMAC_AMD_L2_PROBE", "0")
    unsampled = kermac.cdist(a, b, p=2.0)
    assert float(error.norm()) <= 1.25 * float((unsampled.double() - want).norm())
    assert torch.equal(got, unsampled), "the sample changes nothing here"


@pytest.mark.parametrize("L,M,N,K,k_contiguous", [(1, 600, 3000, 250, True), (2, 448, 1420, 2048, False), (1, 2000, 2000, 784, True)])
def test_near_duplicates_are_left_to_the_direct_kernel(device, monkeypatch, L, M, N, K, k_contiguous):
    """Points in 16 places stored in any order: every tile has near-duplicates, on all k as on the sampled ones."""
    g = torch.Generator(device=device).manual_seed(M + N + K)
    centres = 10.0 * torch.randn(16, K, device=device, generator=g)
    a, b = (_points("places", L, rows, K, k_contiguous, device, g, centres) for rows in (M, N))
    assert any("gram_f16_wide" in name for name in kernels_of(lambda: kermac.cdist(a, b, p=2.0)))
    got = kermac.cdist(a, b, p=2.0)
    monkeypatch.setenv("KERMAC_AMD_NO_CUT", "1")
    with kermac.l2_mode("direct"):
        assert torch.equal(got, kermac.cdist(a, b, p=2.0))
