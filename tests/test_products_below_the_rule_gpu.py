"""Sums of products below the library's rule for the route through fp16 pieces: they stay on the direct kernel, whose error is bounded by the sum of the terms'
magnitudes alone.  Pieces are scaled by the largest magnitude of a row; what lies far below it is held to fewer bits, which is too few where the other operand is large just there.

Tolerance: a product rounds by 2^-24 of itself and a fused sum of K terms by at most K 2^-24 of their magnitudes."""
import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend
from tests.helpers import kernels_of

pytestmark = pytest.mark.gpu


# sizes around 20000 tiles of 128 x 128 times k, where the route was once taken: one problem and batches, both storage orders, a set against itself
@pytest.mark.parametrize("L,M,N,K,k_contiguous", [(1, 640, 4045, 200, True), (2, 6110, 382, 87, False), (1, 1263, 1263, 320, False), (4, 917, 375, 230, True),
                                                  (3, 129, 4500, 131, False), (1, 131, 16001, 93, True), (1, 2000, 2000, 128, True)])
@pytest.mark.parametrize("decades", [0, 6, 8, 10])
def test_features_of_opposite_scales(device, L, M, N, K, k_contiguous, decades):
    g = torch.Generator(device=device).manual_seed(M + N + K)

    def points(rows, scales):
        x = torch.randn(L, rows, K, device=device, generator=g) * scales
        return x if k_contiguous else x.transpose(-1, -2).contiguous().transpose(-1, -2)

    scales = 10.0 ** (decades * (torch.rand(K, device=device, generator=g) - 0.5))
    a, b = points(M, scales), points(N, 1.0 / scales)
    call = lambda: kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)
    got = call().double()
    want, size = a.double() @ b.double().mT, a.double().abs() @ b.double().abs().mT
    assert float(((got - want).abs() / size).max()) <= (K + 1) * 2.0 ** -24
    assert not any("gram_f16_wide" in name for name in kernels_of(call))
    with kermac.l2_mode("direct"):
        assert torch.equal(got.float(), call())
