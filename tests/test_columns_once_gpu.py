"""GPU tests of gram_columns_once: the pieces of operands with the rows contiguous by one launch, at the edges of its groups of k (256, 512, 1024), of
its chunks of longer rows (512, those of gram_rows_once 1024), of its 32 rows and of the slices that pad K.  Distances keep the route's 1e-5 of the float64 truth; rows that differ by powers of two keep their bits."""
import pytest
import torch

import kermac_amd as kermac
from tests.helpers import assert_close_to_truth, kernels_of

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def wide(monkeypatch):
    monkeypatch.setenv("KERMAC_AMD_WIDE_MIN_TILES", "1")
    with kermac.l2_mode("gram_bf16", min_k=0):
        yield


@pytest.mark.parametrize("K", [1, 7, 8, 9, 15, 16, 17, 31, 33, 64, 65, 255, 256, 257, 511, 512, 513, 1009, 1023, 1024, 1025, 1040, 1536, 1537, 2047, 2048, 2049, 3001, 8192, 8193])
@pytest.mark.parametrize("M,N", [(1, 33), (31, 32), (255, 257), (130, 300)])
def test_edges_of_k_and_of_the_rows(device, K, M, N):
    g = torch.Generator().manual_seed(K + M)
    # neither base nor leading dimension aligned; a common offset, so that the centre is subtracted
    a, b = ((torch.randn(K, rows + 3, generator=g) + 30.0).to(device)[:, 1:rows + 1].t() for rows in (M, N))
    names = kernels_of(lambda: kermac.cdist(a, b, p=2.0))
    assert K == 1 or M == 1 or sum("gram_columns_once" in name for name in names) == (1 if K <= 8192 else 0)       # one row or k: of either order
    truth = torch.cdist(a.double(), b.double())[None]
    assert_close_to_truth(kermac.cdist(a, b, p=2.0), truth, rtol=1e-5, what="columns")
    other = b.contiguous()                                  # one operand of either order: a launch each
    names = kernels_of(lambda: kermac.cdist(a, other, p=2.0))
    # rows that cannot be read 16 bytes at a time take one launch up to 8192 k, others up to 2048
    assert (K > 2048 and K % 4 == 0) or K > 8192 or K == 1 or M == 1 or (sum("gram_columns_once" in name for name in names), sum("gram_rows_once" in name for name in names)) == (1, 1)
    assert_close_to_truth(kermac.cdist(a, other, p=2.0), truth, rtol=1e-5, what="columns and rows")


@pytest.mark.parametrize("K", [40, 300, 1000])
def test_batches_scales_and_sums_of_products(device, K):
    g = torch.Generator().manual_seed(K)
    scale = 2.0 ** torch.randint(-40, 40, (3, 1, 200), generator=g)
    a = (torch.randn(3, K, 200, generator=g) * scale).to(device).transpose(1, 2)
    b = torch.randn(K, 150, generator=g).to(device).t()       # shared by the batch
    got = kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)
    plain = kermac.run_kernel(kermac.kernel_descriptor_mma, a / scale.transpose(1, 2).to(device), b)
    assert torch.equal(got, plain * scale.transpose(1, 2).to(device)), "the scale of a row changed more than its exponent"
    size = a.double().abs() @ b.double().abs().t()
    assert torch.all((got.double() - a.double() @ b.double().t()).abs() <= 1e-6 * size)


def test_rows_that_are_not_numbers(device):
    g = torch.Generator().manual_seed(1)
    a, b = (torch.randn(300, rows, generator=g).to(device).t() for rows in (200, 150))
    clean = kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)
    a[33, 299], a[64, 0], b[149, 130] = float("nan"), float("inf"), float("-inf")
    got = kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)[0]
    rows, columns = torch.ones(200, dtype=torch.bool, device=device), torch.ones(150, dtype=torch.bool, device=device)
    rows[[33, 64]], columns[149] = False, False
    assert torch.equal(got[rows][:, columns], clean[0][rows][:, columns])
    assert not torch.isfinite(got[~rows]).any() and not torch.isfinite(got[:, ~columns]).any()
