"""GPU tests of the centre that the route through a workspace makes for itself (KMC_FLAG_GRAM_OWN_CENTRE): data with a common
offset stay on the matrix cores, which they can only if the centre was found and every kernel of the call decided to subtract it."""
import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _backend, build_a_kernel as module
from tests.helpers import assert_close_to_truth, kernels_of, make_operand

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def wide(monkeypatch):
    monkeypatch.setenv("KERMAC_AMD_WIDE_MIN_TILES", "1")
    with kermac.l2_mode("gram_bf16", min_k=0):
        yield


# 512 rows are averaged whole, more in runs of 16 (k contiguous) or 64; 64 pairs of sums to a wave: K = 1024, 256 with the rows contiguous; K above
# 1024 takes the row kernels in two passes; 16 or 64 k per workgroup
@pytest.mark.parametrize("M,N,K,L", [(511, 300, 96, 1), (512, 300, 65, 1), (513, 520, 64, 1), (527, 300, 784, 1), (700, 129, 1024, 1), (2000, 300, 200, 1),
                                     (576, 260, 256, 1), (575, 260, 260, 1), (600, 300, 1030, 1), (129, 200, 1025, 2), (1300, 140, 70, 40), (100, 300, 96, 3)])
@pytest.mark.parametrize("layout", ["cc", "rr", "cr"])
@pytest.mark.parametrize("shared", [False, True])
def test_a_common_offset_stays_on_the_matrix_cores(device, M, N, K, L, layout, shared):
    g = torch.Generator().manual_seed(M + N + K + L)
    # the entries of a batch sit in different places
    offset = 100.0 * torch.arange(1, L + 1).reshape(L, 1, 1)
    if shared:
        offset = offset[:1]
    a = make_operand(1 if shared else L, M, K, layout[0] == "c", device, g) + offset.to(device)
    b = make_operand(L, N, K, layout[1] == "c", device, g) + offset.to(device)
    got = kermac.cdist(a, b, p=2.0)
    assert_close_to_truth(got, torch.cdist(a.double().expand(L, M, K), b.double()), rtol=1e-5, what="own centre")
    with kermac.l2_mode("direct"):
        direct = kermac.cdist(a, b, p=2.0)
    # a part that the repair launch recomputed has the direct kernel's bits
    first = torch.tensor([[torch.equal(got[l, m:m + 128, n:n + 128], direct[l, m:m + 128, n:n + 128]) for m in range(0, M, 128)
                           for n in range(0, N, 128)] for l in range(L)])
    assert first.float().mean() < 0.1, "parts were repaired: the centre was not subtracted"


def test_launches_of_a_call(device):
    """One launch for the centre, none for its flag; none of it for a call whose centre is switched off."""
    a, b = torch.randn(600, 200, device=device), torch.randn(500, 200, device=device)
    names = kernels_of(lambda: kermac.cdist(a, b, p=2.0))
    assert sum("sample_mean" in name for name in names) == 1 and not any("centre_flag" in name for name in names)


def test_points_around_the_origin_are_taken_as_they_are(device, monkeypatch):
    """A centre well inside the cloud of points is not subtracted: the bits are those of a call without one."""
    for rows_contiguous in (False, True):
        g = torch.Generator().manual_seed(7)
        a, b = (make_operand(1, rows, 300, rows_contiguous, device, g, batch=False) for rows in (900, 400))
        with_centre = kermac.cdist(a, b, p=2.0)
        monkeypatch.setenv("KERMAC_AMD_L2_CENTRE", "0")
        assert torch.equal(with_centre, kermac.cdist(a, b, p=2.0))
        monkeypatch.setenv("KERMAC_AMD_L2_CENTRE", "1")


def test_data_that_are_not_numbers(device):
    a, b = torch.randn(600, 200, device=device) + 50.0, torch.randn(300, 200, device=device) + 50.0
    a[5, 7], b[200, 3] = float("nan"), float("inf")
    got = kermac.cdist(a, b, p=2.0)[0]
    with kermac.l2_mode("direct"):
        assert torch.equal(torch.isnan(got), torch.isnan(kermac.cdist(a, b, p=2.0)[0]))
    clean = torch.cdist(a.double(), b.double())
    keep = torch.isfinite(clean)
    assert_close_to_truth(got[keep], clean[keep], rtol=1e-5, what="beside rows that are not numbers")


def test_the_query_counts_the_room_for_it(device):
    a, b = torch.empty(600, 200, device=device), torch.empty(500, 200, device=device)
    plan = module._plan_run_kernel(kermac.kernel_descriptor_l2_norm, a, b, None, None, None, None, None, None, None, 0, 0, False)
    without = _backend.gram_workspace_bytes(plan.params)
    plan.params.flags |= _backend.FLAG_GRAM_OWN_CENTRE
    assert _backend.gram_workspace_bytes(plan.params) >= without + 4 * (2 * 256 + 64)
