"""The product kernel's 128 x 128 tile by 8 waves, which multiplies where the result has at most 512 such tiles: the same sums in the same
order as in the other tiles, so the same bits, and the same order of LDS reads and writes in the compiled kernel."""
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

import kermac_amd as kermac
from kermac_amd import _build
from tests import test_product_kernel_listing as listing
from tests.helpers import kernels_of

VARIANTS = [(symmetric, epilogue) for epilogue in ("GW_EPILOGUE_DISTANCE", "GW_EPILOGUE_DOT") for symmetric in ("true", "false")]
VARIANTS.append(("false", "GW_EPILOGUE_GRADIENT_L2"))


def test_order_of_operands_sums_and_staged_results(tmp_path):
    if shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("no hipcc")
    source, target = tmp_path / "product.hip", tmp_path / "product.s"
    source.write_text("#include <hip/hip_runtime.h>\n" f'#include "{listing.KERNELS / "gram_f16_wide.hpp"}"\n'
                      + "".join(f"template __global__ void kmc::gram_f16_wide<kmc::WideTileFew, {symmetric}, kmc::{epilogue}>(kmc::GramWideArgs);\n"
                                for symmetric, epilogue in VARIANTS))
    done = subprocess.run([_build._hipcc(), *_build.HIPCC_FLAGS, "--offload-device-only", "-S", str(source), "-o", str(target)],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]
    kernels = listing.functions(target.read_text())
    assert len(kernels) == len(VARIANTS)
    assert all(len(listing.Listing(lines).products) == 24 for lines in kernels.values())     # 3 products of 4 x 2 blocks
    listing.test_no_wave_stages_results_over_operands_that_another_has_yet_to_read(kernels)
    listing.test_lanes_of_a_wave_exchange_staged_results_in_order(kernels)
    listing.test_nothing_but_the_products_touches_the_sums_in_the_walk(kernels)


@pytest.mark.gpu
@pytest.mark.parametrize("L,M,N,K", [(1, 1, 1, 1), (1, 128, 128, 32), (1, 129, 127, 33), (3, 255, 257, 65), (9, 300, 140, 96), (2, 2048, 2048, 128),
                                     (1, 2817, 2815, 40), (1, 300, 200, 4096)])
@pytest.mark.parametrize("same", [False, True])
@pytest.mark.parametrize("kernel", ["distance", "laplace", "product"])
def test_same_bits_as_the_large_tile(device, monkeypatch, L, M, N, K, same, kernel):
    monkeypatch.setenv("KERMAC_AMD_WIDE_MIN_TILES", "1")
    gen = torch.Generator(device=device).manual_seed(L + M + N + K)
    # rows contiguous, the result too: M is the kernel's m
    a, b = (torch.randn(L, K, rows, device=device, generator=gen).transpose(1, 2) for rows in (M, N))
    b = a if same else b

    def run():
        with kermac.l2_mode("gram_bf16", min_k=1):
            if kernel == "distance":
                return kermac.cdist(a, b, p=2.0)
            if kernel == "laplace":
                return kermac.run_kernel(kermac.kernel_descriptor_laplace_l2, a, b, bandwidth=2.0)
            return kermac.run_kernel(kermac.kernel_descriptor_mma, a, b)

    assert any("EightWaves" in name for name in kernels_of(run))
    few = run()
    monkeypatch.setenv("KERMAC_AMD_WIDE_LARGE_TILE_MIN_TILES", "0")
    assert not any("EightWaves" in name for name in kernels_of(run))
    assert torch.equal(few, run())
