"""CPU test on the compiler's listing of the product kernel that contracts its tiles: the orders of operands, sums and exchanged values that
test_product_kernel_listing.py asks of the kernels that store them."""
import shutil
import subprocess
from pathlib import Path

import pytest

from kermac_amd import _build
from tests import test_product_kernel_listing as listing


@pytest.mark.parametrize("tile", ["WideTileSmall", "WideTileFew"])
def test_order_of_operands_sums_and_exchanged_values(tmp_path, tile):
    if shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("no hipcc")
    source, target = tmp_path / "product.hip", tmp_path / "product.s"
    kinds = [(value, columns) for value in ("DISTANCE", "DOT") for columns in (16, 32)]
    source.write_text("#include <hip/hip_runtime.h>\n" f'#include "{listing.KERNELS / "gram_f16_wide.hpp"}"\n'
                      + "".join(f"template __global__ void kmc::gram_f16_wide<kmc::{tile}, false, kmc::GW_EPILOGUE_{value} + kmc::GW_CONTRACT_{columns}>"
                                "(kmc::GramWideArgs);\n" for value, columns in kinds))
    done = subprocess.run([_build._hipcc(), *_build.HIPCC_FLAGS, "--offload-device-only", "-S", str(source), "-o", str(target)],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]
    # the products of the contraction are the compiler's own and none of the walk's
    kernels = listing.functions(target.read_text().replace("v_mfma_f32_16x16x4_f32", "v_contract"))
    assert len(kernels) == len(kinds)
    listing.test_no_wave_stages_results_over_operands_that_another_has_yet_to_read(kernels)
    listing.test_lanes_of_a_wave_exchange_staged_results_in_order(kernels)
    listing.test_nothing_but_the_products_touches_the_sums_in_the_walk(kernels)
