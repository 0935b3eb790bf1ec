// A kernel matrix times coefficients by gram_f16_wide: what the caller brings, and where the launch left the products of the tiles.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

#include "../kernels/build_kernel.hpp"
#include "host_common.hpp"

namespace kmc_host {

constexpr int CONTRACTION_MAX_OUTPUTS = 32;

struct Contraction {
    const float *coef; int64_t coef_ld, coef_bs;
    int outputs;
    float *products;      // [tile of 128 n][l][m][outputs padded to 4]
    int *stamps;          // [l][tile of 128 m][tile of 128 n]: tiles whose product is to be recomputed (squared differences)
};

int64_t gram_f16_wide_contraction_bytes(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, int outputs);
hipError_t launch_gram_f16_wide(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, hipStream_t stream, bool *taken,
                                const unsigned **sample = nullptr, Contraction *contraction = nullptr);
hipError_t launch_sum_products(const float *products, int tiles, int l, int m, int outputs, float *out, int64_t out_ld, int64_t out_bs, bool accumulate,
                               hipStream_t stream);

}  // namespace kmc_host
