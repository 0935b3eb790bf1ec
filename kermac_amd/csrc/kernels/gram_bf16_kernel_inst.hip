// Ahead-of-time instantiations of the split-bf16 matrix-core L2 kernel for all 16
// (A loader, B loader) pairs, plus the ragged-K variants of the pairs with 128-bit row-major loads.  Compiled twice: with
// KMC_SAME_POINTS=1 the variants that look for equal points (rows of one set on both sides), which have the same layout on both sides,
// though not always the same alignment.
#include <hip/hip_runtime.h>

#include "launch.hpp"
#include "gram_bf16_kernel.hpp"

namespace kmc_host {

#ifndef KMC_SAME_POINTS
#error "compile with -DKMC_SAME_POINTS=0 and -DKMC_SAME_POINTS=1"
#endif

template <int LOAD_A, int LOAD_B>
static hipError_t launch_one(const kmc::BuildKernelArgs &args, dim3 grid, hipStream_t stream)
{
    constexpr bool same_points = KMC_SAME_POINTS != 0;
    constexpr bool a_rows = LOAD_A == kmc::LOAD_ROW_VEC || LOAD_A == kmc::LOAD_ROW_SCALAR;
    constexpr bool b_rows = LOAD_B == kmc::LOAD_ROW_VEC || LOAD_B == kmc::LOAD_ROW_SCALAR;
    if constexpr (same_points && a_rows != b_rows) {
        return hipErrorInvalidValue;
    } else {
        constexpr bool has_ragged_variant = LOAD_A == kmc::LOAD_ROW_VEC || LOAD_B == kmc::LOAD_ROW_VEC;
        const bool ragged = has_ragged_variant && args.k % kmc::BK_TILE_K != 0;
        if (args.centre)
            return ragged ? launch(kmc::gram_bf16_l2_kernel<LOAD_A, LOAD_B, has_ragged_variant, true, same_points>, grid, dim3(kmc::BK_THREADS), stream, args)
                          : launch(kmc::gram_bf16_l2_kernel<LOAD_A, LOAD_B, false, true, same_points>, grid, dim3(kmc::BK_THREADS), stream, args);
        return ragged ? launch(kmc::gram_bf16_l2_kernel<LOAD_A, LOAD_B, has_ragged_variant, false, same_points>, grid, dim3(kmc::BK_THREADS), stream, args)
                      : launch(kmc::gram_bf16_l2_kernel<LOAD_A, LOAD_B, false, false, same_points>, grid, dim3(kmc::BK_THREADS), stream, args);
    }
}

hipError_t launch_gram_bf16_l2_same_points(int load_a, int load_b, const kmc::BuildKernelArgs &args, dim3 grid, hipStream_t stream);

#if KMC_SAME_POINTS
hipError_t launch_gram_bf16_l2_same_points(int load_a, int load_b, const kmc::BuildKernelArgs &args, dim3 grid, hipStream_t stream)
{
#else
hipError_t launch_gram_bf16_l2(int load_a, int load_b, const kmc::BuildKernelArgs &args, dim3 grid, hipStream_t stream)
{
    // A result of one row of tiles is left to the repair launch all the same: the host takes no such result for a symmetric one, and only
    // the direct kernel gives both halves of it the same bits.
    if (args.same_points && args.tiles_m > 1) return launch_gram_bf16_l2_same_points(load_a, load_b, args, grid, stream);
#endif
    switch (load_a * 4 + load_b) {
    case 0: return launch_one<0, 0>(args, grid, stream);
    case 1: return launch_one<0, 1>(args, grid, stream);
    case 2: return launch_one<0, 2>(args, grid, stream);
    case 3: return launch_one<0, 3>(args, grid, stream);
    case 4: return launch_one<1, 0>(args, grid, stream);
    case 5: return launch_one<1, 1>(args, grid, stream);
    case 6: return launch_one<1, 2>(args, grid, stream);
    case 7: return launch_one<1, 3>(args, grid, stream);
    case 8: return launch_one<2, 0>(args, grid, stream);
    case 9: return launch_one<2, 1>(args, grid, stream);
    case 10: return launch_one<2, 2>(args, grid, stream);
    case 11: return launch_one<2, 3>(args, grid, stream);
    case 12: return launch_one<3, 0>(args, grid, stream);
    case 13: return launch_one<3, 1>(args, grid, stream);
    case 14: return launch_one<3, 2>(args, grid, stream);
    case 15: return launch_one<3, 3>(args, grid, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace kmc_host
