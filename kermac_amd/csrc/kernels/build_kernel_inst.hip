// One (inner operator, inner power) pair of the fused pairwise-reduction
// kernel, instantiated for all 16 (A loader, B loader) combinations.
// Compiled several times with different -DKMC_INNER_OP / -DKMC_INNER_POW.
#include <hip/hip_runtime.h>

#include <cstdlib>

#include "launch.hpp"
#include "build_kernel.hpp"
#include "build_kernel_scalar_b.hpp"
#include "build_kernel_short.hpp"
#include "build_kernel_small.hpp"
#include "../host/dispatch_rules.hpp"

#ifndef KMC_INNER_OP
#error "compile with -DKMC_INNER_OP=<0|1> -DKMC_INNER_POW=<0..4>"
#endif

#define KMC_CAT_(a, b, c, d) a##b##c##d
#define KMC_CAT(a, b, c, d) KMC_CAT_(a, b, c, d)
#define KMC_LAUNCHER_NAME KMC_CAT(launch_build_kernel_, KMC_INNER_OP, _, KMC_INNER_POW)

namespace kmc_host {

// Whether the call is one for build_kernel_scalar_b (its header says what the kernel assumes): enough tiles of
// 256 x 64 in every batch entry to fill the chip twice.  From a sweep against build_kernel / build_kernel_four_waves
// (their time / this kernel's, p = 1 and p = 2, K = 64 .. 4096): 2256 tiles (6000 x 6000) 1.02 .. 1.07 and 1.05 .. 1.10,
// 1876 (1000 x 30000) 1.01 .. 1.02 and 1.03 .. 1.07, 3776 (30000 x 2000) 1.04 .. 1.21, 55342 (30000 x 30000) 1.02 .. 1.05 and
// 1.05 .. 1.08; 1024 tiles (4096 x 4096) 0.96 .. 1.03, and batches of small entries lose: 8 x 2048 x 2048 0.95 .. 1.0,
// 64 x 512 x 512 0.91 .. 1.0 for p = 1.
// A panel against itself (the tiles of one triangle, each stored twice; ordinary kernel's time / this kernel's, p = 1 and
// p = 2, one box): 30000 x 1024, 27966 tiles, 1.02 and 1.05; 16384 x 512, 8320 tiles, 0.99 and 1.05; 8192 x 1024 0.90 and 1.02;
// 12000 x 128 1.03 and 1.05; 6000 x 512 level: taken from 16000 tiles on.
// KERMAC_AMD_SCALAR_B_MIN_TILES=n replaces the size rule by "at least n tiles over the batch, any k" (read on every
// call, so that a test can send small shapes to the kernel).
static bool scalar_b_applies(const kmc::BuildKernelArgs &args, int64_t *grid_width)
{
    if (args.k < 16 || args.k % kmc::BK_TILE_K != 0 || (args.n % kmc::SB_WAVE_N != 0 && !(args.panels & kmc::BK_PANELS_B_PADDED)) ||
        args.k_total != 0 || args.repair_only)
        return false;
    const int64_t tiles_m = (static_cast<int64_t>(args.m) + kmc::SB_TILE_M - 1) / kmc::SB_TILE_M;
    const int64_t tiles_n = (static_cast<int64_t>(args.n) + kmc::SB_TILE_N - 1) / kmc::SB_TILE_N;
    // a panel against itself: tile row r holds the tiles 0 .. 4 r + 3 that reach the diagonal or lie below it
    const int64_t tiles = args.symmetric ? 2 * (tiles_m - 1) * tiles_m + (4 * tiles_m < tiles_n ? 4 * tiles_m : tiles_n) : tiles_m * tiles_n;
    if (tiles > 0x7fffffff || (args.symmetric && args.m != args.n)) return false;
    *grid_width = tiles;
    if (args.panels & kmc::BK_PANELS_COPIED) return true;       // the host made the copies for this kernel
    const char *text = std::getenv("KERMAC_AMD_SCALAR_B_MIN_TILES");
    const int forced = text ? std::atoi(text) : 0;
    if (forced > 0) return tiles * args.l >= forced;
    return tiles >= (args.symmetric ? kmc_rules::DIRECT_SCALAR_B_MIN_TILES_SYMMETRIC : kmc_rules::DIRECT_SCALAR_B_MIN_TILES) &&
           args.k >= kmc_rules::DIRECT_SCALAR_B_MIN_K;
}

constexpr bool HAS_SCALAR_B = KMC_INNER_OP == kmc::OP_DIFF &&
                              (KMC_INNER_POW == kmc::POW_ABS || KMC_INNER_POW == kmc::POW_SQUARE || KMC_INNER_POW == kmc::POW_ABS_CUBE ||
                               KMC_INNER_POW == kmc::POW_ABS_FOURTH);

template <int LOAD_A, int LOAD_B>
static hipError_t launch_one(const kmc::BuildKernelArgs &args, dim3 grid, hipStream_t stream)
{
    // absolute differences, their squares, cubes and fourth powers, of large problems whose rows are contiguous on both
    // sides: b in scalar registers
    if constexpr (LOAD_A == kmc::LOAD_COL_VEC && LOAD_B == kmc::LOAD_COL_VEC && HAS_SCALAR_B) {
        int64_t grid_width = 0;
        if (scalar_b_applies(args, &grid_width)) {
            kmc::BuildKernelArgs copy = args;
            copy.sample = nullptr;          // an ordinary launch computes everything
            const float *a = args.a, *b = args.b;
            float *c = args.c;
            void *kernel_args[] = {&copy, &a, &b, &c};
            return hipLaunchKernel(reinterpret_cast<const void *>(kmc::build_kernel_scalar_b<KMC_INNER_OP, KMC_INNER_POW>),
                                   dim3(static_cast<unsigned>(grid_width), args.l), dim3(kmc::BK_THREADS), kernel_args, 0, stream);
        }
    }
    // contiguous rows on both sides, a contraction long enough for the walk to set the time, and an inner term
    // without transcendentals (whose loop needs more registers): the variant compiled for four waves per SIMD
    if constexpr (LOAD_A == kmc::LOAD_COL_VEC && LOAD_B == kmc::LOAD_COL_VEC && KMC_INNER_POW != kmc::POW_POW) {
        if (args.k >= kmc_rules::DIRECT_FOUR_WAVES_MIN_K && !args.repair_only)
            return launch(kmc::build_kernel_four_waves<KMC_INNER_OP, KMC_INNER_POW>, grid, dim3(kmc::BK_THREADS), stream, args);
    }
#if KMC_INNER_OP == 0 && KMC_INNER_POW == 2
    const int64_t tiles = static_cast<int64_t>(args.grid_width) * args.l;
    if (args.repair_only && args.repair_queue && tiles >= kmc::BK_REPAIR_MIN_TILES && tiles <= kmc::BK_REPAIR_MAX_TILES) {
        const dim3 scan(static_cast<unsigned>((tiles + kmc::BK_THREADS - 1) / kmc::BK_THREADS));
        const hipError_t status = launch(kmc::repair_scan<0>, scan, dim3(kmc::BK_THREADS), stream, args);
        if (status != hipSuccess) return status;
        return launch(kmc::build_kernel_repair<KMC_INNER_OP, KMC_INNER_POW, LOAD_A, LOAD_B>, dim3(kmc::BK_REPAIR_WORKGROUPS), dim3(kmc::BK_THREADS), stream, args);
    }
#endif
    return launch(kmc::build_kernel<KMC_INNER_OP, KMC_INNER_POW, LOAD_A, LOAD_B>, grid, dim3(kmc::BK_THREADS), stream, args);
}

#if KMC_INNER_OP == 0 && KMC_INNER_POW == 2
// For a matrix-core call for squared differences that took a sample (args.sample): when the direct kernel with b in
// scalar registers can take the operands as they are, launches it in front of the repair launch, where it computes
// everything if the sample left the call to the direct kernel and exits at once if not.  Without it the repair launch
// does that work on the ordinary kernel, 8 % slower.  *launched says whether the call qualified.
hipError_t launch_scalar_b_if_the_sample_leaves(int load_a, int load_b, const kmc::BuildKernelArgs &args, hipStream_t stream, bool *launched)
{
    *launched = false;
    int64_t grid_width = 0;
    if (!args.sample || load_a != kmc::LOAD_COL_VEC || load_b != kmc::LOAD_COL_VEC || !scalar_b_applies(args, &grid_width))
        return hipSuccess;
    kmc::BuildKernelArgs copy = args;
    const float *a = args.a, *b = args.b;
    float *c = args.c;
    void *kernel_args[] = {&copy, &a, &b, &c};
    *launched = true;
    return hipLaunchKernel(reinterpret_cast<const void *>(kmc::build_kernel_scalar_b<KMC_INNER_OP, KMC_INNER_POW>),
                           dim3(static_cast<unsigned>(grid_width), args.l), dim3(kmc::BK_THREADS), kernel_args, 0, stream);
}
#endif

// Results of few tiles, in tiles of 64 x 64 (build_kernel_small.hpp).  128 x 128 / 64 x 64 tiles, us, p = 1 and p = 1.3 at
// K = 400: 64 tiles 111 / 30 and 324 / 91; 121 tiles 113 / 45 and 326 / 166; 196 tiles 124 / 85 and 341 / 321; 256 tiles, one
// for every CU, 113 / 77 and 328 / 317; a set against itself of 16 x 16 tiles 142 / 79 and 343 / 318.  Beyond that most single problems
// still gain (324 tiles 148 / 109 and 633 / 468; 400 117 / 126 and 621 / 543) but batches hardly (32 x 500 x 500 162 / 149 and 639 / 618, at
// K = 64 32 / 32 and 113 / 111), and a set against itself, of which this kernel computes both halves, loses (22 x 22 tiles 146 / 144 and 345 / 619).
// Powers with a root or a transcendental function are bound by its issue, and there a fourth workgroup of 64 x 64 per CU brings little:
// up to 192 tiles, three per CU (208 x 128 x 128, p = 1.3, K = 64 58.8 / 58.2; 240 x 128 x 128 x 256 212 / 205; 1792 x 1792 x 256 213 / 205).
// KERMAC_AMD_DIRECT_SMALL_MAX_TILES=n replaces both limits (read on every call, so that a test can choose the kernel).
constexpr bool HAS_ROOT_OR_POWER = KMC_INNER_POW == kmc::POW_POW || KMC_INNER_POW == kmc::POW_SQRT || KMC_INNER_POW == kmc::POW_ABS_HALF ||
                                   KMC_INNER_POW == kmc::POW_ABS_THREE_HALVES;

static bool small_applies(int load_a, int load_b, const kmc::BuildKernelArgs &args)
{
    if (args.repair_only || args.k_total != 0 || args.panels != 0) return false;
    // never so by the size rules of the two kernels, but a test may send results of few tiles to the other one
    int64_t grid_width = 0;
    if (HAS_SCALAR_B && load_a == kmc::LOAD_COL_VEC && load_b == kmc::LOAD_COL_VEC && scalar_b_applies(args, &grid_width)) return false;
    const int64_t tiles = static_cast<int64_t>(args.tiles_m) * args.tiles_n * args.l;
    const char *limit = std::getenv("KERMAC_AMD_DIRECT_SMALL_MAX_TILES");
    return tiles <= (limit ? std::atoi(limit) : HAS_ROOT_OR_POWER ? kmc_rules::DIRECT_SMALL_MAX_TILES_ROOTS : kmc_rules::DIRECT_SMALL_MAX_TILES);
}

// Contractions of up to 24 terms, whose launches the stores of the result bound (build_kernel_short.hpp).  It pays a load of all k of
// its rows per workgroup and a term at 3.5 cycles an instruction, where the ordinary kernel pays whole slices of 16 k.  Ordinary / this kernel,
// us, p = 1, K = 6, 10, 16, 24: 10000 x 10000, rows 16-byte aligned 99 / 80, 103 / 92, 105 / 112, 153 / 150; 2 x 7000 x 7001, result not
// aligned 182 / 84, 184 / 99, 160 / 117, 231 / 154; 5000 x 5000 35 / 24, 37 / 28, 37 / 32, 49 / 45; 3000 x 2500 16.8 / 13.9, 16.7 / 15.8, 16.2 / 17.8,
// 21.6 / 24.4.  A set against itself, computed in full here, 2 x 10000, K = 6 and 12, Laplace kernel 226 / 196 and 223 / 233.
// Few columns, which share a load of all k, gain little or nothing above 8 terms: 10000 x 300 at K = 12 and 24 1.02 and 0.96 .. 1.00, 30000 x 40 0.8 and 0.5.
// Few rows leave tiles of 256 rows unused, in which its arithmetic runs all the same (short_rows_pay).
// KERMAC_AMD_DIRECT_SHORT_MAX_K=n replaces the rule by "at most n terms" (read on every call, so that a test can choose the kernel).
constexpr bool HAS_SHORT = !HAS_ROOT_OR_POWER;

// Columns this many apart start at the same place in a line of 32 floats
static int short_classes(const kmc::BuildKernelArgs &args)
{
    int classes = kmc::BKT_LINE;
    while (classes > 1 && args.c_ld % (2 * kmc::BKT_LINE / classes) == 0) classes /= 2;
    return classes;
}

// Whether the rows fill the tiles well enough.  `waste`: rows of this kernel's tiles of 256 per row of the ordinary kernel's of 128, on average over
// where columns start in a line.  Up to which it pays depends on what an unused row costs, terms and an exponential or logarithm, and on whether
// the ordinary kernel stores 16 bytes at a time; where it does not, it pays for each row that there is, which are few below 100.  Time of the ordinary
// kernel over this one's, distances / Gaussian kernels, results of 4e6 to 6e7 elements, K = 1 .. 4, 5 .. 8, 9 .. 12, and 17 .. 24 (unaligned also 16):
//   aligned, waste 1 (200, 256, 400, 700 rows)   1.04 .. 1.61 / 1.04 .. 1.63, 1.03 .. 1.58 / 1.05 .. 1.43, 1.02 .. 1.36 / 1.00 .. 1.20, 1.02 .. 1.31 / 0.99 .. 1.29
//   aligned, 1.25 (500 rows)                     1.20 .. 1.55 / 1.18 .. 1.33, 1.14 .. 1.37 / 1.00 .. 1.10, 0.98 .. 1.08 / 0.85 .. 0.93, 0.82 .. 0.96 / 0.76 .. 0.88
//   aligned, 1.33 (300, 384)                     1.08 .. 1.49 / 1.11 .. 1.36, 1.01 .. 1.31 / 1.00 .. 1.19, 0.91 .. 1.10 / 0.88 .. 1.07, 0.85 .. 0.98 / 0.84 .. 0.98
//   aligned, 2 (8, 64, 100, 128)                 0.96 .. 1.48 / 0.93 .. 1.11, 0.95 .. 1.13 / 0.77 .. 1.09, 0.69 .. 1.03 / 0.64 .. 0.99, 0.59 .. 0.98 / 0.56 .. 0.97
//   unaligned, 1 (129, 150 rows)                 1.20 .. 2.38 / 1.24 .. 1.97, 1.09 .. 1.98 / 1.16 .. 1.59, 1.07 .. 1.58 / 1.04 .. 1.34, 0.97 .. 1.36 / 1.03 .. 1.27
//   unaligned, 1.2, 1.33 (257, 333, 513)         1.20 .. 2.25 / 1.28 .. 1.98, 1.10 .. 2.07 / 1.21 .. 1.65, 1.09 .. 1.60 / 1.10 .. 1.37, 1.00 .. 1.41 / 0.88 .. 1.37
//   unaligned, 2 (127)                           1.23 .. 1.97 / 1.32 .. 1.45, 1.11 .. 1.75 / 1.16 .. 1.23, 1.06 .. 1.25 / 0.96 .. 1.03, 0.92 .. 1.06 / 0.81 .. 0.97
//   unaligned, 2 (10, 17, 33)                    1.09 .. 1.42 / 0.90 .. 1.04, 0.87 .. 1.07 / 0.76 .. 0.89, 0.68 .. 0.86 / 0.64 .. 0.74, 0.57 .. 0.80 / 0.56 .. 0.72
static bool short_rows_pay(const kmc::BuildKernelArgs &args)
{
    const int classes = short_classes(args);
    int64_t tiles = 0;
    for (int column = 0; column < classes; column++) {
        const uint64_t start = reinterpret_cast<uintptr_t>(args.c) / 4 + static_cast<uint64_t>(column) * static_cast<uint64_t>(args.c_ld);
        tiles += (static_cast<int64_t>(args.m) + static_cast<int64_t>(start % kmc::BKT_LINE) + kmc::BKT_TILE_M - 1) / kmc::BKT_TILE_M;
    }
    const double waste = static_cast<double>(tiles) * kmc::BKT_TILE_M / (static_cast<double>(classes) * args.tiles_m * kmc::BK_TILE_M);
    const bool heavy = args.kernel_type != kmc::KERNEL_NONE || args.outer_power == kmc::POW_POW || KMC_INNER_POW == kmc::POW_ABS_CUBE ||
                       KMC_INNER_POW == kmc::POW_ABS_FOURTH;
    const int k = args.k;
    if (!heavy && k <= 4) return true;
    if (args.c_vec) return waste <= (heavy ? k <= 8 ? 1.34 : 8.0 / 7 : k <= 8 ? 2.0 : k <= kmc::BK_TILE_K ? 1.25 : 8.0 / 7);
    if (k <= (heavy ? 8 : kmc::BK_TILE_K) && args.m >= 100) return true;
    return waste <= (heavy && k > 12 ? 1.25 : 1.34);
}

static bool short_applies(int load_a, int load_b, const kmc::BuildKernelArgs &args)
{
    if (!HAS_SHORT || args.repair_only || args.k_total != 0 || args.panels != 0 || args.k < 1 || args.k > kmc_rules::DIRECT_SHORT_MAX_K ||
        args.l > 65535 || args.n > (1 << 22))
        return false;
    const char *limit = std::getenv("KERMAC_AMD_DIRECT_SHORT_MAX_K");
    if (limit) return args.k <= std::atoi(limit);
    // a test that chooses between the other kernels
    int64_t grid_width = 0;
    if (std::getenv("KERMAC_AMD_DIRECT_SMALL_MAX_TILES") ||
        (HAS_SCALAR_B && load_a == kmc::LOAD_COL_VEC && load_b == kmc::LOAD_COL_VEC && scalar_b_applies(args, &grid_width)))
        return false;
    const int64_t tiles = static_cast<int64_t>(args.tiles_m) * args.tiles_n * args.l;
    if (tiles <= kmc_rules::DIRECT_SMALL_MAX_TILES || !short_rows_pay(args)) return false;          // the first for build_kernel_small
    if (args.k <= kmc_rules::DIRECT_SHORT_ANY_MAX_K) return true;
    if (args.symmetric) return false;
    if (args.n < kmc_rules::DIRECT_SHORT_MIN_COLUMNS) return false;
    if (args.k <= 12) return true;
    if (args.k <= kmc::BK_TILE_K) return !args.c_vec;
    return tiles >= kmc_rules::DIRECT_SHORT_LONG_MIN_TILES;
}

template <int DEPTH>
static hipError_t launch_short(int load_a, int load_b, const kmc::BuildKernelArgs &args, hipStream_t stream)
{
    const int classes = short_classes(args);
    // floats between the start of a line and a column, at most
    uint64_t shift = args.l > 1 && args.c_bs % kmc::BKT_LINE ? kmc::BKT_LINE - 1 : 0;
    for (int column = 0; column < classes; column++) {
        const uint64_t start = reinterpret_cast<uintptr_t>(args.c) / 4 + static_cast<uint64_t>(column) * static_cast<uint64_t>(args.c_ld);
        shift = start % kmc::BKT_LINE > shift ? start % kmc::BKT_LINE : shift;
    }
    const int64_t m_tiles = (static_cast<int64_t>(args.m) + shift + kmc::BKT_TILE_M - 1) / kmc::BKT_TILE_M;
    // rounds of 16 columns per workgroup: as many as the loads of a are worth, as few as fill the chip
    int rounds = kmc::BKT_MAX_ROUNDS;
    while (rounds > 1 && m_tiles * (args.n / (rounds * kmc::BKT_COLUMNS) + 1) * args.l < 1024) rounds /= 2;
    const int64_t per_group = static_cast<int64_t>(rounds) * kmc::BKT_COLUMNS * classes;
    const int64_t groups = (args.n + per_group - 1) / per_group * classes;
    kmc::BuildKernelArgs copy = args;
    void *kernel_args[] = {&copy, &load_a, &load_b, &rounds, const_cast<int *>(&classes)};
    return hipLaunchKernel(reinterpret_cast<const void *>(kmc::build_kernel_short<KMC_INNER_OP, KMC_INNER_POW, DEPTH>),
                           dim3(static_cast<unsigned>(m_tiles), static_cast<unsigned>(groups), args.l), dim3(kmc::BK_THREADS), kernel_args, 0, stream);
}

hipError_t KMC_LAUNCHER_NAME(int load_a, int load_b, const kmc::BuildKernelArgs &args, dim3 grid, hipStream_t stream)
{
    if constexpr (HAS_SHORT)
        if (short_applies(load_a, load_b, args)) {
            switch ((args.k + 3) / 4) {
            case 1: return launch_short<4>(load_a, load_b, args, stream);
            case 2: return launch_short<8>(load_a, load_b, args, stream);
            case 3: return launch_short<12>(load_a, load_b, args, stream);
            case 4: return launch_short<16>(load_a, load_b, args, stream);
            case 5: return launch_short<20>(load_a, load_b, args, stream);
            default: return launch_short<24>(load_a, load_b, args, stream);
            }
        }
    if (small_applies(load_a, load_b, args)) {
        const int across = (args.m + kmc::BKS_TILE - 1) / kmc::BKS_TILE, down = (args.n + kmc::BKS_TILE - 1) / kmc::BKS_TILE;
        kmc::BuildKernelArgs copy = args;
        void *kernel_args[] = {&copy, &load_a, &load_b, const_cast<int *>(&down)};
        return hipLaunchKernel(reinterpret_cast<const void *>(kmc::build_kernel_small<KMC_INNER_OP, KMC_INNER_POW>),
                               dim3(static_cast<unsigned>(across) * down, args.l), dim3(kmc::BKS_THREADS), kernel_args, 0, stream);
    }
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
