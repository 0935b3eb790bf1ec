// Matrix-core path for squared differences, large problems: the cross term of
//
//   sum_k (b[n,k] - a[m,k])^2  =  |a_m|^2 + |b_n|^2 - 2 * sum_k a[m,k] * b[n,k]
//
// on the fp16 matrix instruction (v_mfma_f32_16x16x32_f16, the rate of the bf16 one), from two
// fp16 pieces per fp32 value and three piece products, in three launches with a workspace
// between them:
//
//   gram_row_stats   per row of an operand: sum of squares (the norms of the expansion) and
//                    largest magnitude, both after the centre has been subtracted.
//                    (As a rule by one launch, gram_rows_once or gram_columns_once.)
//   gram_f16_split   scales every row by a power of two that puts its largest magnitude into
//                    [2^14, 2^15), splits every scaled value x into h1 = fp16(x), h2 = fp16(x - h1)
//                    and writes the pieces in the order the matrix instruction reads them.
//   gram_f16_wide    one workgroup of 4 waves per 256 x 128 tile of the result (128 x 128 where those are few): copies
//                    pieces from the workspace into LDS and multiplies; a1 b2 + a1 b1 + a2 b1, fp32 accumulators.
//
// Accuracy.  x - h1 is exact in fp32 and h2 keeps 11 of its bits: |x - h1 - h2| <= 2^-22 |x|, or
// 2^-25 where h2 is subnormal, which is 2^-39 of the row's largest magnitude.  The dropped product
// a2 b2 is below 2^-22 |a_k b_k|.  The error of a dot product from the pieces is therefore below
// 3 * 2^-22 sum_k |a_k b_k| + k 2^-38 max|a| max|b| <= (3.6e-7 + k 2^-39) (|a|^2 + |b|^2), in practice far less since the roundings
// do not line up, beside the rounding of the fp32 accumulation that every matrix-core path has
// (products of fp16 pieces are exact in fp32).  The scale per row is what makes the bound relative
// to that row's norm, which is what the trust rule of gram_kernel.hpp needs: with one scale per
// operand a row of small values next to a row of large ones would sit in fp16's subnormals.
// Scales are powers of two, so scaling and unscaling round nothing.  Rows that hold an infinity or
// a NaN produce results that are not numbers, which are distrusted and recomputed like any other.
//
// Why two fp16 pieces and not the three bf16 pieces of gram_bf16_kernel.hpp: the board is power-limited under this kernel
// (at 16384 x 16384 x 4096 it multiplies at 1785 TFLOP/s on operands of zeros and at 1352 on normal ones, plain fp16
// library products of the same size at 1718 and 1452), so time follows energy, and three products cost half of six.
// Why a workspace: a value is split once instead of once per tile that needs it (in the one-step kernel the split
// takes as long as the matrix instructions it hides behind), and the layout of an operand in memory
// only matters to the split.
//
// What the shape of the product kernel is worth, whole call at M = N = 30000, K = 1024, and sums of products at
// 16384 x 16384 x 256: one workgroup of 8 waves per 256 x 256 tile and CU on v_mfma_f32_32x32x16_f16, with nothing beside
// its prologue and stores, 5.83 and 0.686 ms; two workgroups of 256 x 128 on v_mfma_f32_16x16x32_f16 4.87 and 0.513 ms.
//
// Workspace of one operand and batch entry, in 16-byte chunks of 8 fp16 (one row, one half of a
// 16-deep K slice, one piece):  chunk[slice][piece][half][row 0 .. rows_pad),  rows_pad a multiple
// of 256; rows that do not exist and k beyond K hold zeros, so the product kernel has no edge
// handling in its walk.  K is padded to whole steps of 32.
// Statistics: partial[range][row] for the sums of squares and for the magnitudes, one partial per
// range of K slices that a workgroup walks, combined in the order of the ranges.
// The reference has no such path (include/build_a_kernel.cuh:339-370 is SIMT only).
#pragma once

#include "gram_bf16_kernel.hpp"
#include "gram_probe.hpp"

namespace kmc {

typedef _Float16 gram_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 gram_half2 __attribute__((ext_vector_type(2)));

constexpr int GW_TILE = 256;                                  // rows of an operand are padded to this
constexpr int GW_PIECES = 2;
constexpr int GW_SEGMENTS = 2 * GW_PIECES;                    // (piece, half) pairs of one slice
constexpr int GW_BAND_N = 64;                                 // tile order: n tiles per band
constexpr int GW_ROW_THREADS = 256;
constexpr int GW_SCALE_EXPONENT = 14;                         // a row's largest magnitude goes to [2^14, 2^15)

// One operand, for gram_row_stats and gram_f16_split.
struct GramRowsArgs {
    const float *x; i64 ld, bs;
    int rows, k, row_major, vec;          // vec: 128-bit loads along k are allowed (row-major only)
    const float *centre; i64 centre_bs;   // as BuildKernelArgs::centre, or null
    int centre_pairs;                     // as GramProbeArgs
    gram_chunk *pieces; i64 pieces_bs;    // per batch entry, in chunks
    float *squares; float *magnitudes;    // [batch][range][rows_pad]
    float *unscale;                       // [batch][rows_pad]: 1 / the row's scale
    i64 stats_bs, unscale_bs;
    int rows_pad, slices, slices_per_range, ranges;
    int magnitude_ranges;                 // partial magnitudes per row: `ranges`, or what another launch has left
    int zero_slices;                      // slices behind the last that gram_f16_split fills with zeros (for
                                          // walks in steps of more than one slice)
};

struct GramWideArgs {
    BuildKernelArgs kernel;               // extents, result, epilogue, trust; tiles_* are not used
    const gram_chunk *pieces_a, *pieces_b;
    i64 pieces_a_bs, pieces_b_bs;
    const float *squares_a, *squares_b;
    i64 stats_a_bs, stats_b_bs;
    const float *unscale_a, *unscale_b;
    i64 unscale_a_bs, unscale_b_bs;
    int rows_pad_a, rows_pad_b, slices, ranges_a, ranges_b;
    int wide_tiles_m, wide_tiles_n, wide_tiles_n_padded;
    int entry_per_xcd;                    // wide_tile_of_workgroup
    // GW_EPILOGUE_GRADIENT_L2 only: row r of b stands for (o, n) = (r / gradient_n, r % gradient_n) and
    // the result is (d[n][m] - shift[n]) * g[m][o] - a[m] . b[r]
    const float *gradient_d; i64 gradient_d_ld, gradient_d_bs;
    const float *gradient_g; i64 gradient_g_ld, gradient_g_bs;
    const float *gradient_shift; i64 gradient_shift_bs;
    int gradient_n;
    // COLUMNS > 0 only: the matrix times coefficients, tile by tile (gram_f16_wide)
    const float *coef; i64 coef_ld, coef_bs;      // [n][o], o contiguous
    int outputs;
    float *products; i64 products_ld, products_bs, products_tile;      // [tile of 128 n][batch][m][o], products_ld a multiple of 4
    int *stamps; int stamps_m, stamps_n;          // [batch][tile of 128 m][tile of 128 n]: 1 where the repair launch recomputes the tile's product
};

constexpr int GW_MAX_RANGES = 9;      // ranges of K per row: ceil(slices / 8) up to 71 slices, 8 beyond

constexpr int GW_EPILOGUE_DISTANCE = 0;
constexpr int GW_EPILOGUE_GRADIENT_L2 = 1;
constexpr int GW_EPILOGUE_DOT = 2;
// added to GW_EPILOGUE_DISTANCE or GW_EPILOGUE_DOT: contracted with up to 16 or 32 columns of coefficients instead of stored
constexpr int GW_CONTRACT_16 = 4, GW_CONTRACT_32 = 8;

// The 16 values of row `row` in slice `slice`, centre subtracted; zeros where the row or k does not exist.
__device__ __forceinline__ void gram_load_row_slice(const GramRowsArgs &args, const float *x, const float *centre, int row,
                                                    int slice, float (&v)[BK_TILE_K])
{
    const bool live = row < args.rows;
    const int k0 = slice * BK_TILE_K;
    if (args.row_major) {
        const float *src = x + (i64)row * args.ld + k0;
        if (live && args.vec && k0 + BK_TILE_K <= args.k) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 f = reinterpret_cast<const float4 *>(src)[q];
                v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < BK_TILE_K; e++) v[e] = (live && k0 + e < args.k) ? src[e] : 0.0f;
        }
    } else {
#pragma unroll
        for (int e = 0; e < BK_TILE_K; e++) v[e] = (live && k0 + e < args.k) ? x[(i64)(k0 + e) * args.ld + row] : 0.0f;
    }
    if (centre) {
        // beyond K the centre is padded with zeros, like the values
#pragma unroll
        for (int e = 0; e < BK_TILE_K; e++) v[e] = live ? v[e] - centre[k0 + e] : 0.0f;
    }
}

__device__ __forceinline__ const float *gram_rows_centre(const GramRowsArgs &args, int batch)
{
    if (!args.centre) return nullptr;
    const float *centre = args.centre + batch * args.centre_bs;
    if (args.centre_pairs) {
        CentreSums sums;
        sums.load(centre, args.k, args.centre_pairs);
        return sums.needless() ? nullptr : centre;
    }
    const int padded = (args.k + GRAM_CENTRE_PAD - 1) / GRAM_CENTRE_PAD * GRAM_CENTRE_PAD;
    return centre[padded] != 0.0f ? centre : nullptr;      // the flag behind the vector: see centre_to_subtract
}

// One thread per row, one workgroup per 256 rows and range of slices.  (The row kernels are
// templates only so that every translation unit that includes this header may hold them.)
__device__ __forceinline__ void gram_row_stats_of(const GramRowsArgs &args, int block)
{
    const int row = block * GW_ROW_THREADS + threadIdx.x;
    const int range = blockIdx.y, batch = blockIdx.z;
    const float *x = args.x + batch * args.bs;
    const float *centre = gram_rows_centre(args, batch);
    const int first = range * args.slices_per_range;
    const int last = min(first + args.slices_per_range, args.slices);
    float square = 0.0f, magnitude = 0.0f;
    bool not_a_number = false;
    for (int slice = first; slice < last; slice++) {
        float v[BK_TILE_K];
        gram_load_row_slice(args, x, centre, row, slice, v);
        float of_slice = 0.0f;                              // its own sum first: a longer one rounds more
#pragma unroll
        for (int e = 0; e < BK_TILE_K; e++) {
            of_slice += v[e] * v[e];
            magnitude = fmaxf(magnitude, fabsf(v[e]));      // skips NaNs
            not_a_number |= v[e] != v[e];
        }
        square += of_slice;
    }
    const i64 at = batch * args.stats_bs + (i64)range * args.rows_pad + row;
    args.squares[at] = square;
    args.magnitudes[at] = not_a_number ? __builtin_nanf("") : magnitude;
}

template <int UNUSED = 0>
__global__ __launch_bounds__(GW_ROW_THREADS) void gram_row_stats(const GramRowsArgs args)
{
    gram_row_stats_of(args, blockIdx.x);
}

// scale = 2^(GW_SCALE_EXPONENT - floor(log2 magnitude)), from the exponent field.  Rows of
// zeros or of values below 2^-111 take the largest scale used, 2^125 (the scale and its
// inverse must both be normal numbers); a row with a NaN or an infinity takes the smallest:
// its products are not numbers whatever the scale.
__device__ __forceinline__ int gram_scale_exponent(float magnitude)
{
    return max((int)(__float_as_uint(magnitude) >> 23) & 0xff, 16);
}
__device__ __forceinline__ float gram_scale(int exponent_field)
{
    return __uint_as_float((unsigned)(127 + GW_SCALE_EXPONENT + 127 - exponent_field) << 23);
}
__device__ __forceinline__ float gram_unscale(int exponent_field)
{
    return __uint_as_float((unsigned)(exponent_field - GW_SCALE_EXPONENT) << 23);
}

// Two scaled values into their two pieces, packed.
__device__ __forceinline__ void gram_split_pair(float x0, float x1, unsigned &first, unsigned &second)
{
    const gram_half2 h1 = __builtin_convertvector(gram_float2{x0, x1}, gram_half2);
    const gram_float2 back = __builtin_convertvector(h1, gram_float2);
    const gram_half2 h2 = __builtin_convertvector(gram_float2{x0 - back.x, x1 - back.y}, gram_half2);
    first = __builtin_bit_cast(unsigned, h1);
    second = __builtin_bit_cast(unsigned, h2);
}

__device__ __forceinline__ void gram_f16_split_of(const GramRowsArgs &args, int block)
{
    const int row = block * GW_ROW_THREADS + threadIdx.x;
    const int range = blockIdx.y, batch = blockIdx.z;
    const float *x = args.x + batch * args.bs;
    const float *centre = gram_rows_centre(args, batch);

    float magnitude = 0.0f;
    for (int r = 0; r < args.magnitude_ranges; r++) {
        const float part = args.magnitudes[batch * args.stats_bs + (i64)r * args.rows_pad + row];
        magnitude = part != part ? part : fmaxf(magnitude, part);
        if (part != part) break;
    }
    const int exponent_field = gram_scale_exponent(magnitude);
    const float scale = gram_scale(exponent_field);
    if (range == 0) args.unscale[batch * args.unscale_bs + row] = gram_unscale(exponent_field);

    gram_chunk *pieces = args.pieces + batch * args.pieces_bs;
    const int first = range * args.slices_per_range;
    const int last = min(first + args.slices_per_range, args.slices);
    for (int slice = first; slice < last; slice++) {
        float v[BK_TILE_K];
        gram_load_row_slice(args, x, centre, row, slice, v);
        unsigned int piece[GW_PIECES][8];
#pragma unroll
        for (int q = 0; q < 8; q++) gram_split_pair(v[2 * q] * scale, v[2 * q + 1] * scale, piece[0][q], piece[1][q]);
        gram_chunk *dst = pieces + (i64)slice * GW_SEGMENTS * args.rows_pad + row;
#pragma unroll
        for (int p = 0; p < GW_PIECES; p++)
#pragma unroll
            for (int half = 0; half < 2; half++)
                dst[(i64)(2 * p + half) * args.rows_pad] =
                    gram_chunk{piece[p][4 * half], piece[p][4 * half + 1], piece[p][4 * half + 2], piece[p][4 * half + 3]};
    }
    if (range == args.ranges - 1) {
        for (int slice = args.slices; slice < args.slices + args.zero_slices; slice++) {
            gram_chunk *dst = pieces + (i64)slice * GW_SEGMENTS * args.rows_pad + row;
#pragma unroll
            for (int segment = 0; segment < GW_SEGMENTS; segment++) dst[(i64)segment * args.rows_pad] = gram_chunk{0u, 0u, 0u, 0u};
        }
    }
}

template <int UNUSED = 0>
__global__ __launch_bounds__(GW_ROW_THREADS) void gram_f16_split(const GramRowsArgs args)
{
    gram_f16_split_of(args, blockIdx.x);
}

// Both operands of a call in one launch each (at a few thousand rows a launch of these kernels is its own latency, and
// two of them one after the other cost twice that): the first `first_blocks` workgroups along x take the first operand.
// Both have the same ranges of slices; an operand with fewer batch entries than the grid leaves the surplus idle.
struct GramRowsPair {
    GramRowsArgs first, second;
    int first_blocks, first_batches, second_batches;
};

template <int UNUSED = 0>
__global__ __launch_bounds__(GW_ROW_THREADS) void gram_row_stats_pair(const GramRowsPair pair)
{
    if ((int)blockIdx.x < pair.first_blocks) {
        if ((int)blockIdx.z < pair.first_batches) gram_row_stats_of(pair.first, blockIdx.x);
    } else if ((int)blockIdx.z < pair.second_batches) {
        gram_row_stats_of(pair.second, blockIdx.x - pair.first_blocks);
    }
}

template <int UNUSED = 0>
__global__ __launch_bounds__(GW_ROW_THREADS) void gram_f16_split_pair(const GramRowsPair pair)
{
    if ((int)blockIdx.x < pair.first_blocks) {
        if ((int)blockIdx.z < pair.first_batches) gram_f16_split_of(pair.first, blockIdx.x);
    } else if ((int)blockIdx.z < pair.second_batches) {
        gram_f16_split_of(pair.second, blockIdx.x - pair.first_blocks);
    }
}

// Both steps in one pass for operands with k contiguous and up to 2048 of them: a workgroup holds 16 whole rows in its
// registers, so the values are read once and the scale is known before the pieces are written.  Wave w takes the slices w,
// w + 4, ..; four lanes share a slice of a row, 4 k each (a load instruction reads 64 consecutive bytes of 16 rows, the four
// waves together 256); two neighbours exchange halves so that one stores the chunk of the first piece and the other that
// of the second, and a store instruction writes four runs of 256 bytes.  (A wave on four rows of 64 lanes' k wrote runs of 64
// bytes.)  Bound by its bytes, 4 read and 4 written per value.  The squares are one sum
// per row.  In front of the row workgroups in the grid stand those of the sample (gram_probe.hpp), which needs
// nothing of theirs: at a few thousand rows every launch of this prelude is its own latency.  Statistics, split and sample in three launches, and now:
// 1000 + 60000 rows of K = 784 53 + 89 + 12 -> 110 us, 10000 rows 12 + 13 + 10 -> 27 us, 2 x 2000 rows 10 + 12 + 11 -> 18 us.
constexpr int GRO_ROWS = 16;                                  // per workgroup
constexpr int GRO_WAVES = GW_ROW_THREADS / 64;
constexpr int GRO_HELD_K = 1024;                              // k of a row in the registers: twice as many in the widest gram_rows_once
constexpr int GRO_MAX_K = 8192;                               // ... and in all

struct GramRowsOnceArgs {
    GramRowsArgs first, second;
    int samples, first_blocks;                 // workgroups along x: those of the sample (in the first batch), then of the first operand
    int first_batches, second_batches;
    GramProbeArgs probe;
};

// The values of a lane of a row workgroup: 4 k of every 64 from k_base on, of row `row`, with the centre subtracted; zeros where the row or k does not exist.
template <int GROUPS>
struct RowValues {
    float v[GROUPS][4];

    __device__ __forceinline__ void load(const GramRowsArgs &args, const float *src, int k0)
    {
        // Loads of what does not exist go to the last element that does and are dropped: with a branch per load they would be
        // waited for one by one (198 instead of 110 us for 61000 rows).
        if (args.vec && args.k % 4 == 0) {
#pragma unroll
            for (int g = 0; g < GROUPS; g++) {
                const float4 f = *reinterpret_cast<const float4 *>(src + min(64 * g + k0, args.k - 4));
                v[g][0] = f.x; v[g][1] = f.y; v[g][2] = f.z; v[g][3] = f.w;
            }
        } else {
#pragma unroll
            for (int g = 0; g < GROUPS; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) v[g][e] = src[min(64 * g + k0 + e, args.k - 1)];
        }
    }
    __device__ __forceinline__ void centre(const GramRowsArgs &args, const float *centre, int k0, bool subtract, bool live)
    {
        if (subtract) {
            // padded with zeros to whole groups of 64 k
            const bool aligned = (reinterpret_cast<unsigned long>(centre) & 15) == 0;
            const int last = (args.k + 63) / 64 * 64 - 4;
            if (aligned) {
#pragma unroll
                for (int g = 0; g < GROUPS; g++) {
                    const float4 f = *reinterpret_cast<const float4 *>(centre + min(64 * g + k0, last));
                    v[g][0] -= f.x; v[g][1] -= f.y; v[g][2] -= f.z; v[g][3] -= f.w;
                }
            } else {
#pragma unroll
                for (int g = 0; g < GROUPS; g++)
#pragma unroll
                    for (int e = 0; e < 4; e++) v[g][e] -= centre[min(64 * g + k0, last) + e];
            }
        }
#pragma unroll
        for (int g = 0; g < GROUPS; g++)
#pragma unroll
            for (int e = 0; e < 4; e++) v[g][e] = live && 64 * g + k0 + e < args.k ? v[g][e] : 0.0f;
    }
    __device__ __forceinline__ void statistics(float &square, float &magnitude) const
    {
        bool not_a_number = false;
        float of_chunk = 0.0f;
#pragma unroll
        for (int g = 0; g < GROUPS; g++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                of_chunk += v[g][e] * v[g][e];
                magnitude = fmaxf(magnitude, fabsf(v[g][e]));      // skips NaNs
                not_a_number |= v[g][e] != v[g][e];
            }
        square += of_chunk;
        if (not_a_number) magnitude = __builtin_inff();            // takes the same scale as a NaN
    }
    // the chunks of slices slice0, slice0 + 4, ..; two neighbours exchange halves
    __device__ __forceinline__ void split(const GramRowsArgs &args, gram_chunk *pieces, int row, int slice0, int quarter, float scale) const
    {
        const int all_slices = args.slices + args.zero_slices;
        const bool second = quarter & 1;
        const int segment = 2 * (second ? 1 : 0) + (quarter >> 1);
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            const int slice = 4 * g + slice0;
            unsigned h1[2], h2[2];
#pragma unroll
            for (int q = 0; q < 2; q++) gram_split_pair(v[g][2 * q] * scale, v[g][2 * q + 1] * scale, h1[q], h2[q]);
            // the even lane holds the first half of both pieces' chunks, the odd one the second half
            const unsigned give0 = second ? h1[0] : h2[0], give1 = second ? h1[1] : h2[1];
            const unsigned got0 = (unsigned)__shfl_xor((int)give0, 1), got1 = (unsigned)__shfl_xor((int)give1, 1);
            const gram_chunk chunk = second ? gram_chunk{got0, got1, h2[0], h2[1]} : gram_chunk{h1[0], h1[1], got0, got1};
            if (slice < all_slices) pieces[((i64)slice * GW_SEGMENTS + segment) * args.rows_pad + row] = chunk;
        }
    }
};

// LONG: rows of more than 64 GROUPS k, in chunks of that many: read for the statistics, and once more, as a rule from a cache, for the pieces.
template <int GROUPS, bool LONG>
__device__ __forceinline__ void gram_rows_once_of(const GramRowsArgs &args, int block)
{
    __shared__ float squares[GRO_WAVES][GRO_ROWS], magnitudes[GRO_WAVES][GRO_ROWS];
    const int wave = threadIdx.x >> 6, r = (threadIdx.x & 63) >> 2, quarter = threadIdx.x & 3;
    const int row = block * GRO_ROWS + r, batch = blockIdx.z;
    const bool live = row < args.rows;
    const float *src = args.x + batch * args.bs + (i64)(live ? row : args.rows - 1) * args.ld;
    const float *centre = args.centre ? args.centre + batch * args.centre_bs : nullptr;
    CentreSums sums;
    if (centre && args.centre_pairs) sums.load(centre, args.k, args.centre_pairs);
    const int k0 = BK_TILE_K * wave + 4 * quarter;             // and every 64 behind it
    constexpr int CHUNK = 64 * GROUPS;
    RowValues<GROUPS> values;
    values.load(args, src, k0);
    const bool subtract = centre && args.centre_pairs ? !sums.needless() : gram_rows_centre(args, batch) != nullptr;
    values.centre(args, centre, k0, subtract, live);
    float square = 0.0f, magnitude = 0.0f;
    values.statistics(square, magnitude);
    if constexpr (LONG)
        for (int at = CHUNK; at < args.k; at += CHUNK) {
            values.load(args, src, at + k0);
            values.centre(args, centre, at + k0, subtract, live);
            values.statistics(square, magnitude);
        }
#pragma unroll
    for (int offset = 2; offset > 0; offset >>= 1) {
        square += __shfl_xor(square, offset);
        magnitude = fmaxf(magnitude, __shfl_xor(magnitude, offset));
    }
    if (quarter == 0) {
        squares[wave][r] = square;
        magnitudes[wave][r] = magnitude;
    }
    __syncthreads();
    magnitude = fmaxf(fmaxf(magnitudes[0][r], magnitudes[1][r]), fmaxf(magnitudes[2][r], magnitudes[3][r]));
    const int exponent_field = gram_scale_exponent(magnitude);
    const float scale = gram_scale(exponent_field);
    if (wave == 0 && quarter == 0) {
        args.squares[batch * args.stats_bs + row] = (squares[0][r] + squares[1][r]) + (squares[2][r] + squares[3][r]);
        args.unscale[batch * args.unscale_bs + row] = gram_unscale(exponent_field);
    }
    gram_chunk *pieces = args.pieces + batch * args.pieces_bs;
    if constexpr (LONG) {
        // the last chunk is still here: backwards, so that the next one is the one read last
        const int last = (args.k - 1) / CHUNK * CHUNK;
        values.split(args, pieces, row, last / BK_TILE_K + wave, quarter, scale);
        for (int at = last - CHUNK; at >= 0; at -= CHUNK) {
            values.load(args, src, at + k0);
            values.centre(args, centre, at + k0, subtract, live);
            values.split(args, pieces, row, at / BK_TILE_K + wave, quarter, scale);
        }
    } else {
        values.split(args, pieces, row, wave, quarter, scale);
    }
}

template <int GROUPS, bool LONG = false>
__global__ __launch_bounds__(GW_ROW_THREADS, 2) void gram_rows_once(const GramRowsOnceArgs args)
{
    static_assert(GW_ROW_THREADS == GP_THREADS, "both parts of the launch");
    const int block = (int)blockIdx.x - args.samples;
    if (block < 0) {
        if (blockIdx.z == 0) gram_probe_tile(args.probe, blockIdx.x);
        return;
    }
    const bool first = block < args.first_blocks;
    if ((int)blockIdx.z < (first ? args.first_batches : args.second_batches))
        gram_rows_once_of<GROUPS, LONG>(first ? args.first : args.second, first ? block : block - args.first_blocks);
}

// The same for operands with the rows contiguous: a workgroup holds 32 whole rows, a line of memory per k.  Wave w takes the slices w, w + 4, ..; a half
// wave has one half of each, so that a lane makes whole chunks.  In place of gram_row_stats_pair, gram_f16_split_pair and the sample in three launches, which read
// the operands twice: 30000 + 30000 rows of K = 1024 178 -> 121 us and the call 4911 -> 4753, calls of 2000 x 2000 x 784 64 -> 43.5, 4000 x 4000 x 256
// 77 -> 51, 2 x 1503 x 1503 x 128 57 -> 34.5, 8000 x 8000 x 512 235 -> 212, 10000 x 10000 x 128 188 -> 155 (with the centre in one launch).
constexpr int GCO_ROWS = 32;                                  // per workgroup

// The values of a lane of such a workgroup: one half of the slices slice0, slice0 + 4, .. of a row.
template <int GROUPS>
struct ColumnValues {
    float v[GROUPS][8];

    __device__ __forceinline__ void load(const GramRowsArgs &args, const float *src, int slice0, int half)
    {
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            const int slice = slice0 + GRO_WAVES * g, k0 = BK_TILE_K * slice + 8 * half;
            if (BK_TILE_K * (slice + 1) <= args.k) {              // uniform: a wave has whole slices
                const float *from = src + (i64)k0 * args.ld;
#pragma unroll
                for (int e = 0; e < 8; e++) v[g][e] = from[e * args.ld];
            } else {
                // loads of what does not exist go to the last k that does, as in RowValues
#pragma unroll
                for (int e = 0; e < 8; e++) v[g][e] = src[(i64)min(k0 + e, args.k - 1) * args.ld];
            }
        }
    }
    __device__ __forceinline__ void centre(const GramRowsArgs &args, const float *centre, int slice0, int half, bool subtract, bool live)
    {
        if (subtract) {
            // padded with zeros to whole groups of 64 k, and 16-byte aligned
            const int last = (args.k + GRAM_CENTRE_PAD - 1) / GRAM_CENTRE_PAD * GRAM_CENTRE_PAD - 8;
#pragma unroll
            for (int g = 0; g < GROUPS; g++) {
                const float4 *of = reinterpret_cast<const float4 *>(centre + min(BK_TILE_K * (slice0 + GRO_WAVES * g) + 8 * half, last));
                const float4 lo = of[0], hi = of[1];
                v[g][0] -= lo.x; v[g][1] -= lo.y; v[g][2] -= lo.z; v[g][3] -= lo.w;
                v[g][4] -= hi.x; v[g][5] -= hi.y; v[g][6] -= hi.z; v[g][7] -= hi.w;
            }
        }
#pragma unroll
        for (int g = 0; g < GROUPS; g++)
#pragma unroll
            for (int e = 0; e < 8; e++) v[g][e] = live && BK_TILE_K * (slice0 + GRO_WAVES * g) + 8 * half + e < args.k ? v[g][e] : 0.0f;
    }
    __device__ __forceinline__ void statistics(float &square, float &magnitude) const
    {
        bool not_a_number = false;
        float of_chunk = 0.0f;
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            float of_group = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                of_group += v[g][e] * v[g][e];
                magnitude = fmaxf(magnitude, fabsf(v[g][e]));      // skips NaNs
                not_a_number |= v[g][e] != v[g][e];
            }
            of_chunk += of_group;
        }
        square += of_chunk;
        if (not_a_number) magnitude = __builtin_inff();            // takes the same scale as a NaN
    }
    __device__ __forceinline__ void split(const GramRowsArgs &args, gram_chunk *pieces, int row, int slice0, int half, float scale) const
    {
        const int all_slices = args.slices + args.zero_slices;
#pragma unroll
        for (int g = 0; g < GROUPS; g++) {
            const int slice = slice0 + GRO_WAVES * g;
            if (slice >= all_slices) break;
            unsigned h1[4], h2[4];
#pragma unroll
            for (int q = 0; q < 4; q++) gram_split_pair(v[g][2 * q] * scale, v[g][2 * q + 1] * scale, h1[q], h2[q]);
            gram_chunk *dst = pieces + ((i64)slice * GW_SEGMENTS + half) * args.rows_pad + row;
            dst[0] = gram_chunk{h1[0], h1[1], h1[2], h1[3]};
            dst[2 * (i64)args.rows_pad] = gram_chunk{h2[0], h2[1], h2[2], h2[3]};
        }
    }
};

// LONG: as in gram_rows_once_of, in chunks of 64 GROUPS k.
template <int GROUPS, bool LONG>
__device__ __forceinline__ void gram_columns_once_of(const GramRowsArgs &args, int block)
{
    __shared__ float squares[GRO_WAVES][GCO_ROWS], magnitudes[GRO_WAVES][GCO_ROWS];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), r = threadIdx.x & 31, half = (threadIdx.x >> 5) & 1;
    const int row = block * GCO_ROWS + r, batch = blockIdx.z;
    const bool live = row < args.rows;
    const float *src = args.x + batch * args.bs + (live ? row : args.rows - 1);
    const float *centre = args.centre ? args.centre + batch * args.centre_bs : nullptr;
    CentreSums sums;
    if (centre && args.centre_pairs) sums.load(centre, args.k, args.centre_pairs);
    constexpr int CHUNK = GRO_WAVES * GROUPS;                  // slices
    ColumnValues<GROUPS> values;
    values.load(args, src, wave, half);
    const bool subtract = centre && args.centre_pairs ? !sums.needless() : gram_rows_centre(args, batch) != nullptr;
    values.centre(args, centre, wave, half, subtract, live);
    float square = 0.0f, magnitude = 0.0f;
    values.statistics(square, magnitude);
    if constexpr (LONG)
        for (int at = CHUNK; at < args.slices; at += CHUNK) {
            values.load(args, src, at + wave, half);
            values.centre(args, centre, at + wave, half, subtract, live);
            values.statistics(square, magnitude);
        }
    square += __shfl_xor(square, 32);
    magnitude = fmaxf(magnitude, __shfl_xor(magnitude, 32));
    if (half == 0) {
        squares[wave][r] = square;
        magnitudes[wave][r] = magnitude;
    }
    __syncthreads();
    magnitude = fmaxf(fmaxf(magnitudes[0][r], magnitudes[1][r]), fmaxf(magnitudes[2][r], magnitudes[3][r]));
    const int exponent_field = gram_scale_exponent(magnitude);
    const float scale = gram_scale(exponent_field);
    if (threadIdx.x < GCO_ROWS) {
        args.squares[batch * args.stats_bs + row] = (squares[0][r] + squares[1][r]) + (squares[2][r] + squares[3][r]);
        args.unscale[batch * args.unscale_bs + row] = gram_unscale(exponent_field);
    }
    gram_chunk *pieces = args.pieces + batch * args.pieces_bs;
    if constexpr (LONG) {
        const int last = (args.slices - 1) / CHUNK * CHUNK;
        values.split(args, pieces, row, last + wave, half, scale);
        for (int at = last - CHUNK; at >= 0; at -= CHUNK) {
            values.load(args, src, at + wave, half);
            values.centre(args, centre, at + wave, half, subtract, live);
            values.split(args, pieces, row, at + wave, half, scale);
        }
    } else {
        values.split(args, pieces, row, wave, half, scale);
    }
}

template <int GROUPS, bool LONG = false>
__global__ __launch_bounds__(GW_ROW_THREADS, 2) void gram_columns_once(const GramRowsOnceArgs args)
{
    const int block = (int)blockIdx.x - args.samples;
    if (block < 0) {
        if (blockIdx.z == 0) gram_probe_tile(args.probe, blockIdx.x);
        return;
    }
    const bool first = block < args.first_blocks;
    if ((int)blockIdx.z < (first ? args.first_batches : args.second_batches))
        gram_columns_once_of<GROUPS, LONG>(first ? args.first : args.second, first ? block : block - args.first_blocks);
}

// Tile shapes of the product kernel.  A workgroup is 4 waves (8: EightWaves); a wave owns WAVE_M rows of a and WAVE_N rows of b as
// 16 x 16 blocks of the matrix instruction.  Two workgroups (three of the small shape) share a CU, so that one's
// prologue, epilogue and result stores run beside the other's matrix instructions.
template <int TILE_M_, int TILE_N_, int WAVES_N_, int SLOTS_>
struct WideShape {
    static constexpr int TILE_M = TILE_M_, TILE_N = TILE_N_;
    static constexpr int WAVES_M = 2, WAVES_N = WAVES_N_, WAVES = WAVES_M * WAVES_N, THREADS = 64 * WAVES;
    static constexpr int WAVE_M = TILE_M / WAVES_M, WAVE_N = TILE_N / WAVES_N;
    static constexpr int MT = WAVE_M / 16, NT = WAVE_N / 16;
    static constexpr int PARTS_M = TILE_M / 128, PARTS_N = TILE_N / 128, PARTS = PARTS_M * PARTS_N;
    static constexpr int GRANULE_CHUNKS = 4 * (TILE_M + TILE_N);          // 32 k of one piece of a and one of b
    static constexpr int COPIES_A = TILE_M / 16 / WAVES, COPIES_B = TILE_N / 16 / WAVES;  // runs of 64 chunks per wave and granule
    static constexpr int COPIES = COPIES_A + COPIES_B;
    static constexpr int SLOTS = SLOTS_;
    static constexpr int PER_CU = WAVES == 8 || TILE_M * TILE_N >= 256 * 128 ? 2 : 3;      // workgroups
    static constexpr int MIN_WAVES = PER_CU * WAVES / 4;                                   // per SIMD
};
template <int TILE_M, int TILE_N>
struct WideTile : WideShape<TILE_M, TILE_N, 2, 3> {};
// The small tile by 8 waves of 64 x 32, for results of at most two tiles per CU: four waves leave a SIMD one or two, and it waits at every
// granule's barrier for the reads of its operands.  With 8 a SIMD has two or four, and LDS for two whole steps of k, one barrier each.
// A workgroup reads half as much again from LDS, which is why three workgroups of four waves are the better where there are tiles for them.
// Product alone, 2000 x 2000 (256 tiles), 4 waves / 8: K = 784 47.3 / 41.4 us at the profiler's clock, K = 3072 155.6 / 139.8; calls at the rule.
// A ring of four steps in 128 KB, one workgroup per CU: 148.5 at K = 3072; XCDs that share rectangles of tiles in place of columns: 141.7.
template <typename Tile>
struct EightWaves : WideShape<Tile::TILE_M, Tile::TILE_N, 4, 4> {};
typedef WideTile<256, 128> WideTileLarge;
typedef WideTile<128, 128> WideTileSmall;
typedef EightWaves<WideTileSmall> WideTileFew;

// Workgroup -> tile, as tile_of_workgroup of build_kernel.hpp with bands of GW_BAND_N n tiles: n fastest inside a band,
// so the workgroups resident on an XCD (the hardware deals ids round-robin) cover a block of about 8 n tiles x 8 m tiles.
// SYMMETRIC (a panel against itself): the ids count through the 256 x 256 blocks on and below the diagonal (row r of
// the triangle starts at block r (r + 1) / 2), each of them the tiles of TILE_M x TILE_N it holds.
// args.entry_per_xcd (batches of small entries): of eight consecutive batch entries each has an XCD to itself, so that the tiles of
// an entry read their operands through one L2 instead of each through another; what is left over behind the last eight goes the ordinary way.
template <typename Tile, bool SYMMETRIC>
__device__ __forceinline__ bool wide_tile_of_workgroup(const GramWideArgs &args, int &batch, int &tile_m, int &tile_n)
{
    const int rotated = blockIdx.x + blockIdx.y % gridDim.x;
    int linear = rotated >= (int)gridDim.x ? rotated - (int)gridDim.x : rotated;
    batch = blockIdx.y;
    if (args.entry_per_xcd && (blockIdx.y | (BK_XCDS - 1)) < gridDim.y) {
        const int in_eight = (int)((blockIdx.y % BK_XCDS) * gridDim.x + blockIdx.x);
        batch = (int)(blockIdx.y / BK_XCDS * BK_XCDS) + in_eight % BK_XCDS;
        linear = in_eight / BK_XCDS;
    }
    if (SYMMETRIC) {
        constexpr int PER_M = GW_TILE / Tile::TILE_M, PER_N = GW_TILE / Tile::TILE_N;
        const int block = linear / (PER_M * PER_N), inside = linear - block * (PER_M * PER_N);
        int row = (int)((sqrtf(8.0f * (float)block + 1.0f) - 1.0f) * 0.5f);
        while (row * (row + 1) / 2 > block) row--;
        while ((row + 1) * (row + 2) / 2 <= block) row++;
        tile_m = row * PER_M + inside % PER_M;
        tile_n = (block - row * (row + 1) / 2) * PER_N + inside / PER_M;
        return tile_m < args.wide_tiles_m && tile_n < args.wide_tiles_n && tile_n * Tile::TILE_N < (tile_m + 1) * Tile::TILE_M;
    }
    const int band_tiles = GW_BAND_N * args.wide_tiles_m;
    const int band = linear / band_tiles;
    const int band_height = min(GW_BAND_N, args.wide_tiles_n_padded - band * GW_BAND_N);
    const int in_band = linear - band * band_tiles;
    tile_m = in_band / band_height;
    tile_n = band * GW_BAND_N + in_band % band_height;
    return tile_n < args.wide_tiles_n;
}

// The walk.  A step is 32 k: three products of pieces, a1 b2 + a1 b1 + a2 b1, on v_mfma_f32_16x16x32_f16.
//
// Why the 16 x 16 form: with real data in the registers this instruction sustains 1.93 PFLOP/s and the 32 x 32 x 16 one
// 1.71 (2.47 both on zeros: the board is power-limited, and the smaller tile moves half the accumulator words per
// multiply-add).
//
// The pieces go from the workspace straight into LDS (global_load_lds_dwordx4: a wave copies 64 consecutive chunks, no
// registers involved) in granules of one piece of a and one of b, in the order the products need them: a granule G1 is
// {a1, b2} of a step, G2 is {a2, b1}; three slots of LDS in turn.  One set of operand registers is enough: a1 and b2
// are not needed behind the product a1 b1, so the G1 of the next step is read during a2 b1; b1 and a2 are free behind
// a2 b1, so G2 is read during a1 b2.  A barrier stands in front of each read: behind it the granule to be read has
// arrived for every wave, and the one read before is free to be filled again.
//
// The copies are written as instructions: through the compiler's builtin every later LDS read waits for every copy
// under way (the copies carry no information on which array they fill), which leaves nothing in flight.  The compiler
// therefore does not count these copies either; the walk waits for them itself, and no other vector load is issued
// between the first copy and the end of the walk.  Nothing is copied beyond the last step.
template <typename Tile>
struct WideWalk {
    typedef const __attribute__((address_space(1))) char *global_address;
    typedef __attribute__((address_space(3))) void *lds_address;

    const char *run_a[Tile::COPIES_A], *run_b[Tile::COPIES_B];      // uniform: piece 1 of a, piece 1 of b, step 0
    i64 piece_a, piece_b, step_a, step_b;                           // bytes
    unsigned lane_offset, lds_base, lds_run_a[Tile::COPIES_A], lds_run_b[Tile::COPIES_B];
    gram_chunk *ring;
    int read_a, read_b;

    __device__ __forceinline__ void init(const gram_chunk *pieces_a, int rows_pad_a, int m0, const gram_chunk *pieces_b, int rows_pad_b,
                                         int n0, gram_chunk *ring_, int lane, int wave, int wave_m, int wave_n)
    {
        ring = ring_;
        lane_offset = 16u * lane;
        lds_base = (unsigned)(unsigned long)(lds_address)ring;
        // quarter q of a step's 32 k: slice q / 2, half q % 2 of the workspace's [slice][piece][half][row]
        auto segment = [](int quarter, int rows_pad) { return (i64)((quarter >> 1) * GW_SEGMENTS + (quarter & 1)) * rows_pad; };
#pragma unroll
        for (int j = 0; j < Tile::COPIES_A; j++) {
            const int run = wave + Tile::WAVES * j, quarter = run / (Tile::TILE_M / 64), part = run % (Tile::TILE_M / 64);
            run_a[j] = reinterpret_cast<const char *>(pieces_a + segment(quarter, rows_pad_a) + m0 + 64 * part);
            lds_run_a[j] = 1024u * run;
        }
#pragma unroll
        for (int j = 0; j < Tile::COPIES_B; j++) {
            const int run = wave + Tile::WAVES * j, quarter = run / (Tile::TILE_N / 64), part = run % (Tile::TILE_N / 64);
            run_b[j] = reinterpret_cast<const char *>(pieces_b + segment(quarter, rows_pad_b) + n0 + 64 * part);
            lds_run_b[j] = 64u * Tile::TILE_M + 1024u * run;
        }
        piece_a = 32ll * rows_pad_a; piece_b = 32ll * rows_pad_b;              // two segments of rows_pad chunks
        step_a = 2 * 16ll * GW_SEGMENTS * rows_pad_a; step_b = 2 * 16ll * GW_SEGMENTS * rows_pad_b;
        read_a = (lane >> 4) * Tile::TILE_M + wave_m + (lane & 15);
        read_b = 4 * Tile::TILE_M + (lane >> 4) * Tile::TILE_N + wave_n + (lane & 15);
    }

    // Granule SECOND (0: {a1, b2}, 1: {a2, b1}) of step `step` into slot `slot`.
    template <int SECOND>
    __device__ __forceinline__ void copy(int step, int slot) const
    {
        const unsigned to = lds_base + (unsigned)slot * (16u * Tile::GRANULE_CHUNKS);
        const i64 at_a = (i64)step * step_a + (SECOND ? piece_a : 0), at_b = (i64)step * step_b + (SECOND ? 0 : piece_b);
#pragma unroll
        for (int j = 0; j < Tile::COPIES_A; j++)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         : : "v"(lane_offset), "s"((global_address)(run_a[j] + at_a)), "s"(to + lds_run_a[j]) : "memory", "m0");
#pragma unroll
        for (int j = 0; j < Tile::COPIES_B; j++)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         : : "v"(lane_offset), "s"((global_address)(run_b[j] + at_b)), "s"(to + lds_run_b[j]) : "memory", "m0");
    }

    __device__ __forceinline__ void read(gram_half8 (&fa)[Tile::MT], gram_half8 (&fb)[Tile::NT], int slot, bool b_first) const
    {
        const gram_chunk *from = ring + slot * Tile::GRANULE_CHUNKS;
        if (b_first) {
#pragma unroll
            for (int nt = 0; nt < Tile::NT; nt++) fb[nt] = __builtin_bit_cast(gram_half8, from[read_b + 16 * nt]);
        }
#pragma unroll
        for (int mt = 0; mt < Tile::MT; mt++) fa[mt] = __builtin_bit_cast(gram_half8, from[read_a + 16 * mt]);
        if (!b_first) {
#pragma unroll
            for (int nt = 0; nt < Tile::NT; nt++) fb[nt] = __builtin_bit_cast(gram_half8, from[read_b + 16 * nt]);
        }
    }
};

template <int COUNT>
__device__ __forceinline__ void wide_wait_copies()
{
    static_assert(COUNT < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (COUNT & 15) | ((COUNT >> 4) << 14));     // vmcnt(COUNT), nothing else
}

// Between writes and reads of LDS through which the lanes of a wave hand values to each other: the hardware keeps a wave's LDS
// instructions in order, the compiler by itself only those of one lane.  No instruction comes of it.
__device__ __forceinline__ void wide_lanes_exchange()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The matrix instructions are written out: left to itself the compiler gives their results other registers than their
// sums came from, which does not fit beside the operands.  Two products into the same sums are at least 16 matrix
// instructions apart (8 in EightWaves), and the walk ends with the wait states that vector instructions need before they read the sums.
// The blocks are walked back and forth, so that an instruction always shares one operand with the one in front of it: the board
// is power-limited here and a new operand costs energy.  With every row of blocks walked from its first, and now: 30000 x 30000 x 1024 4908 -> 4878 us,
// 1000 x 60000 x 784 and its product 452 -> 449, where two runs differ by 0.2 %; four pairs of runs of the gradient at 2 x 10000 x 768 x 16 x 10000
// 0.8 .. 1.5 % apart, a fifth level.  (Columns of blocks back and forth, where the first operand changes more often: half of that; column by column without
// turning: nothing.  Tiles of 128 x 256, 64 x 128 per wave: level, but 13.3 against 12.5 ms for the gradient, whose epilogue fetches more; of 256 x 256 by 8
// waves, one workgroup per CU: 2 .. 5 % slower, also at K = 10000.)
// The compiler, which keeps such distances for instructions it knows, does not see these: nothing else may read or move a sum between
// the first product and those wait states, which holds as long as the sums stay where they are (the test of the kernel's listing
// looks at every instruction in between).
template <int MT, int NT, int FIRST, int LAST>
__device__ __forceinline__ void wide_multiply(gram_float4 (&acc)[MT][NT], const gram_half8 (&fa)[MT], const gram_half8 (&fb)[NT])
{
#pragma unroll
    for (int mt = FIRST; mt < LAST; mt++)
#pragma unroll
        for (int turn = 0; turn < NT; turn++) {
            const int nt = mt % 2 == 0 ? turn : NT - 1 - turn;
            asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc[mt][nt]) : "v"(fa[mt]), "v"(fb[nt]));
        }
}

template <typename Tile>
__device__ __forceinline__ void wide_walk(gram_float4 (&acc)[Tile::MT][Tile::NT], const WideWalk<Tile> &walk, int steps)
{
    constexpr int MT = Tile::MT, NT = Tile::NT, COPIES = Tile::COPIES;
    gram_half8 a1[MT], a2[MT], b1[NT], b2[NT];
    walk.template copy<0>(0, 0);
    walk.template copy<1>(0, 1);
    if (steps > 1) {
        walk.template copy<0>(1, 2);
        wide_wait_copies<2 * COPIES>();
    } else {
        wide_wait_copies<COPIES>();
    }
    __syncthreads();
    walk.read(a1, b2, 0, true);
    int slot = 0;                                       // of this step's first granule
    for (int step = 0; step < steps; step++) {
        const int second = slot == 2 ? 0 : slot + 1, third = second == 2 ? 0 : second + 1;
        const bool more = step + 1 < steps;
        wide_multiply<MT, NT, 0, MT / 2>(acc, a1, b2);
        __builtin_amdgcn_sched_barrier(0);
        if (more) wide_wait_copies<COPIES>();            // the second granule has arrived; the next step's first may be under way
        else wide_wait_copies<0>();
        __syncthreads();
        walk.read(a2, b1, second, true);
        if (more) walk.template copy<1>(step + 1, slot);
        __builtin_amdgcn_sched_barrier(0);
        wide_multiply<MT, NT, MT / 2, MT>(acc, a1, b2);
        wide_multiply<MT, NT, 0, MT>(acc, a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
            wide_wait_copies<COPIES>();
            __syncthreads();
            walk.read(a1, b2, third, true);
            if (step + 2 < steps) walk.template copy<0>(step + 2, second);
            __builtin_amdgcn_sched_barrier(0);
        } else {
            // said out loud: with unread operands on one of the two ways here, the products below would wait for the
            // reads just issued on the other
            __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0), nothing else
        }
        wide_multiply<MT, NT, 0, MT>(acc, a2, b1);
        __builtin_amdgcn_sched_barrier(0);
        slot = third;
    }
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) asm volatile("" : "+v"(acc[mt][nt]));
}

// The walk of EightWaves: a ring of two whole steps and one barrier per step, in front of the read of a step's first granule.  Behind it both
// granules of that step have arrived for every wave, and the step before has been read.  The products go into a sum in wide_walk's order.
template <typename Tile>
__device__ __forceinline__ void wide_walk_steps(gram_float4 (&acc)[Tile::MT][Tile::NT], const WideWalk<Tile> &walk, int steps)
{
    static_assert(Tile::SLOTS == 4, "two steps of two granules");
    constexpr int MT = Tile::MT, NT = Tile::NT, COPIES = Tile::COPIES;
    gram_half8 a1[MT], a2[MT], b1[NT], b2[NT];
    walk.template copy<0>(0, 0);
    walk.template copy<1>(0, 1);
    if (steps > 1) {
        walk.template copy<0>(1, 2);
        walk.template copy<1>(1, 3);
        wide_wait_copies<2 * COPIES>();
    } else {
        wide_wait_copies<0>();
    }
    __syncthreads();
    walk.read(a1, b2, 0, true);
    int slot = 0;                                       // of this step's first granule
    for (int step = 0; step < steps; step++) {
        const int next = 2 - slot;
        walk.read(a2, b1, slot + 1, true);
        __builtin_amdgcn_sched_barrier(0);
        wide_multiply<MT, NT, 0, MT>(acc, a1, b2);
        wide_multiply<MT, NT, 0, MT>(acc, a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        if (step + 1 < steps) {
            wide_wait_copies<0>();                       // only the next step's copies are under way
            __syncthreads();
            walk.read(a1, b2, next, true);
            if (step + 2 < steps) {
                walk.template copy<0>(step + 2, slot);
                walk.template copy<1>(step + 2, slot + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        } else {
            __builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0), nothing else; why: at the end of wide_walk
        }
        wide_multiply<MT, NT, 0, MT>(acc, a2, b1);
        __builtin_amdgcn_sched_barrier(0);
        slot = next;
    }
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) asm volatile("" : "+v"(acc[mt][nt]));
}

// SYMMETRIC: b is a, the result is symmetric, and it is made so bit for bit: the tiles on or below the diagonal are
// computed; what lies below the diagonal is stored a second time, mirrored; of a 128 x 128 part on the diagonal the
// lower triangle is stored and mirrored (the two halves of such a part are computed with the pieces in exchanged
// roles and differ in the last bit); a part above the diagonal inside a tile is not stored from its own values at
// all.  A distrusted part is left to the repair launch, which mirrors what it recomputes.
//
// EPILOGUE GW_EPILOGUE_GRADIENT_L2: the same walk as a plain product of the pieces, for the gradient
// of the L2 norm (norm_gradient_l2_wide.hpp): no norms, no trust check, the epilogue combines the
// product with d and g as GramWideArgs says.
//
// EPILOGUE GW_EPILOGUE_DOT: the inner operator DOT (sum_k a b): the product of the pieces is the
// value itself, nothing cancels, so there is no trust check and no repair; outer power, kernel
// function, regularised diagonal and the stores, mirrored ones included, are those of the distance.
//
// GW_CONTRACT_16, GW_CONTRACT_32 (COLUMNS = 16, 32): the values are not stored but contracted with up to COLUMNS columns of coefficients, and the product of
// every tile of 128 n goes to a place of its own, to be added up by sum_products: out[m, o] = sum_n C(m, n) coef[n, o].  A wave stages 16
// columns n as for the stores and multiplies them with v_mfma_f32_16x16x4_f32 (fp32 operands and sums), lane q of four
// groups on n = 4 q + step, so that its reads of the staged values fall into banks of their own.  Panels of the matrix stored
// and contracted by a kernel of their own / this, us: 1000 x 60000 x 784, 10 columns 461 / 391, 32 columns 457 / 414; 4 x 16384 x 16384 x 256, 32 columns
// 3679 / 2967, 10 columns 3664 / 2407; 30000 x 30000 x 1024, 16 columns 5846 / 5070; 8192 x 65536 x 128, 8 columns 1436 / 1002; 4096 x 4096 x 256,
// 32 columns 87 / 76; 500 x 500 x 2000, 10 columns 113 / 101; none of 24 shapes was slower.
template <typename Tile, bool SYMMETRIC, int WHAT = GW_EPILOGUE_DISTANCE>
__global__ __launch_bounds__(Tile::THREADS, Tile::MIN_WAVES) void gram_f16_wide(const GramWideArgs args)
{
    constexpr int EPILOGUE = WHAT % GW_CONTRACT_16, COLUMNS = WHAT / GW_CONTRACT_16 * 16;
    static_assert(COLUMNS == 0 || (!SYMMETRIC && EPILOGUE != GW_EPILOGUE_GRADIENT_L2 && Tile::TILE_N == 128), "what the contraction is for");
    constexpr int TILE_M = Tile::TILE_M, TILE_N = Tile::TILE_N, MT = Tile::MT, NT = Tile::NT;
    __shared__ gram_chunk ring[Tile::SLOTS * Tile::GRANULE_CHUNKS];
    __shared__ __attribute__((aligned(16))) float lds_norm_a[TILE_M], lds_norm_b[TILE_N];
    __shared__ __attribute__((aligned(16))) float lds_unscale_a[TILE_M], lds_unscale_b[TILE_N];
    __shared__ int lds_distrust[Tile::PARTS];

    const int tid = threadIdx.x;
    int batch, tile_m, tile_n;
    if (!wide_tile_of_workgroup<Tile, SYMMETRIC>(args, batch, tile_m, tile_n)) return;
    const int m0 = tile_m * TILE_M;
    const int n0 = tile_n * TILE_N;
    const int m_valid = args.kernel.m - m0;
    const int n_valid = args.kernel.n - n0;

    if constexpr (EPILOGUE == GW_EPILOGUE_DISTANCE) {
        // The sample of the result says that the repair launch would redo (nearly) every part: stamp them all
        // and leave (the branch is uniform over the launch: every workgroup reads the same words).  Parts above the diagonal of a symmetric result belong to nobody.
        if (args.kernel.sample && sample_leaves_it_to_the_direct_kernel(args.kernel.sample)) {
            if (tid < Tile::PARTS) {
                const int part_m = tid % Tile::PARTS_M * 128, part_n = tid / Tile::PARTS_M * 128;
                const bool above = SYMMETRIC && m0 + part_m < n0 + part_n;
                if constexpr (COLUMNS > 0) {
                    if (part_m < m_valid) args.stamps[((i64)batch * args.stamps_m + (m0 + part_m) / 128) * args.stamps_n + tile_n] = 1;
                } else if (!above && part_m < m_valid && part_n < n_valid)
                    args.kernel.c[batch * args.kernel.c_bs + (i64)(n0 + part_n) * args.kernel.c_ld + m0 + part_m] =
                        __uint_as_float(BK_REPAIR_MARKER);
            }
            return;
        }
    }

    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = (wave % Tile::WAVES_M) * Tile::WAVE_M;
    const int wave_n = (wave / Tile::WAVES_M) * Tile::WAVE_N;

    // Norms of this tile's rows (the partial sums in the order of their ranges) and their scales.
    for (int at = tid; at < TILE_M + TILE_N; at += Tile::THREADS) {
        const bool of_a = at < TILE_M;
        const int r = of_a ? at : at - TILE_M;
        if constexpr (EPILOGUE == GW_EPILOGUE_DISTANCE) {
            const float *partial = of_a ? args.squares_a + batch * args.stats_a_bs + m0 + r : args.squares_b + batch * args.stats_b_bs + n0 + r;
            const int pitch = of_a ? args.rows_pad_a : args.rows_pad_b, ranges = of_a ? args.ranges_a : args.ranges_b;
            // all loads first, then the sum in range order: a loop would wait for each load in turn
            float parts[GW_MAX_RANGES];
#pragma unroll
            for (int range = 0; range < GW_MAX_RANGES; range++) parts[range] = range < ranges ? partial[(i64)range * pitch] : 0.0f;
            float norm = 0.0f;
#pragma unroll
            for (int range = 0; range < GW_MAX_RANGES; range++) norm += range < ranges ? parts[range] : 0.0f;
            (of_a ? lds_norm_a : lds_norm_b)[r] = norm;
        }
        (of_a ? lds_unscale_a : lds_unscale_b)[r] =
            of_a ? args.unscale_a[batch * args.unscale_a_bs + m0 + r] : args.unscale_b[batch * args.unscale_b_bs + n0 + r];
    }
    if (tid < Tile::PARTS) lds_distrust[tid] = 0;

    gram_float4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = gram_float4{0.0f, 0.0f, 0.0f, 0.0f};
    {
        WideWalk<Tile> walk;
        walk.init(args.pieces_a + batch * args.pieces_a_bs, args.rows_pad_a, m0, args.pieces_b + batch * args.pieces_b_bs, args.rows_pad_b, n0,
                  ring, lane, wave, wave_m, wave_n);
        if constexpr (Tile::SLOTS == 3) wide_walk<Tile>(acc, walk, (args.slices + 1) / 2);
        else wide_walk_steps<Tile>(acc, walk, (args.slices + 1) / 2);
    }
    // The last barrier of the walk stands in front of its last reads; behind this one every wave has its operands, and the
    // ring is free for the staging of the results (the gradient's epilogue stages nothing).
    if constexpr (EPILOGUE != GW_EPILOGUE_GRADIENT_L2) __syncthreads();

    // Everything behind the walk is derived from a copy of the lane id and of the argument block's address that the
    // compiler cannot see through: computed before the walk and kept through it, it would push the walk's operands
    // into scratch memory.
    int lane_after = lane;
    asm volatile("" : "+v"(lane_after));
    typedef const __attribute__((address_space(4))) GramWideArgs *argument_pointer;
    argument_pointer late = (argument_pointer)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(late));
    const auto *kernel = &late->kernel;
    // A lane holds, of every 16 x 16 block, one row of b (its lane number modulo 16) and 4 consecutive m:
    //   acc[mt][nt][v]:  m = wave_m + 16 mt + 4 q + v,  n = wave_n + 16 nt + i
    const int q = lane_after >> 4;
    const int i = lane_after & 15;
    const int rows = kernel->m - m0, columns = kernel->n - n0;      // of the result, from this tile's first element on
    float *c_tile = kernel->c + batch * kernel->c_bs + (i64)n0 * kernel->c_ld + m0;
    const i64 c_ld = kernel->c_ld;
    const bool c_vec = kernel->c_vec != 0;
    if constexpr (EPILOGUE == GW_EPILOGUE_GRADIENT_L2) {
        const int gradient_n = late->gradient_n;
        const i64 g_ld = late->gradient_g_ld;
        const float *g_tile = late->gradient_g + batch * late->gradient_g_bs + (i64)m0 * g_ld;
        const float *d_tile = late->gradient_d + batch * late->gradient_d_bs + m0;
        const float *shifts = late->gradient_shift + batch * late->gradient_shift_bs;
        const i64 d_ld = late->gradient_d_ld;
        const bool full = rows >= TILE_M;
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int r_local = wave_n + nt * 16 + i;
            if (r_local >= columns) continue;
            const int r = n0 + r_local;
            const int o = r / gradient_n, n = r - o * gradient_n;
            const float unscale_b = lds_unscale_b[r_local];
            const float shift = shifts[n];
            const float *d_row = d_tile + (i64)n * d_ld;
            float *row = c_tile + (i64)r_local * c_ld;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int m_local = wave_m + mt * 16 + 4 * q;
                const float4 unscale_a = *reinterpret_cast<const float4 *>(&lds_unscale_a[m_local]);
                const float unscales_a[4] = {unscale_a.x, unscale_a.y, unscale_a.z, unscale_a.w};
                float v4[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const bool exists = full || m_local + e < rows;
                    const float d = exists ? d_row[m_local + e] - shift : 0.0f;
                    const float weight = exists ? g_tile[(i64)(m_local + e) * g_ld + o] : 0.0f;
                    v4[e] = d * weight - (acc[mt][nt][e] * unscales_a[e]) * unscale_b;
                }
                if (c_vec && (full || m_local + 3 < rows)) {
                    *reinterpret_cast<float4 *>(row + m_local) = make_float4(v4[0], v4[1], v4[2], v4[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (m_local + e < rows) row[m_local + e] = v4[e];
                }
            }
        }
        return;
    }

    const int part_m = wave_m / 128, part_n = wave_n / 128;
    const int part = part_m + Tile::PARTS_M * part_n;
    // where this wave's part lies: below the diagonal of the result (stored and mirrored), on it
    // (lower triangle stored and mirrored), above it inside a tile (not stored)
    const bool on_diagonal = SYMMETRIC && m0 + 128 * part_m == n0 + 128 * part_n;
    const bool above = SYMMETRIC && m0 + 128 * part_m < n0 + 128 * part_n;

    const int outer_power = kernel->outer_power;
    const int kernel_type = kernel->kernel_type;
    const float trust = kernel->gram_trust;
    const float epsilon = kernel->epsilon;
    float p_outer = 0.0f, neg_gamma = 0.0f, diagonal_value = 0.0f;
    if (outer_power == POW_POW) p_outer = kernel->p_outer ? kernel->p_outer[batch * kernel->p_outer_bs] : kernel->p_outer_value;
    // element (m, n) is regularised when reg_off_x + m == reg_off_y + n: 16 mt + 4 q + v == diagonal + 16 nt + i
    const int diagonal = kernel->reg_off_y + n0 + wave_n - kernel->reg_off_x - m0 - wave_m;
    bool regularize = false;
    if (kernel_type != KERNEL_NONE) {
        neg_gamma = kernel_neg_gamma(kernel_type, kernel->bandwidth ? kernel->bandwidth[batch * kernel->bandwidth_bs] : kernel->bandwidth_value);
        const float regularization =
            kernel->regularization ? kernel->regularization[batch * kernel->regularization_bs] : kernel->regularization_value;
        diagonal_value = 1.0f + regularization;
        regularize = regularization != 0.0f && diagonal < Tile::WAVE_M && diagonal > -Tile::WAVE_N;
    }

    // 16 columns n at a time: d^2 = |a|^2 + |b|^2 - 2 a.b and the trust check per 128 x 128 part (the unit the repair
    // launch works in; every wave lies inside one part), the outer function and the kernel function, the stores.
    // A result is trusted when d^2 >= trust * norms, judged as norms * (1 - trust) - 2 a.b >= 0; a lane keeps its least
    // such margin (v_minimum3_f32 hands a NaN on: overflowing squares and NaN data are not trusted).  Rows and columns
    // that do not exist have pieces and norms of zero: with a row or column that does exist they give d^2 = norms,
    // which is trusted unless that row's norm is not a number -- and then its own elements are not trusted either.
    // A point against itself (BuildKernelArgs::same_points) is at distance zero, exactly, if its norm is a number: without
    // that the parts on the diagonal are all distrusted, and the repair launch walks each of them on one CU (10000 points of
    // K = 784 against themselves: 254 of 590 us; 338 with it).
    // The stores go through this wave's share of the ring (free since the barrier behind the walk), so that an instruction
    // writes runs of WAVE_M floats of a column.
    float least_margin = 0.0f;
    const int self_diagonal = n0 + wave_n + kernel->same_shift - m0 - wave_m;
    const bool same_points = kernel->same_points != 0 && self_diagonal < Tile::WAVE_M && self_diagonal > -Tile::WAVE_N;
    float *stage = reinterpret_cast<float *>(ring) + wave * (4 * Tile::SLOTS * Tile::GRANULE_CHUNKS / Tile::WAVES);
    {
        constexpr int PITCH = Tile::WAVE_M + 4, LANES = Tile::WAVE_M / 4, PER_PASS = 64 / LANES;
        static_assert(16 * PITCH <= 4 * Tile::SLOTS * Tile::GRANULE_CHUNKS / Tile::WAVES, "the staging fits a wave's share of the ring");
        const int row = wave_m + 4 * (lane_after % LANES);
        const bool whole = c_vec && row + 3 < rows;
        constexpr int OB = COLUMNS > 0 ? COLUMNS / 16 : 1;
        gram_float4 products[COLUMNS > 0 ? MT : 1][OB];          // [m block][o block]: o = 16 ob + 4 q + v, m = wave_m + 16 mt + i
        const float *coef = nullptr;
        if constexpr (COLUMNS > 0) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int ob = 0; ob < OB; ob++) products[mt][ob] = gram_float4{0.0f, 0.0f, 0.0f, 0.0f};
            coef = late->coef + batch * late->coef_bs;
        }
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            float weights[COLUMNS > 0 ? 4 : 1][OB];              // of n = 16 nt + 4 q + step, o = 16 ob + i
            if constexpr (COLUMNS > 0) {
#pragma unroll
                for (int step = 0; step < 4; step++)
#pragma unroll
                    for (int ob = 0; ob < OB; ob++) {
                        const int n_local = wave_n + 16 * nt + 4 * q + step, o = 16 * ob + i;
                        weights[step][ob] = n_local < columns && o < late->outputs ? coef[(i64)(n0 + n_local) * late->coef_ld + o] : 0.0f;
                    }
            }
            const float norm_b = EPILOGUE == GW_EPILOGUE_DISTANCE ? lds_norm_b[wave_n + nt * 16 + i] : 0.0f;
            const float unscale_b = (EPILOGUE == GW_EPILOGUE_DISTANCE ? -2.0f : 1.0f) * lds_unscale_b[wave_n + nt * 16 + i];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int m_local = wave_m + mt * 16 + 4 * q;
                const gram_float4 unscale_a = *reinterpret_cast<const gram_float4 *>(&lds_unscale_a[m_local]);
                if constexpr (EPILOGUE == GW_EPILOGUE_DOT) {
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[mt][nt][e] = (acc[mt][nt][e] * unscale_a[e]) * unscale_b;
                } else {
                    const gram_float4 norm_a = *reinterpret_cast<const gram_float4 *>(&lds_norm_a[m_local]);
                    float margin[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float norms = norm_a[e] + norm_b;
                        const float minus_twice = (acc[mt][nt][e] * unscale_a[e]) * unscale_b;
                        acc[mt][nt][e] = norms + minus_twice;
                        margin[e] = norms * (1.0f - trust) + minus_twice;
                        if (same_points) {
                            const bool same = 16 * mt + 4 * q + e == self_diagonal + 16 * nt + i;
                            acc[mt][nt][e] = same ? norms - norms : acc[mt][nt][e];
                            margin[e] = same ? norms - norms : margin[e];
                        }
                    }
                    asm("v_minimum3_f32 %0, %1, %2, %0" : "+v"(least_margin) : "v"(margin[0]), "v"(margin[1]));
                    asm("v_minimum3_f32 %0, %1, %2, %0" : "+v"(least_margin) : "v"(margin[2]), "v"(margin[3]));
                }
            }
            // the outer function and the kernel function of epilogue_value (device_common.hpp), the switches outside the loops
            auto for_each = [&](auto &&f) {
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int v = 0; v < 4; v++) acc[mt][nt][v] = f(acc[mt][nt][v]);
            };
            switch (outer_power) {
            case POW_ABS: for_each([](float v) { return fabsf(v); }); break;
            case POW_SQUARE: for_each([](float v) { return v * v; }); break;
            case POW_SQRT: for_each([](float v) { return __builtin_amdgcn_sqrtf(v); }); break;
            case POW_POW: for_each([=](float v) { return epilogue_value(v, POW_POW, KERNEL_NONE, p_outer, 0.0f, 0.0f); }); break;
            default: break;
            }
            if (kernel_type != KERNEL_NONE) {
                for_each([=](float v) { return epilogue_value(v, POW_NOOP, kernel_type, 0.0f, neg_gamma, epsilon); });
                if (regularize) {
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
#pragma unroll
                        for (int v = 0; v < 4; v++)
                            acc[mt][nt][v] = 16 * mt + 4 * q + v == diagonal + 16 * nt + i ? diagonal_value : acc[mt][nt][v];
                }
            }
            if (above) continue;
            if constexpr (COLUMNS > 0) {
                // columns that do not exist may hold anything, which is no factor of a zero coefficient
                const bool exists = wave_n + 16 * nt + i < columns;
                wide_lanes_exchange();
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    *reinterpret_cast<gram_float4 *>(stage + i * PITCH + 16 * mt + 4 * q) = exists ? acc[mt][nt] : gram_float4{0.0f, 0.0f, 0.0f, 0.0f};
                wide_lanes_exchange();
#pragma unroll
                for (int step = 0; step < 4; step++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        const float value = stage[(4 * q + step) * PITCH + 16 * mt + i];
#pragma unroll
                        for (int ob = 0; ob < OB; ob++)
                            products[mt][ob] = __builtin_amdgcn_mfma_f32_16x16x4f32(weights[step][ob], value, products[mt][ob], 0, 0, 0);
                    }
                continue;
            }
            wide_lanes_exchange();
#pragma unroll
            for (int mt = 0; mt < MT; mt++) *reinterpret_cast<gram_float4 *>(stage + i * PITCH + 16 * mt + 4 * q) = acc[mt][nt];
            wide_lanes_exchange();
#pragma unroll
            for (int pass = 0; pass < 16 / PER_PASS; pass++) {
                const int column = pass * PER_PASS + lane_after / LANES;
                const gram_float4 v = *reinterpret_cast<const gram_float4 *>(stage + column * PITCH + 4 * (lane_after % LANES));
                const int n_local = wave_n + 16 * nt + column;
                float *to = c_tile + (i64)n_local * c_ld + row;
                // on the diagonal only m >= n
                const int first = SYMMETRIC && on_diagonal ? n0 + n_local - (m0 + row) : 0;
                if (n_local < columns) {
                    if (whole && first <= 0) {
                        *reinterpret_cast<gram_float4 *>(to) = v;
                    } else {
                        for (int e = first > 0 ? first : 0; e < 4 && row + e < rows; e++) to[e] = e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (COLUMNS > 0) {
            // The products of the waves side by side along n, added in their order.  (The ring holds the staged values of every wave until here.)
            constexpr int QUADS = MT * OB;
            static_assert(64 * QUADS * (Tile::WAVES - Tile::WAVES_M) <= Tile::SLOTS * Tile::GRANULE_CHUNKS, "the products of all but the first fit the ring");
            gram_float4 *shared = reinterpret_cast<gram_float4 *>(ring);
            const int along_m = wave % Tile::WAVES_M, along_n = wave / Tile::WAVES_M;
            if (EPILOGUE == GW_EPILOGUE_DISTANCE && !(least_margin >= 0.0f)) lds_distrust[part] = 1;
            __syncthreads();
            if (along_n > 0) {
#pragma unroll
                for (int at = 0; at < QUADS; at++)
                    shared[(((along_n - 1) * Tile::WAVES_M + along_m) * QUADS + at) * 64 + lane_after] = products[at / OB][at % OB];
            }
            __syncthreads();
            if (EPILOGUE == GW_EPILOGUE_DISTANCE && wave == 0 && lane_after < Tile::PARTS && 128 * lane_after < rows)
                late->stamps[((i64)batch * late->stamps_m + m0 / 128 + lane_after) * late->stamps_n + tile_n] = lds_distrust[lane_after];
            if (along_n > 0) return;
            float *to = late->products + tile_n * late->products_tile + batch * late->products_bs + (i64)m0 * late->products_ld;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int ob = 0; ob < OB; ob++) {
                    gram_float4 sum = products[mt][ob];
#pragma unroll
                    for (int team = 1; team < Tile::WAVES_N; team++)
                        sum += shared[(((team - 1) * Tile::WAVES_M + along_m) * QUADS + mt * OB + ob) * 64 + lane_after];
                    const int m_local = wave_m + 16 * mt + i, o = 16 * ob + 4 * q;
                    if (m_local < rows && o < late->outputs) *reinterpret_cast<gram_float4 *>(to + m_local * late->products_ld + o) = sum;
                }
            return;
        }
    }
    if constexpr (EPILOGUE == GW_EPILOGUE_DISTANCE) {
        // A part with a distrusted element is stamped: its first element, stored a second time by the wave that stored
        // it first.  The repair launch recomputes the part (and mirrors it).
        if (!(least_margin >= 0.0f) && !above) lds_distrust[part] = 1;
        __syncthreads();
        if (lds_distrust[part] != 0 && lane_after == 0 && !above && (wave_m & 127) == 0 && (wave_n & 127) == 0 && wave_m < rows && wave_n < columns)
            c_tile[(i64)wave_n * c_ld + wave_m] = __uint_as_float(BK_REPAIR_MARKER);
    }
    if (above) return;

    // The same values at C(n, m): 32 rows m at a time through the same memory.
    if (SYMMETRIC) {
        constexpr int PITCH = Tile::WAVE_N + 4, LANES = Tile::WAVE_N / 4, PER_PASS = 64 / LANES;
        static_assert(32 * PITCH <= 4 * Tile::SLOTS * Tile::GRANULE_CHUNKS / Tile::WAVES, "the staging fits a wave's share of the ring");
        float *mirror = kernel->c + batch * kernel->c_bs + (i64)m0 * c_ld + n0;
        const int column = wave_n + 4 * (lane_after % LANES);
        const bool whole = c_vec && column + 3 < columns;
#pragma unroll
        for (int pair = 0; pair < MT / 2; pair++) {
            wide_lanes_exchange();
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int v = 0; v < 4; v++) stage[(16 * mt + 4 * q + v) * PITCH + 16 * nt + i] = acc[2 * pair + mt][nt][v];
            wide_lanes_exchange();
#pragma unroll
            for (int pass = 0; pass < 32 / PER_PASS; pass++) {
                const int row = pass * PER_PASS + lane_after / LANES;
                const gram_float4 v = *reinterpret_cast<const gram_float4 *>(stage + row * PITCH + 4 * (lane_after % LANES));
                const int m_local = wave_m + 32 * pair + row;
                float *to = mirror + (i64)m_local * c_ld + column;
                // on the diagonal only n < m
                const int last = on_diagonal ? m0 + m_local - (n0 + column) : 4;
                if (m_local < rows) {
                    if (whole && last >= 4) {
                        *reinterpret_cast<gram_float4 *>(to) = v;
                    } else {
                        for (int e = 0; e < 4 && e < last && column + e < columns; e++) to[e] = e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3];
                    }
                }
            }
        }
    }
}

}  // namespace kmc
