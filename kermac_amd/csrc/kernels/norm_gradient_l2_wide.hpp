// The gradient of the L2 norm as one matrix product on the fp16 matrix instruction.
//
//   e[o][n][m] = sum_k c[o][k] a[k][m] (d[n][m] - b[n][k])
//              = (d[n][m] - s[n]) g[m][o] - sum_k p[o N + n][k] a[k][m],
//   g[m][o] = sum_k a[k][m] c[o][k],   p[o N + n][k] = c[o][k] (b[n][k] - s[n]),
//
// for any shift s[n]; with s[n] the mean of row n of b both terms are as small as the data allows
// (a common offset of d and b, which the difference d - b never sees, would otherwise be multiplied
// out and cancelled).  The second term is a product of an (O N) x K matrix with a K x M one: the
// rows of p and the columns of a are split into two fp16 pieces per value with a scale per row,
// exactly as the squared-difference route does it (gram_f16_wide.hpp), and the same kernel walks
// the pieces (GW_EPILOGUE_GRADIENT_L2: three piece products per 32 k); its epilogue fetches d and g
// and stores e.  Where the fp32 kernels build c a (d - b) value by value on the vector ALU and
// contract it on the fp32 matrix instruction, this route has no work per (o, n, m, k) outside the
// matrix instruction.  Error of the product from the pieces below 3 * 2^-22 sum_k |c a (b - s)| +
// k 2^-38 max|a| max|c (b - s)|; g and the rest are fp32.
//
// This header: the kernels that prepare s, the transposed c, and the pieces of a and p (g itself comes from
// kmc_matrix_times_coefficients with a as the stored panel).  p is never stored: its values are made from b and c
// twice, for the largest magnitude of every row and for the pieces (written in fp32 and read twice it cost 0.9 of 13.5 ms at
// 2 x 10000 x 768 x 16 x 10000).  The magnitudes of a come from the kernel that makes g, which reads all of a anyway.  Everything in front of the
// product is its bytes there, us: g 254 -> 269, statistics of p 61 (of a and p 321), split 621 (667; c by vector loads), 982 (1273) in all, where 2.4 GB of a and
// 1 GB of p take 700 at a copy's rate.
#pragma once

#include <hip/hip_runtime.h>

#include "gram_f16_wide.hpp"

namespace kmc {

struct GradientL2PrepareArgs {
    const float *b; i64 b_ld, b_bs;          // [n][k], k contiguous
    const float *c; i64 c_ld, c_bs;          // [o][k], k contiguous
    float *shift; i64 shift_bs;              // [n]
    float *c_transposed; i64 c_transposed_ld, c_transposed_bs;   // [k][o]
    int n, o, k;
};

// gradient_l2_pieces_stats and gradient_l2_pieces_split: the operand a, and p row o n + n' of which is c[o] (b[n'] - shift[n'])
struct GradientL2PiecesArgs {
    GramRowsArgs a, p;                       // p.x is not read
    int a_blocks, a_batches;                 // workgroups along x: those of a, then of p
    int outputs;                             // rows of p per row n and workgroup of p, up to GL2_OUTPUTS
    GradientL2PrepareArgs from;
};

constexpr int GL2_THREADS = 256;
constexpr int GL2_ROWS = 64;         // rows n of a workgroup: a lane each
constexpr int GL2_DEPTH = 64;        // k at a time, a slice of 16 per wave
constexpr int GL2_OUTPUTS = 4;       // rows of p per row n and workgroup, at most

// The mean of row n of b (sums in a fixed order), one workgroup per row; behind them c_transposed[k][o] = c[o][k].
__global__ __launch_bounds__(GL2_THREADS) void gradient_l2_prepare(const GradientL2PrepareArgs args)
{
    __shared__ float partial[GL2_THREADS];
    const int batch = blockIdx.y;
    if ((int)blockIdx.x >= args.n) {
        const int k = (blockIdx.x - args.n) * GL2_THREADS + threadIdx.x;
        if (k >= args.k) return;
        const float *c = args.c + batch * args.c_bs;
        float *row = args.c_transposed + batch * args.c_transposed_bs + (i64)k * args.c_transposed_ld;
        for (int o = 0; o < args.o; ++o) row[o] = c[(i64)o * args.c_ld + k];
        return;
    }
    const int n = blockIdx.x;
    const float *b_row = args.b + batch * args.b_bs + (i64)n * args.b_ld;
    float sum = 0.0f;
    for (int k = threadIdx.x; k < args.k; k += GL2_THREADS) sum += b_row[k];
    partial[threadIdx.x] = sum;
    __syncthreads();
    for (int width = GL2_THREADS / 2; width > 0; width >>= 1) {
        if ((int)threadIdx.x < width) partial[threadIdx.x] += partial[threadIdx.x + width];
        __syncthreads();
    }
    const float mean = partial[0] / (float)args.k;
    // not-a-number or infinite rows: no shift (the product then carries them as the fp32 kernels would)
    if (threadIdx.x == 0) args.shift[batch * args.shift_bs + n] = (mean - mean == 0.0f) ? mean : 0.0f;
}

// For 64 rows n, GL2_OUTPUTS outputs from o_begin on and one range of k: `use(j, slice, values)` for every slice of 16 values of p of output
// o_begin + j, lane = row n, wave = every fourth slice (uniform, so that c comes by scalar loads).  b passes through LDS, since a lane's k are contiguous in memory and the lanes' rows are not.
template <typename Use>
__device__ __forceinline__ void gradient_l2_walk(const GradientL2PiecesArgs &args, int n0, int o_begin, int o_end, int first, int last, Use &&use)
{
    __shared__ float tile[GL2_DEPTH * (GL2_ROWS + 1)];
    const GradientL2PrepareArgs &from = args.from;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), batch = blockIdx.z;
    const float *b = from.b + batch * from.b_bs, *c = from.c + batch * from.c_bs;
    const int n = n0 + lane;
    const float shift = n < from.n ? from.shift[batch * from.shift_bs + n] : 0.0f;
    constexpr int LOADS = GL2_ROWS * GL2_DEPTH / GL2_THREADS;
    float v[LOADS];
    auto load = [&](int slice) {
        const int k = slice * BK_TILE_K + lane;
#pragma unroll
        for (int j = 0; j < LOADS; j++) {
            const int row = n0 + wave + 4 * j;
            v[j] = row < from.n && k < from.k ? b[(i64)row * from.b_ld + k] : 0.0f;
        }
    };
    load(first);
    for (int group = first; group < last; group += GL2_DEPTH / BK_TILE_K) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < LOADS; j++) tile[lane * (GL2_ROWS + 1) + wave + 4 * j] = v[j];
        __syncthreads();
        if (group + GL2_DEPTH / BK_TILE_K < last) load(group + GL2_DEPTH / BK_TILE_K);
        const int slice = group + wave;
        if (slice >= last) continue;
        float centred[BK_TILE_K];
#pragma unroll
        for (int e = 0; e < BK_TILE_K; e++) centred[e] = tile[(BK_TILE_K * wave + e) * (GL2_ROWS + 1) + lane] - shift;
        const int k0 = slice * BK_TILE_K;
#pragma unroll
        for (int j = 0; j < GL2_OUTPUTS; j++) {
            if (o_begin + j >= o_end) break;
            const float *c_row = c + (i64)(o_begin + j) * from.c_ld + k0;
            float value[BK_TILE_K];
            if (k0 + BK_TILE_K <= from.k) {
#pragma unroll
                for (int e = 0; e < BK_TILE_K; e++) value[e] = c_row[e] * centred[e];
            } else {
#pragma unroll
                for (int e = 0; e < BK_TILE_K; e++) value[e] = k0 + e < from.k ? c_row[e] * centred[e] : 0.0f;
            }
            use(j, slice, value);
        }
    }
}

__global__ __launch_bounds__(GL2_THREADS) void gradient_l2_pieces_stats(const GradientL2PiecesArgs args)
{
    if ((int)blockIdx.x < args.a_blocks) {
        if ((int)blockIdx.z < args.a_batches && (int)blockIdx.y < args.a.ranges) gram_row_stats_of(args.a, blockIdx.x);
        return;
    }
    __shared__ unsigned shared[4][GL2_OUTPUTS][GL2_ROWS];
    const int groups = (args.from.o + args.outputs - 1) / args.outputs, block = blockIdx.x - args.a_blocks;
    const int n0 = block / groups * GL2_ROWS, o_begin = block % groups * args.outputs, o_end = min(o_begin + args.outputs, args.from.o);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, range = blockIdx.y;
    const int first = range * args.p.slices_per_range, last = min(first + args.p.slices_per_range, args.p.slices);
    if (first >= last) return;
    // as integers: the order of floats without a sign, NaNs above infinity, whose scale they take
    unsigned magnitude[GL2_OUTPUTS] = {};
    gradient_l2_walk(args, n0, o_begin, o_end, first, last, [&](int j, int, const float (&value)[BK_TILE_K]) {
#pragma unroll
        for (int e = 0; e < BK_TILE_K; e++) magnitude[j] = max(magnitude[j], __float_as_uint(value[e]) & 0x7fffffffu);
    });
#pragma unroll
    for (int j = 0; j < GL2_OUTPUTS; j++) shared[wave][j][lane] = magnitude[j];
    __syncthreads();
    const int n = n0 + lane, o = o_begin + wave;
    static_assert(GL2_OUTPUTS == 4, "a wave each");
    if (n < args.from.n && o < o_end)
        args.p.magnitudes[blockIdx.z * args.p.stats_bs + (i64)range * args.p.rows_pad + (i64)o * args.from.n + n] =
            __uint_as_float(max(max(shared[0][wave][lane], shared[1][wave][lane]), max(shared[2][wave][lane], shared[3][wave][lane])));
}

// Bound by the chunks it writes: a wave stores 1 KB of consecutive rows per piece and half.
__global__ __launch_bounds__(GL2_THREADS) void gradient_l2_pieces_split(const GradientL2PiecesArgs args)
{
    if ((int)blockIdx.x < args.a_blocks) {
        if ((int)blockIdx.z < args.a_batches && (int)blockIdx.y < args.a.ranges) gram_f16_split_of(args.a, blockIdx.x);
        return;
    }
    const int groups = (args.from.o + args.outputs - 1) / args.outputs, block = blockIdx.x - args.a_blocks;
    const int n0 = block / groups * GL2_ROWS, o_begin = block % groups * args.outputs, o_end = min(o_begin + args.outputs, args.from.o);
    const int lane = threadIdx.x & 63, range = blockIdx.y, batch = blockIdx.z;
    const int first = range * args.p.slices_per_range, all_slices = args.p.slices + args.p.zero_slices;
    const int last = range == args.p.ranges - 1 ? all_slices : min(first + args.p.slices_per_range, args.p.slices);
    if (first >= last) return;
    const int n = n0 + lane;
    const bool live = n < args.from.n;
    float scale[GL2_OUTPUTS];
#pragma unroll
    for (int j = 0; j < GL2_OUTPUTS; j++) {
        const i64 row = (i64)(o_begin + j) * args.from.n + n;
        float magnitude = 0.0f;
        if (live && o_begin + j < o_end)
            for (int r = 0; r < args.p.ranges; r++)
                magnitude = __uint_as_float(max(__float_as_uint(magnitude),
                                                __float_as_uint(args.p.magnitudes[batch * args.p.stats_bs + (i64)r * args.p.rows_pad + row])));
        const int exponent_field = gram_scale_exponent(magnitude);
        scale[j] = gram_scale(exponent_field);
        if (range == 0 && threadIdx.x < 64 && live && o_begin + j < o_end) args.p.unscale[batch * args.p.unscale_bs + row] = gram_unscale(exponent_field);
    }
    gram_chunk *pieces = args.p.pieces + batch * args.p.pieces_bs;
    gradient_l2_walk(args, n0, o_begin, o_end, first, last, [&](int j, int slice, const float (&value)[BK_TILE_K]) {
        const float s = scale[j];
        unsigned piece[GW_PIECES][8];
#pragma unroll
        for (int q = 0; q < 8; q++) gram_split_pair(value[2 * q] * s, value[2 * q + 1] * s, piece[0][q], piece[1][q]);
        gram_chunk *dst = pieces + (i64)slice * GW_SEGMENTS * args.p.rows_pad + (i64)(o_begin + j) * args.from.n + n;
#pragma unroll
        for (int p = 0; p < GW_PIECES; p++)
#pragma unroll
            for (int half = 0; half < 2; half++)
                if (live)
                    dst[(i64)(2 * p + half) * args.p.rows_pad] =
                        gram_chunk{piece[p][4 * half], piece[p][4 * half + 1], piece[p][4 * half + 2], piece[p][4 * half + 3]};
    });
    // the rows that pad p: by the last workgroup
    if (block == (int)gridDim.x - args.a_blocks - 1) {
        for (int slice = first + (threadIdx.x >> 6); slice < last; slice += 4)
            for (int row = args.p.rows + lane; row < args.p.rows_pad; row += 64)
#pragma unroll
                for (int segment = 0; segment < GW_SEGMENTS; segment++)
                    pieces[((i64)slice * GW_SEGMENTS + segment) * args.p.rows_pad + row] = gram_chunk{0u, 0u, 0u, 0u};
        if (range == 0)
            for (int row = args.p.rows + threadIdx.x; row < args.p.rows_pad; row += GL2_THREADS) args.p.unscale[batch * args.p.unscale_bs + row] = 1.0f;
    }
}

// g = the sum of `parts` partial products, in their order (kmc_matrix_times_coefficients with n_splits)
struct GradientL2SumArgs {
    const float *partial;
    float *sum;
    i64 count, stride;
    int parts;
};

__global__ __launch_bounds__(GL2_THREADS) void gradient_l2_sum_parts(const GradientL2SumArgs args)
{
    const i64 at = (i64)blockIdx.x * GL2_THREADS + threadIdx.x;
    if (at >= args.count) return;
    float total = args.partial[at];
    for (int part = 1; part < args.parts; ++part) total += args.partial[part * args.stride + at];
    args.sum[at] = total;
}

}  // namespace kmc
