// The direct kernel for results of few tiles: build_kernel.hpp in tiles of 64 x 64 instead of 128 x 128.
//
// A result of 1024 x 1024 is 64 tiles of 128 x 128: a quarter of the CUs work, each lane through 64 results of its own, and what
// stands in front of and behind the walk (first loads, epilogue, stores) is hidden by nothing.  Here a workgroup of 8 waves holds a
// tile of 64 x 64 and a lane 4 x 2 results, so that the same result is four times the workgroups at an eighth of the
// serial work per lane.  LDS then feeds a third as many terms per byte, which is why large results stay with the other
// tile.
//
// Up to 256 of these tiles a workgroup has its CU to itself, and two waves on a SIMD are what hides the reads from LDS: with 4 waves of 4 x 4
// results per lane, one on each SIMD, a term of k took 0.11 us where it now takes 0.06 (LDS alone 0.04).  4 / 8 waves, kernels back to back, us:
// 1024 x 1024 at K = 64 p = 1 13.9 / 8.0, p = 2 13.3 / 8.1, p = 1.3 24.8 / 18.5, at K = 400 p = 1 51 / 28, p = 1.3 117 / 89, |x|^4 61 / 34; 64 x 64 x 16
// 6.3 / 4.4; 1200 x 1200 x 200 (361 tiles) p = 1 31.2 / 23.8; 2048 x 2048 x 128 (1024, four workgroups per CU) 31.1 / 28.3, |x|^4 42.9 / 37.7;
// 192 x 128 x 128 x 64 18.3 / 15.5; no size of this kernel's range was slower.
//
// The terms, their order in every sum and the epilogue are those of build_kernel: the bits are the same.  Slices of 32 k, double
// buffered.  The loaders are chosen at run time (uniform branches in front of a slice's loads): few launches are worth sixteen instantiations.  A
// symmetric result is computed whole.
#pragma once

#include "build_kernel.hpp"

namespace kmc {

constexpr int BKS_TILE = 64;
constexpr int BKS_DEPTH = 32;
constexpr int BKS_PITCH = BKS_TILE + 4;
constexpr int BKS_THREADS = 512;

// One operand's share of a 64 x 32 slice: 4 consecutive floats per lane.
struct SmallLoader {
    const float *base;      // row 0 of the tile, k = 0
    i64 ld;
    int rows, mode, tid;    // rows that exist from the tile's first on

    // this lane's first row and k, relative to the tile and the slice
    __device__ __forceinline__ bool k_runs() const { return mode == LOAD_ROW_VEC || mode == LOAD_ROW_SCALAR; }
    __device__ __forceinline__ int row() const { return k_runs() ? tid >> 3 : (tid & 15) * 4; }
    __device__ __forceinline__ int k_row() const { return k_runs() ? (tid & 7) * 4 : tid >> 4; }

    __device__ __forceinline__ float4 load(int k0, int k) const
    {
        const bool vec = mode == LOAD_COL_VEC || mode == LOAD_ROW_VEC;
        const int at = k0 + k_row();
        const float4 nothing = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (k_runs()) return row() < rows ? load4_guarded(base + (i64)row() * ld + at, k - at, vec) : nothing;
        return at < k ? load4_guarded(base + (i64)at * ld + row(), rows - row(), vec) : nothing;
    }

    __device__ __forceinline__ void store(float *slice, const float4 &r) const
    {
        float *to = slice + k_row() * BKS_PITCH + row();
        if (k_runs()) {
            to[0] = r.x; to[BKS_PITCH] = r.y; to[2 * BKS_PITCH] = r.z; to[3 * BKS_PITCH] = r.w;
        } else {
            *reinterpret_cast<float4 *>(to) = r;
        }
    }
};

template <int INNER_OP, int INNER_POW>
__global__ __launch_bounds__(BKS_THREADS) void build_kernel_small(const BuildKernelArgs args, int load_a, int load_b, int tiles_n)
{
    __shared__ __attribute__((aligned(16))) float lds_a[2][BKS_DEPTH * BKS_PITCH];
    __shared__ __attribute__((aligned(16))) float lds_b[2][BKS_DEPTH * BKS_PITCH];
    const int tid = threadIdx.x, batch = blockIdx.y;
    const int m0 = blockIdx.x / tiles_n * BKS_TILE, n0 = blockIdx.x % tiles_n * BKS_TILE;
    const int tx = tid & 15, ty = tid >> 4;
    float p_inner = 0.0f;
    if (INNER_POW == POW_POW) p_inner = args.p_inner ? args.p_inner[batch * args.p_inner_bs] : args.p_inner_value;

    auto first = [](int mode, i64 row, i64 ld) { return mode == LOAD_ROW_VEC || mode == LOAD_ROW_SCALAR ? row * ld : row; };
    const SmallLoader from_a{args.a + batch * args.a_bs + first(load_a, m0, args.a_ld), args.a_ld, args.m - m0, load_a, tid};
    const SmallLoader from_b{args.b + batch * args.b_bs + first(load_b, n0, args.b_ld), args.b_ld, args.n - n0, load_b, tid};

    float acc[2][4];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[j][i] = 0.0f;
    if (args.k > 0) {
        float4 stage_a = from_a.load(0, args.k), stage_b = from_b.load(0, args.k);
        from_a.store(lds_a[0], stage_a);
        from_b.store(lds_b[0], stage_b);
        __syncthreads();
        for (int k0 = 0, cur = 0; k0 < args.k; k0 += BKS_DEPTH, cur ^= 1) {
            const bool more = k0 + BKS_DEPTH < args.k;
            if (more) {
                stage_a = from_a.load(k0 + BKS_DEPTH, args.k);
                stage_b = from_b.load(k0 + BKS_DEPTH, args.k);
            }
            const float *row_a = lds_a[cur] + 4 * tx, *row_b = lds_b[cur] + 2 * ty;
            // padding of k up to a multiple of 16 takes part, as in the other tile
            const int depth = min(BKS_DEPTH, (args.k - k0 + BK_TILE_K - 1) / BK_TILE_K * BK_TILE_K);
#pragma unroll 4
            for (int kk = 0; kk < depth; kk++) {
                const float4 va = *reinterpret_cast<const float4 *>(row_a + kk * BKS_PITCH);
                const float2 vb = *reinterpret_cast<const float2 *>(row_b + kk * BKS_PITCH);
                const float fa[4] = {va.x, va.y, va.z, va.w}, fb[2] = {vb.x, vb.y};
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        if (INNER_OP == OP_DIFF && INNER_POW == POW_SQUARE) {
                            const float d = fb[j] - fa[i];
                            acc[j][i] = __builtin_fmaf(d, d, acc[j][i]);
                        } else {
                            acc[j][i] += inner_term<INNER_OP, INNER_POW>(fa[i], fb[j], p_inner, args.diff_sign);
                        }
                    }
            }
            if (more) {
                from_a.store(lds_a[cur ^ 1], stage_a);
                from_b.store(lds_b[cur ^ 1], stage_b);
                __syncthreads();
            }
        }
    }

    const int outer_power = args.outer_power, kernel_type = args.kernel_type;
    float p_outer = 0.0f, neg_gamma = 0.0f, regularization = 0.0f;
    if (outer_power == POW_POW) p_outer = args.p_outer ? args.p_outer[batch * args.p_outer_bs] : args.p_outer_value;
    if (kernel_type != KERNEL_NONE) {
        neg_gamma = kernel_neg_gamma(kernel_type, args.bandwidth ? args.bandwidth[batch * args.bandwidth_bs] : args.bandwidth_value);
        regularization = args.regularization ? args.regularization[batch * args.regularization_bs] : args.regularization_value;
    }
    const bool regularize = kernel_type != KERNEL_NONE && regularization != 0.0f;
    const int m = m0 + 4 * tx;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int n = n0 + 2 * ty + j;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = epilogue_value(acc[j][i], outer_power, kernel_type, p_outer, neg_gamma, args.epsilon);
            if (regularize && args.reg_off_x + m + i == args.reg_off_y + n) v[i] = 1.0f + regularization;
        }
        if (n >= args.n) continue;
        float *to = args.c + batch * args.c_bs + (i64)n * args.c_ld + m;
        if (args.c_vec && m + 3 < args.m) {
            *reinterpret_cast<float4 *>(to) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (m + i < args.m) to[i] = v[i];
        }
    }
}

}  // namespace kmc
