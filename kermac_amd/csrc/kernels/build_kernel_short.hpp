// The direct kernel for short contractions: launches that are bound by the stores of the result.
//
// build_kernel (build_kernel.hpp) walks k in slices of 16 through LDS and lets a workgroup load, compute and store one tile of 128 x
// 128 after the other, which leaves the memory idle while it loads and computes: 10000 x 10000 of K = 6 take 105 us, 3.8 TB/s,
// where filling the same 400 MB takes 58 (6.9 TB/s).  Here a lane holds all k of its 4 rows m in registers and
// goes through columns n, so that a wave stores 1 KB of consecutive m per column, one behind the other and with nothing
// to wait for but the memory.  The values of b for the workgroup's columns are staged in LDS once, zero beyond K, and
// read as broadcasts (all lanes the same 16 bytes), whatever their storage.
//
// What stores cost depends on whether they fill whole lines (stores alone, 10000 x 10000 in pieces of 1 KB: 4.7 TB/s where
// rows start in the middle of a line of 128 bytes, 6.3 where they do not).  Columns start at any multiple of 4 bytes (ld is
// the caller's), but columns n that are `classes` apart (1, 2, 4 .. 32) start at the same place in a line: a workgroup takes columns of
// one class and shifts its rows m, so that every store of a wave is 1 KB that begins on a line.
//
// Results are those of build_kernel bit for bit: every element sums its terms over k in the same order, and zeros
// beyond K add nothing for the inner terms that this kernel has.  A set against itself is computed in full: its
// arithmetic is cheaper than a second, mirrored store, and equal bits on both sides follow from the terms.
#pragma once

#include "build_kernel.hpp"

namespace kmc {

constexpr int BKT_WAVES = 4;
constexpr int BKT_TILE_M = 256;                      // 64 lanes x 4 rows, the same for all waves
constexpr int BKT_QUAD = 4;                          // columns n that a wave has under way
constexpr int BKT_COLUMNS = BKT_WAVES * BKT_QUAD;    // columns per round of the workgroup ...
constexpr int BKT_MAX_ROUNDS = 8;                    // ... and rounds
constexpr int BKT_PITCH = BKT_TILE_M + 4;            // of a k-row in LDS
constexpr int BKT_CHUNK = 8;                         // k of an operand with k contiguous, staged at a time
constexpr int BKT_LINE = 32;                         // floats

// acc0 and acc1 += inner(b0 and b1, a) for four rows: eight independent subtractions, then eight independent accumulations, as
// row_abs_diff and row_square_diff of build_kernel.hpp (left to itself the compiler sinks each row's whole chain into the
// branches of the epilogue, one after the other)
template <int INNER_OP, int INNER_POW>
__device__ __forceinline__ void short_pair(float (&acc0)[4], float (&acc1)[4], const float (&fa)[4], float b0, float b1, float diff_sign)
{
    if constexpr (INNER_OP == OP_DIFF && (INNER_POW == POW_ABS || INNER_POW == POW_SQUARE)) {
        float t0, t1, t2, t3, t4, t5, t6, t7;
#define KMC_SHORT_OPERANDS \
        : "+v"(acc0[0]), "+v"(acc0[1]), "+v"(acc0[2]), "+v"(acc0[3]), "+v"(acc1[0]), "+v"(acc1[1]), "+v"(acc1[2]), "+v"(acc1[3]), \
          "=&v"(t0), "=&v"(t1), "=&v"(t2), "=&v"(t3), "=&v"(t4), "=&v"(t5), "=&v"(t6), "=&v"(t7) \
        : "v"(fa[0]), "v"(fa[1]), "v"(fa[2]), "v"(fa[3]), "v"(b0), "v"(b1)
        if constexpr (INNER_POW == POW_ABS) {
            asm volatile("v_sub_f32 %8, %20, %16\n\tv_sub_f32 %9, %20, %17\n\tv_sub_f32 %10, %20, %18\n\tv_sub_f32 %11, %20, %19\n\t"
                         "v_sub_f32 %12, %21, %16\n\tv_sub_f32 %13, %21, %17\n\tv_sub_f32 %14, %21, %18\n\tv_sub_f32 %15, %21, %19\n\t"
                         "v_add_f32 %0, |%8|, %0\n\tv_add_f32 %1, |%9|, %1\n\tv_add_f32 %2, |%10|, %2\n\tv_add_f32 %3, |%11|, %3\n\t"
                         "v_add_f32 %4, |%12|, %4\n\tv_add_f32 %5, |%13|, %5\n\tv_add_f32 %6, |%14|, %6\n\tv_add_f32 %7, |%15|, %7"
                         KMC_SHORT_OPERANDS);
        } else {
            asm volatile("v_sub_f32 %8, %20, %16\n\tv_sub_f32 %9, %20, %17\n\tv_sub_f32 %10, %20, %18\n\tv_sub_f32 %11, %20, %19\n\t"
                         "v_sub_f32 %12, %21, %16\n\tv_sub_f32 %13, %21, %17\n\tv_sub_f32 %14, %21, %18\n\tv_sub_f32 %15, %21, %19\n\t"
                         "v_fmac_f32 %0, %8, %8\n\tv_fmac_f32 %1, %9, %9\n\tv_fmac_f32 %2, %10, %10\n\tv_fmac_f32 %3, %11, %11\n\t"
                         "v_fmac_f32 %4, %12, %12\n\tv_fmac_f32 %5, %13, %13\n\tv_fmac_f32 %6, %14, %14\n\tv_fmac_f32 %7, %15, %15"
                         KMC_SHORT_OPERANDS);
        }
#undef KMC_SHORT_OPERANDS
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            acc0[i] += inner_term<INNER_OP, INNER_POW>(fa[i], b0, 0.0f, diff_sign);
            acc1[i] += inner_term<INNER_OP, INNER_POW>(fa[i], b1, 0.0f, diff_sign);
        }
        asm volatile("" : "+v"(acc0[0]), "+v"(acc0[1]), "+v"(acc0[2]), "+v"(acc0[3]), "+v"(acc1[0]), "+v"(acc1[1]), "+v"(acc1[2]), "+v"(acc1[3]));
    }
}

template <int INNER_OP, int INNER_POW, int DEPTH>
__global__ __launch_bounds__(BK_THREADS) void build_kernel_short(const BuildKernelArgs args, int load_a, int load_b, int rounds, int classes)
{
    __shared__ __attribute__((aligned(16))) float lds_b[BKT_MAX_ROUNDS * BKT_COLUMNS * DEPTH];
    __shared__ __attribute__((aligned(16))) float staged[BKT_CHUNK * BKT_PITCH];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int batch = blockIdx.z;
    // columns n = n_first + classes * j, j = 0 .. columns - 1
    const int columns = rounds * BKT_COLUMNS;
    const int n_first = (int)(blockIdx.y / classes) * columns * classes + (int)(blockIdx.y % classes);
    if (n_first >= args.n) return;
    float *const c_batch = args.c + batch * args.c_bs;
    // floats between the start of a line and C(0, n)
    const int shift = (int)((reinterpret_cast<unsigned long long>(c_batch) / 4 + (unsigned long long)n_first * (unsigned long long)args.c_ld) % BKT_LINE);
    // Rows are added up without a sign, and compared with differences of M: for M near 2^31 those beyond it are negative, not small.
    // The last tile exists for some shifts only.  Tiles are dealt out in another order for every group of columns, or it would fall to
    // the same of the 8 XCDs each time and leave them idle.
    const unsigned m_tile = (blockIdx.x + blockIdx.y) % gridDim.x;
    if ((i64)m_tile * BKT_TILE_M - shift >= args.m) return;
    const int m0 = (int)(m_tile * BKT_TILE_M - (unsigned)shift);
    auto row_at = [m0](int at) { return (int)((unsigned)m0 + (unsigned)at); };
    const int m_first = row_at(4 * lane);
    const bool whole = m0 >= 0 && m0 <= args.m - BKT_TILE_M, whole_quad = m_first >= 0 && m_first <= args.m - 4;

    const float *b = args.b + batch * args.b_bs;
    const bool b_rows = load_b == LOAD_ROW_VEC || load_b == LOAD_ROW_SCALAR;
    for (int e = tid; e < columns * DEPTH; e += BK_THREADS) {
        // consecutive lanes along what is contiguous
        const int j = b_rows ? e / DEPTH : e % columns, k = b_rows ? e % DEPTH : e / columns;
        const i64 n = n_first + (i64)classes * j;
        lds_b[j * DEPTH + k] = n < args.n && k < args.k ? b[b_rows ? n * args.b_ld + k : k * args.b_ld + n] : 0.0f;
    }
    float a[DEPTH][4];
    const float *from = args.a + batch * args.a_bs;
    if (load_a == LOAD_ROW_VEC || load_a == LOAD_ROW_SCALAR) {
        // k contiguous: 8 k of all rows at a time through LDS, lanes along k (a lane's own loads, rows apart, would touch a line each)
        constexpr int ROWS = BK_THREADS / BKT_CHUNK, LOADS = BKT_TILE_M / ROWS;
        const int kk = tid % BKT_CHUNK, row = tid / BKT_CHUNK;
#pragma unroll
        for (int k0 = 0; k0 < DEPTH; k0 += BKT_CHUNK) {
            float v[LOADS];
#pragma unroll
            for (int j = 0; j < LOADS; j++) {
                const int m = row_at(j * ROWS + row);
                v[j] = m >= 0 && m < args.m && k0 + kk < args.k ? from[(i64)m * args.a_ld + k0 + kk] : 0.0f;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < LOADS; j++) staged[kk * BKT_PITCH + j * ROWS + row] = v[j];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < BKT_CHUNK && k0 + j < DEPTH; j++) {
                const float4 x = *reinterpret_cast<const float4 *>(staged + j * BKT_PITCH + 4 * lane);
                a[k0 + j][0] = x.x; a[k0 + j][1] = x.y; a[k0 + j][2] = x.z; a[k0 + j][3] = x.w;
            }
        }
    } else if (load_a == LOAD_COL_VEC && shift % 4 == 0 && whole) {
#pragma unroll
        for (int k = 0; k < DEPTH; k++) {
            const float4 v = k < args.k ? *reinterpret_cast<const float4 *>(from + (i64)k * args.a_ld + m_first) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            a[k][0] = v.x; a[k][1] = v.y; a[k][2] = v.z; a[k][3] = v.w;
        }
    } else {
        // m contiguous, but not where a lane could load its 4 rows at once: 8 k of all rows at a time through LDS, lanes along m.  Loads of what does
        // not exist go to the last row and k that do, and are dropped: with a branch for each they would be waited for one by one
        const int m = row_at(tid);
        const bool live = m >= 0 && m < args.m;
        const float *column = from + min(max(m, 0), args.m - 1);
#pragma unroll
        for (int k0 = 0; k0 < DEPTH; k0 += BKT_CHUNK) {
            float v[BKT_CHUNK];
#pragma unroll
            for (int j = 0; j < BKT_CHUNK && k0 + j < DEPTH; j++) v[j] = column[(i64)min(k0 + j, args.k - 1) * args.a_ld];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < BKT_CHUNK && k0 + j < DEPTH; j++) staged[j * BKT_PITCH + tid] = live && k0 + j < args.k ? v[j] : 0.0f;
            __syncthreads();
#pragma unroll
            for (int j = 0; j < BKT_CHUNK && k0 + j < DEPTH; j++) {
                const float4 x = *reinterpret_cast<const float4 *>(staged + j * BKT_PITCH + 4 * lane);
                a[k0 + j][0] = x.x; a[k0 + j][1] = x.y; a[k0 + j][2] = x.z; a[k0 + j][3] = x.w;
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
    const float diff_sign = args.diff_sign, epsilon = args.epsilon;
    __syncthreads();

    for (int round = 0; round < rounds; round++) {
        // this wave's columns j: the waves side by side
        const int j_first = round * BKT_COLUMNS + wave;
        if (n_first + (i64)classes * j_first >= args.n) break;
        float acc[BKT_QUAD][4];
#pragma unroll
        for (int c = 0; c < BKT_QUAD; c++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[c][i] = 0.0f;
#pragma unroll
        for (int k = 0; k < DEPTH; k += 4) {
            float fb[BKT_QUAD][4];
#pragma unroll
            for (int c = 0; c < BKT_QUAD; c++) {
                const float4 v = *reinterpret_cast<const float4 *>(lds_b + (j_first + BKT_WAVES * c) * DEPTH + k);
                fb[c][0] = v.x; fb[c][1] = v.y; fb[c][2] = v.z; fb[c][3] = v.w;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
#pragma unroll
                for (int c = 0; c < BKT_QUAD; c += 2)
                    short_pair<INNER_OP, INNER_POW>(acc[c], acc[c + 1], a[k + j], fb[c][j], fb[c + 1][j], diff_sign);
            }
        }
        auto for_each = [&](auto &&f) {
#pragma unroll
            for (int c = 0; c < BKT_QUAD; c++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[c][i] = f(acc[c][i]);
        };
        switch (outer_power) {
        case POW_ABS: for_each([](float v) { return __builtin_fabsf(v); }); break;
        case POW_SQUARE: for_each([](float v) { return v * v; }); break;
        case POW_SQRT: for_each([](float v) { return __builtin_amdgcn_sqrtf(v); }); break;
        case POW_POW: for_each([p_outer](float v) { return exp2f(p_outer * log2f(v)); }); break;
        default: break;
        }
        if (kernel_type != KERNEL_NONE) for_each([epsilon, neg_gamma](float v) { return expf((v < epsilon ? 0.0f : v) * neg_gamma); });
#pragma unroll
        for (int c = 0; c < BKT_QUAD; c++) {
            const i64 n = n_first + (i64)classes * (j_first + BKT_WAVES * c);
            if (n >= args.n) break;
            if (regularize) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if ((unsigned)args.reg_off_x + (unsigned)m_first + i == (unsigned)args.reg_off_y + (unsigned)n) acc[c][i] = 1.0f + regularization;
            }
            float *to = c_batch + n * args.c_ld + m_first;
            if (whole || whole_quad) {
                *reinterpret_cast<float4 *>(to) = make_float4(acc[c][0], acc[c][1], acc[c][2], acc[c][3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (row_at(4 * lane + i) >= 0 && row_at(4 * lane + i) < args.m) to[i] = acc[c][i];
            }
        }
    }
}

}  // namespace kmc
