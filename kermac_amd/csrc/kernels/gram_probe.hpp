// The sample of the result that is taken in front of a matrix-core launch for squared differences.
//
// |a|^2 + |b|^2 - 2 a.b cancels for pairs of near-duplicate points; a 128 x 128 part of the result that holds
// such a pair is stamped by the matrix-core kernel and recomputed by the direct kernel behind it.  Data that
// has such pairs in every part (points drawn around a few centres, in any order) would pay for both kernels.
// This kernel looks first, at the operands as the caller holds them: BK_SAMPLE_TILES tiles of the result over
// the batch, 16 consecutive rows of each operand from each, their 256 pairs over up to 128 of the k (8 runs of
// 16 spread over the contraction), judged by the matrix-core kernels' own criterion on those k -- near-duplicates
// fail it on any subset of k -- and one of those that a wave finds close there on all k.  A workgroup owns one sampled tile and one word of the result, which it writes
// whole: nothing is accumulated across workgroups, so nothing has to be cleared and the order of the workgroups
// does not matter.  build_kernel.hpp's sample_leaves_it_to_the_direct_kernel turns the words into the decision,
// inside the matrix-core kernels.  The reference has no counterpart (it has no matrix-core path).
#pragma once

#include "build_kernel.hpp"

namespace kmc {

constexpr int GP_RUNS = 8;                     // runs of 16 consecutive k
constexpr int GP_K = GP_RUNS * BK_TILE_K;      // k per pair
constexpr int GP_THREADS = BK_SAMPLE_ROWS * BK_SAMPLE_ROWS;

struct GramProbeArgs {
    const float *a, *b;
    i64 a_ld, a_bs, b_ld, b_bs;
    int a_k_contiguous, b_k_contiguous;
    int m, n, k, l;
    const float *centre; i64 centre_bs;        // as in BuildKernelArgs; the flag sits behind the padded centre
    int centre_pairs;                          // > 0: no flag was stored, these many pairs say it (CentreSums)
    float trust;
    unsigned *sample;                          // [BK_SAMPLE_TILES]
    int queues;                                // that many words behind it are cleared, for the repair launches
};

// Whether subtracting the centre would lower the norms, and with them the error of the expansion, by under 2 %: |c|^2 against the variances.
// sample_mean.hip leaves both as one pair of floats per workgroup of its own behind the centre ([centre, padded][64 unused][pairs]).  Every wave
// adds them up in the same order, so that all of a call decide alike.  Data that are not numbers keep the subtraction (the
// comparison is false), the repair decides.  In place of a launch that stores the answer for all: at 2000 x 2000 x 784 that
// launch was 3 of 55 us on the stream, and one call of the host.  (From the means and variances of all k, by a workgroup with a barrier: 2 us dearer than the launch.)
// (`load` in front of other loads, `needless` behind them, so that its wait is not one more round trip.)
struct CentreSums {
    float norm = 0.0f, spread = 0.0f;

    __device__ __forceinline__ void load(const float *centre, int k, int pairs)
    {
        const float2 *pair = reinterpret_cast<const float2 *>(centre + (k + GRAM_CENTRE_PAD - 1) / GRAM_CENTRE_PAD * GRAM_CENTRE_PAD + GRAM_CENTRE_PAD);
        const int q = threadIdx.x & 63;
        const float2 of = pair[min(q, pairs - 1)];
        norm = q < pairs ? of.x : 0.0f;
        spread = q < pairs ? of.y : 0.0f;
        for (int more = q + 64; more < pairs; more += 64) {
            norm += pair[more].x;
            spread += pair[more].y;
        }
    }
    __device__ __forceinline__ bool needless()
    {
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            norm += __shfl_xor(norm, offset);
            spread += __shfl_xor(spread, offset);
        }
        return norm <= spread * (1.0f / 64.0f);
    }
};

__device__ __forceinline__ float probe_element(const float *x, i64 ld, int k_contiguous, int row, int k)
{
    return k_contiguous ? x[(i64)row * ld + k] : x[(i64)k * ld + row];
}

// Sampled tile `tile`; the workgroup has GP_THREADS threads.
__device__ __forceinline__ void gram_probe_tile(const GramProbeArgs &args, int tile)
{
    __shared__ float rows_a[GP_K][BK_SAMPLE_ROWS + 1];      // + 1: no bank is hit twice whichever way the rows are loaded
    __shared__ float rows_b[GP_K][BK_SAMPLE_ROWS + 1];
    __shared__ unsigned below_in_tile;
    const int t = threadIdx.x;
    if (t == 0) below_in_tile = 0u;
    if (tile == 0 && t < args.queues) args.sample[BK_SAMPLE_TILES + t] = 0u;
    unsigned h = (unsigned)tile * 2654435761u + 0x9e3779b9u;
    h ^= h >> 15; h *= 0x846ca68bu; h ^= h >> 13;
    const int batch = (int)(h % (unsigned)args.l);
    h = h * 0x7feb352du + 0x1234567u; h ^= h >> 16;
    const int m0 = (int)(h % (unsigned)((args.m + BK_TILE_M - 1) / BK_TILE_M)) * BK_TILE_M + (int)((h >> 20) & 7u) * BK_SAMPLE_ROWS;
    h = h * 0x7feb352du + 0x1234567u; h ^= h >> 16;
    const int n0 = (int)(h % (unsigned)((args.n + BK_TILE_N - 1) / BK_TILE_N)) * BK_TILE_N + (int)((h >> 20) & 7u) * BK_SAMPLE_ROWS;

    const float *a = args.a + batch * args.a_bs, *b = args.b + batch * args.b_bs;
    const int k_padded = (args.k + GRAM_CENTRE_PAD - 1) / GRAM_CENTRE_PAD * GRAM_CENTRE_PAD;
    const float *centre = args.centre ? args.centre + batch * args.centre_bs : nullptr;
    CentreSums sums;
    if (centre && args.centre_pairs) sums.load(centre, args.k, args.centre_pairs);
    else if (centre && centre[k_padded] == 0.0f) centre = nullptr;        // the flag: this batch entry is taken as it is

    // Lane t fetches, for each run, one value of a and one of b: 16 rows x 16 k per run, along whichever
    // direction is contiguous.  Rows beyond the panel repeat its last row (a pair counted twice biases nothing
    // that matters here); k beyond the contraction contributes nothing.
    const int slices = (args.k + BK_TILE_K - 1) / BK_TILE_K;
    const int runs = slices < GP_RUNS ? slices : GP_RUNS;
    const int row_a = args.a_k_contiguous ? t / BK_TILE_K : t % BK_SAMPLE_ROWS, k_a = args.a_k_contiguous ? t % BK_TILE_K : t / BK_SAMPLE_ROWS;
    const int row_b = args.b_k_contiguous ? t / BK_TILE_K : t % BK_SAMPLE_ROWS, k_b = args.b_k_contiguous ? t % BK_TILE_K : t / BK_SAMPLE_ROWS;
    const int m = min(m0 + row_a, args.m - 1), n = min(n0 + row_b, args.n - 1);
    // first k of run r: floor(r slices / runs) slices on
    auto first_of = [&](int r) { return (slices < GP_RUNS ? r : (int)((i64)r * slices / GP_RUNS)) * BK_TILE_K; };
    // Loads of what does not exist go to the last k that does and are dropped, and the centre is loaded behind all of them: with a
    // branch per load each would be waited for by itself (2000 x 2000 x 784, where the sample is taken beside gram_rows_once: a call 49.1 -> 46.7 us;
    // in front of 30000 x 30000 x 1024 the call is the same within the 0.3 % by which its runs differ).
    float va[GP_RUNS], vb[GP_RUNS];
#pragma unroll
    for (int r = 0; r < GP_RUNS; r++) {
        va[r] = probe_element(a, args.a_ld, args.a_k_contiguous, m, min(first_of(r) + k_a, args.k - 1));
        vb[r] = probe_element(b, args.b_ld, args.b_k_contiguous, n, min(first_of(r) + k_b, args.k - 1));
    }
    if (centre && args.centre_pairs && sums.needless()) centre = nullptr;
    if (centre) {
#pragma unroll
        for (int r = 0; r < GP_RUNS; r++) {
            va[r] -= centre[min(first_of(r) + k_a, args.k - 1)];
            vb[r] -= centre[min(first_of(r) + k_b, args.k - 1)];
        }
    }
#pragma unroll
    for (int r = 0; r < GP_RUNS; r++) {
        va[r] = r < runs && first_of(r) + k_a < args.k ? va[r] : 0.0f;
        vb[r] = r < runs && first_of(r) + k_b < args.k ? vb[r] : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < GP_RUNS; r++) {
        rows_a[r * BK_TILE_K + k_a][row_a] = va[r];
        rows_b[r * BK_TILE_K + k_b][row_b] = vb[r];
    }
    __syncthreads();
    const int i = t % BK_SAMPLE_ROWS, j = t / BK_SAMPLE_ROWS;      // this lane's pair: row i of a, row j of b
    float d2 = 0.0f, norms = 0.0f;
#pragma unroll 8
    for (int q = 0; q < GP_K; q++) {
        const float x = rows_a[q][i], y = rows_b[q][j];
        d2 += (y - x) * (y - x);
        norms += x * x + y * y;
    }
    const unsigned long long close = __ballot(!(d2 >= args.trust * norms));
    unsigned below = (unsigned)__popcll(close);
    if (below > 0u && slices > GP_RUNS) {
        // A pair that is close on these k need not be on all of them: where a few k hold most of every distance, as features of very different scales do, the others
        // say nothing.  The wave takes the first of its close pairs, over all k, for all of them.  (Calls of such data that were mistaken for
        // near-duplicates, without / with this, us and the error's 2-norm: 390 x 448 x 1552 twice, scales over 3 decades, 550 / 89, 6.3e-7 / 4.0e-8; 734 x 3776 x 3805 times 10
        // coefficients, 6 decades, 1258 / 227, 2.0e-6 / 1.7e-7; 7358 x 1472 x 426, 8 decades, 272 / 76.  Near-duplicates: 2000 x 2000 x 784 265 / 265, 3000 x 3000 x 3072 1644 / 1649;
        // with all pairs of such a tile looked at through LDS, 64 k at a time, 287 and 1745.)
        const int pair = (t & ~63) + __builtin_ctzll(close);
        const int pair_m = min(m0 + pair % BK_SAMPLE_ROWS, args.m - 1), pair_n = min(n0 + pair / BK_SAMPLE_ROWS, args.n - 1);
        d2 = norms = 0.0f;
#pragma unroll 4
        for (int k = t & 63; k < args.k; k += 64) {
            const float at = centre ? centre[k] : 0.0f;
            const float x = probe_element(a, args.a_ld, args.a_k_contiguous, pair_m, k) - at, y = probe_element(b, args.b_ld, args.b_k_contiguous, pair_n, k) - at;
            d2 += (y - x) * (y - x);
            norms += x * x + y * y;
        }
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            d2 += __shfl_xor(d2, offset);
            norms += __shfl_xor(norms, offset);
        }
        if (d2 >= args.trust * norms) below = 0u;
    }
    if ((t & 63) == 0 && below > 0u) atomicAdd(&below_in_tile, below);
    __syncthreads();
    if (t == 0) args.sample[tile] = below_in_tile | (below_in_tile > 0u ? 0x10000u : 0u);
}

}  // namespace kmc
