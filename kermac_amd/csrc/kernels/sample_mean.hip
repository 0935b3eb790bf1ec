// kmc_sample_mean: the mean point of (a sample of) the rows of an operand panel, the
// centre that the matrix-core kernels subtract from both operands while they stage them
// (|a|^2 + |b|^2 - 2 a.b cancels in proportion to the norms, and the norms that matter are
// those around the centre).  Up to 4096 rows are averaged exactly as given; of a longer panel
// 16 runs of 256 consecutive rows, evenly spaced from the first row to the last.  The sums run
// in a fixed order, so the same panel always gives the same centre.  The result is padded with
// zeros to a multiple of GRAM_CENTRE_PAD floats, as the kernels expect it, and followed by a
// flag: 1 when subtracting the centre is worth its cost, 0 when the centre is so close to the
// origin, measured against the spread of the sampled rows around it (|c|^2 <= spread^2 / 64), that
// the norms -- and with them the cancellation -- would change by less than 2 %.  The matrix-core
// kernels then skip the subtraction for that batch entry.  Layout per batch entry:
// [centre, padded][flag, 63 unused floats][variance per k, padded] = 2 * padded + 64 floats.
#include <hip/hip_runtime.h>

#include "../host/host_common.hpp"
#include "build_kernel.hpp"
#include "launch.hpp"

namespace kmc {

struct SampleMeanArgs {
    const float *x; i64 ld, bs;
    int rows, k, k_padded;
    float *mean; i64 mean_bs;
    int pairs;           // 1: of |mean|^2 and the variances one pair of sums per workgroup, in place of the variances (CentreSums)
    int samples, run;    // rows that are averaged; of a longer panel they are samples / run runs of `run` consecutive rows
    int step;            // > 0: rows from the start of a run to that of the next; 0: the runs reach from the first row to the last
};

// mean of squares minus square of mean, per k, goes behind the centre and its flag
__device__ __forceinline__ float *variance_of(const SampleMeanArgs &args, int batch)
{
    return args.mean + batch * args.mean_bs + args.k_padded + GRAM_CENTRE_PAD;
}

constexpr int SM_MAX_SAMPLES = 4096;
constexpr int SM_RUN = 256;
constexpr int SM_COLUMNS_PER_WORKGROUP = 4;      // sample_mean_columns

__device__ __forceinline__ i64 sampled_row(const SampleMeanArgs &args, int s)
{
    if (args.rows <= args.samples) return s;
    if (args.step) return (i64)(s / args.run) * args.step + s % args.run;
    const int run = s / args.run;
    return (i64)run * (args.rows - args.run) / (args.samples / args.run - 1) + (s - run * args.run);
}

// k contiguous (row-major panel): a workgroup owns SPAN k, 1024 / SPAN groups of SPAN lanes share the rows, and a lane has eight
// rows under way at once (eight sums per lane, added in a fixed order at the end): the panel's rows lie K floats apart, so the
// time of a single panel is that of the loads' latency, not of their bytes, and shrinks with more groups: SPAN 16 instead of 64 is 64
// groups instead of 16 and four times as many workgroups (K = 784, 4096 rows: 43 -> 16 us; 2000 rows 14 -> 7).  A batch that
// fills the chip with workgroups of SPAN 64 is bound by what it loads and adds up, which runs of 64 k do better, and up to 128 rows are
// one round trip either way.  SPAN 16 / SPAN 64, us, by workgroups of SPAN 64: 32 of them 4.7 / 7.8 for 1000 rows, 14 / 24 for 4096; 64
// 4.8 / 7.8 and 22 / 27; 96 10.4 / 8.0 and 33 / 27; 128 12 / 8.8 and 41 / 28; 512 40 / 21 and 166 / 98; the sample of 30000 rows, 16
// runs far apart, 96 34 / 44, 128 42 / 44, 156 48 / 46, 512 170 / 96; 100 rows 3.8 / 3.2 in 16 workgroups, 11 / 4 in 512.
constexpr int SM_ROW_THREADS = 1024;
constexpr int SM_ROW_UNROLL = 8;
constexpr int SM_ROW_WIDE_MIN_WORKGROUPS = 96;              // of SPAN 64, all rows averaged
constexpr int SM_ROW_WIDE_MIN_WORKGROUPS_SAMPLED = 144;     // ... and where they are a sample
constexpr int SM_ROW_WIDE_MAX_FEW_ROWS = 128;

template <int SPAN>
__global__ __launch_bounds__(SM_ROW_THREADS) void sample_mean_rows(const SampleMeanArgs args)
{
    constexpr int GROUPS = SM_ROW_THREADS / SPAN;
    __shared__ float partial[SM_ROW_THREADS / 64][SPAN];
    __shared__ float partial_squares[SM_ROW_THREADS / 64][SPAN];
    const int kk = threadIdx.x % SPAN, group = threadIdx.x / SPAN;
    const int k = blockIdx.x * SPAN + kk;
    const float *x = args.x + blockIdx.y * args.bs;
    float sum[SM_ROW_UNROLL], squares[SM_ROW_UNROLL];
#pragma unroll
    for (int u = 0; u < SM_ROW_UNROLL; ++u) sum[u] = squares[u] = 0.0f;
    if (k < args.k) {
        for (int first = group; first < args.samples; first += SM_ROW_UNROLL * GROUPS) {
            float v[SM_ROW_UNROLL];
#pragma unroll
            for (int u = 0; u < SM_ROW_UNROLL; ++u) {
                const int s = first + u * GROUPS;
                v[u] = s < args.samples ? x[sampled_row(args, s) * args.ld + k] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < SM_ROW_UNROLL; ++u) {
                sum[u] += v[u];
                squares[u] += v[u] * v[u];
            }
        }
    }
    float mine = 0.0f, mine_squares = 0.0f;
#pragma unroll
    for (int u = 0; u < SM_ROW_UNROLL; ++u) {
        mine += sum[u];
        mine_squares += squares[u];
    }
    // the groups of a wave first, then the waves in their order
#pragma unroll
    for (int offset = SPAN; offset < 64; offset <<= 1) {
        mine += __shfl_xor(mine, offset);
        mine_squares += __shfl_xor(mine_squares, offset);
    }
    if ((threadIdx.x & 63) < SPAN) {
        partial[threadIdx.x >> 6][kk] = mine;
        partial_squares[threadIdx.x >> 6][kk] = mine_squares;
    }
    __syncthreads();
    if (group == 0) {
        float total = 0.0f, total_squares = 0.0f;
#pragma unroll
        for (int w = 0; w < SM_ROW_THREADS / 64; ++w) {
            total += partial[w][kk];
            total_squares += partial_squares[w][kk];
        }
        const bool live = k < args.k && args.samples > 0;
        const float mean = live ? total / (float)args.samples : 0.0f;
        const float variance = live ? fmaxf(total_squares / (float)args.samples - mean * mean, 0.0f) : 0.0f;
        if (k < args.k_padded) args.mean[blockIdx.y * args.mean_bs + k] = mean;
        if (args.pairs) {
            float norm = mean * mean, spread = variance;
#pragma unroll
            for (int offset = SPAN / 2; offset > 0; offset >>= 1) {
                norm += __shfl_xor(norm, offset);
                spread += __shfl_xor(spread, offset);
            }
            if (kk == 0) reinterpret_cast<float2 *>(variance_of(args, blockIdx.y))[blockIdx.x] = make_float2(norm, spread);
        } else if (k < args.k_padded) {
            variance_of(args, blockIdx.y)[k] = variance;
        }
    }
}

// rows contiguous (K-major panel): a wave owns one k, its lanes take consecutive rows.
__global__ __launch_bounds__(256) void sample_mean_columns(const SampleMeanArgs args)
{
    __shared__ float norms[SM_COLUMNS_PER_WORKGROUP], spreads[SM_COLUMNS_PER_WORKGROUP];
    static_assert(SM_COLUMNS_PER_WORKGROUP == 4, "a wave each");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x * SM_COLUMNS_PER_WORKGROUP + wave;
    const float *x = args.x + blockIdx.y * args.bs;
    float sum = 0.0f, squares = 0.0f;
    if (k < args.k) {
        // eight loads under way per lane, added in the order of the rows: the sampled rows of a long panel lie far apart,
        // and one load at a time made this launch 20 us of waiting (4096 rows: 64 round trips) where it now takes a few
        constexpr int IN_FLIGHT = 8;
        for (int first = lane; first < args.samples; first += 64 * IN_FLIGHT) {
            float v[IN_FLIGHT];
#pragma unroll
            for (int u = 0; u < IN_FLIGHT; u++) {
                const int s = first + 64 * u;
                v[u] = s < args.samples ? x[(i64)k * args.ld + sampled_row(args, s)] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < IN_FLIGHT; u++)
                if (first + 64 * u < args.samples) {
                    sum += v[u];
                    squares += v[u] * v[u];
                }
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        sum += __shfl_xor(sum, offset);
        squares += __shfl_xor(squares, offset);
    }
    if (lane == 0 && k < args.k_padded) {
        const float total = sum, total_squares = squares;
        const bool live = k < args.k && args.samples > 0;
        const float mean = live ? total / (float)args.samples : 0.0f;
        const float variance = live ? fmaxf(total_squares / (float)args.samples - mean * mean, 0.0f) : 0.0f;
        args.mean[blockIdx.y * args.mean_bs + k] = mean;
        if (!args.pairs) variance_of(args, blockIdx.y)[k] = variance;
        norms[wave] = mean * mean;
        spreads[wave] = variance;
    }
    if (!args.pairs) return;
    __syncthreads();
    if (threadIdx.x == 0)          // k_padded is a multiple of the waves: all of them have a k
        reinterpret_cast<float2 *>(variance_of(args, blockIdx.y))[blockIdx.x] =
            make_float2((norms[0] + norms[1]) + (norms[2] + norms[3]), (spreads[0] + spreads[1]) + (spreads[2] + spreads[3]));
}

// One workgroup per batch entry: |c|^2 against the summed variance, both added in a fixed order.
__global__ __launch_bounds__(256) void centre_flag(const SampleMeanArgs args)
{
    __shared__ float norms[256], spreads[256];
    const float *centre = args.mean + blockIdx.x * args.mean_bs;
    const float *variance = variance_of(args, blockIdx.x);
    float norm = 0.0f, spread = 0.0f;
    for (int k = threadIdx.x; k < args.k; k += 256) {
        norm += centre[k] * centre[k];
        spread += variance[k];
    }
    norms[threadIdx.x] = norm;
    spreads[threadIdx.x] = spread;
    __syncthreads();
    for (int width = 128; width > 0; width >>= 1) {
        if ((int)threadIdx.x < width) {
            norms[threadIdx.x] += norms[threadIdx.x + width];
            spreads[threadIdx.x] += spreads[threadIdx.x + width];
        }
        __syncthreads();
    }
    if (threadIdx.x < GRAM_CENTRE_PAD) {
        // not-a-number data: keep the subtraction (the comparison is false), the repair decides
        const bool needless = norms[0] <= spreads[0] * (1.0f / 64.0f);
        args.mean[blockIdx.x * args.mean_bs + args.k_padded + threadIdx.x] = (threadIdx.x == 0 && !needless) ? 1.0f : 0.0f;
    }
}

}  // namespace kmc

namespace kmc_host {

// k per workgroup of sample_mean_rows, 0: sample_mean_columns
static int mean_span(int majorness, int rows, int k_padded, int l, int max_samples)
{
    if (majorness != KMC_ROW_MAJOR) return 0;
    const int64_t wide_workgroups = static_cast<int64_t>(k_padded / 64) * l;
    const bool wide = rows <= kmc::SM_ROW_WIDE_MAX_FEW_ROWS ||
                      wide_workgroups >= (rows > max_samples ? kmc::SM_ROW_WIDE_MIN_WORKGROUPS_SAMPLED : kmc::SM_ROW_WIDE_MIN_WORKGROUPS);
    return wide ? 64 : 16;
}

// Means and variances of k columns over the sampled rows, without the flag.  `run` divides `max_samples`, which is at least two runs.
hipError_t launch_sample_mean(const float *x, int majorness, int rows, int k, int64_t ld, int64_t bs, int l, float *mean, int64_t mean_bs,
                              int max_samples, int run, int step, bool pairs, hipStream_t stream, kmc::SampleMeanArgs *launched)
{
    kmc::SampleMeanArgs args;
    args.x = x; args.ld = ld; args.bs = bs;
    args.rows = rows; args.k = k; args.k_padded = (k + kmc::GRAM_CENTRE_PAD - 1) / kmc::GRAM_CENTRE_PAD * kmc::GRAM_CENTRE_PAD;
    args.mean = mean; args.mean_bs = mean_bs;
    args.samples = rows < max_samples ? rows : max_samples;
    args.run = run; args.step = step; args.pairs = pairs;
    if (launched) *launched = args;
    const int span = mean_span(majorness, rows, args.k_padded, l, max_samples);
    if (span == 64)
        return launch(kmc::sample_mean_rows<64>, dim3(args.k_padded / 64, l), dim3(kmc::SM_ROW_THREADS), stream, args);
    if (span == 16)
        return launch(kmc::sample_mean_rows<16>, dim3(args.k_padded / 16, l), dim3(kmc::SM_ROW_THREADS), stream, args);
    return launch(kmc::sample_mean_columns, dim3(args.k_padded / kmc::SM_COLUMNS_PER_WORKGROUP, l), dim3(64 * kmc::SM_COLUMNS_PER_WORKGROUP), stream, args);
}

// The centre that gram_f16_wide's route takes for itself.  512 rows place it within a twentieth of the spread per k, which raises the
// norms by a five-hundredth, in one round of loads.  Runs that fill the lines of memory.  With kmc_sample_mean's 4096 rows and a launch for the flag / now:
// 2000 x 2000 x 784 45.9 / 43.4 us, 10000 points of K = 784 against themselves 302.8 / 292.9, 1000 x 60000 x 784 and its product 448.5 / 445.2.
constexpr int SM_ROUTE_SAMPLES = 512, SM_ROUTE_RUN_ROWS = 16, SM_ROUTE_RUN_COLUMNS = 64;
hipError_t launch_route_centre(const float *x, int majorness, int rows, int k, int64_t ld, int64_t bs, int l, float *mean, int64_t mean_bs, hipStream_t stream)
{
    const int run = majorness == KMC_ROW_MAJOR ? SM_ROUTE_RUN_ROWS : SM_ROUTE_RUN_COLUMNS;
    // the last run ends with the last row, or less than a step in front of it
    const int step = rows > SM_ROUTE_SAMPLES ? (rows - run) / (SM_ROUTE_SAMPLES / run - 1) : 0;
    return launch_sample_mean(x, majorness, rows, k, ld, bs, l, mean, mean_bs, SM_ROUTE_SAMPLES, run, step, true, stream, nullptr);
}

// The pairs that it leaves behind each centre: at most half as many floats as the variances they stand in place of
int route_centre_pairs(int majorness, int rows, int k, int l)
{
    const int k_padded = (k + kmc::GRAM_CENTRE_PAD - 1) / kmc::GRAM_CENTRE_PAD * kmc::GRAM_CENTRE_PAD;
    const int span = mean_span(majorness, rows, k_padded, l, SM_ROUTE_SAMPLES);
    return k_padded / (span ? span : kmc::SM_COLUMNS_PER_WORKGROUP);
}

}  // namespace kmc_host

extern "C" int kmc_sample_mean(const float *x, int32_t majorness, int32_t rows, int32_t k, int64_t ld, int64_t bs, int32_t l,
                               float *mean, int64_t mean_bs, void *stream)
{
    using kmc_host::fail;
    if (majorness != KMC_COL_MAJOR && majorness != KMC_ROW_MAJOR)
        return fail(KMC_ERR_INVALID_ARGUMENT, "majorness %d is not a kmc_majorness", majorness);
    if (rows < 0 || k < 0 || l < 0 || ld < 0 || bs < 0 || mean_bs < 0)
        return fail(KMC_ERR_INVALID_ARGUMENT, "negative extent or stride");
    if (l > 65535) return fail(KMC_ERR_INVALID_ARGUMENT, "batch count %d exceeds 65535", l);
    const int k_padded = (k + kmc::GRAM_CENTRE_PAD - 1) / kmc::GRAM_CENTRE_PAD * kmc::GRAM_CENTRE_PAD;
    if (k == 0 || l == 0) return KMC_OK;
    if (!mean || (rows > 0 && !x)) return fail(KMC_ERR_INVALID_ARGUMENT, "null pointer");
    if (l > 1 && mean_bs < 2 * k_padded + kmc::GRAM_CENTRE_PAD)
        return fail(KMC_ERR_INVALID_ARGUMENT, "mean_bs = %lld is smaller than 2 * %d + %d", static_cast<long long>(mean_bs), k_padded,
                    kmc::GRAM_CENTRE_PAD);
    int status = kmc_host::require_gfx950();
    if (status != KMC_OK) return status;
    kmc::SampleMeanArgs args;
    hipError_t e = kmc_host::launch_sample_mean(x, majorness, rows, k, ld, bs, l, mean, mean_bs, kmc::SM_MAX_SAMPLES, kmc::SM_RUN, 0, false, static_cast<hipStream_t>(stream), &args);
    if (e != hipSuccess) return kmc_host::fail_hip(e, "sample_mean launch");
    e = kmc_host::launch(kmc::centre_flag, dim3(l), dim3(256), static_cast<hipStream_t>(stream), args);
    if (e != hipSuccess) return kmc_host::fail_hip(e, "centre_flag launch");
    return KMC_OK;
}
