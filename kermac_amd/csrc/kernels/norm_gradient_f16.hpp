// Kernel-gradient contraction for the L1 norm on the fp16 matrix instruction:
//
//   E[m, n, o, l] = sum_k C[o,k,l] * A[m,k,l] * s(m,n,k),     s = copysign(1, D[m,n,l] - B[n,k,l])
//
// (reference: include/p_norm_gradient.cuh:407-497 with NormType::L1, whose weight of a term is
// the sign of d - b, :373-394).  For a fixed m this is a product of two matrices,
//
//   E[n, o] = sum_k (2 S[n, k] - 1) * W[k, o],     S = 1 where d >= b and 0 where not,    W[k, o] = A[m, k] * C[o, k],
//
// whose left operand is exact in 16 bits.  W is what has to be split into two fp16 pieces, and it is made once per
// (m, k, o) and meets every n, so a term (m, n, k) costs two matrix instruction slots (S w1 + S w2) and half a vector
// instruction for S:
//
// gradient_signs_prepare   per row n of B: the position of every b[n, k] in the sorted row, and for every d[n, m] how
//                          many b of the row are not above it.  d >= b is then position < count, for integers below
//                          14335, written as fp16 numbers that lie at least 1 apart (signs_half): one packed
//                          subtraction with the clamp to [0, 1] compares two k and gives S in fp16.  The keys that are
//                          sorted order -0 below +0, so that signed zeros and ties come out as copysign(1, d - b).
//                          Rows of B longer than that are cut into chunks with positions of their own.
//                          The same launch copies A into the order in which a wave reads it, scales C by a power of two per
//                          row o, and bounds |A[m, k] C[o, k]| for every m and o by its sum over 128 k or fewer.
// norm_gradient_l1_f16     the product.
//
// Accuracy: S is exact.  w = a c 2^F with its largest sum over those k in [2^14, 2^15.2), F of every m and o from the launch before; w1 =
// fp16(w), w2 = fp16(w - w1), so |w - w1 - w2| <= 2^-22 |w| + 2^-39 sum_k|w|, however far max_k|a c| is below max|a| max|c|.  Doubled
// with the result, that is below 3 * 2^-22 sum_k |c a| up to K = 2^16, beside the fp32 accumulation.  (A scale per row m of A times one per
// row o of C is not enough: in rows with a large value whose partner is zero, 1 beside 2^-16 say, fp16's smallest step takes the place
// of the others' last bits, 6e-6 of sum_k |c a| and more.)  Sums of zero count as 2^-127, which shows where max|a| or max|c| is above
// 2^100 times the products; rows of A below 2^-112 keep fewer bits.  The sums run over S W, so  1/2 sum_k W  is taken off them again: every 256
// k, since a partial sum of S W alone drifts away from the one of the signed terms, and rounding follows the partial sums.
//
// Workgroup of norm_gradient_l1_f16: 8 waves, 16 m x 16 BLOCKS n x 16 o; wave w owns the 2 m  2w, 2w + 1  and all n, as
// BLOCKS x 2 results of v_mfma_f32_16x16x32_f16 (rows n, columns o).  The more n a wave holds, the less W costs: at 256
// n the 64 matrix instructions of a step of 32 k stand beside 128 packed subtractions and about 100 other vector instructions, two
// thirds of them the cheap ones of fp32.
// Bound by the two together: on registers alone a v_mfma_f32_16x16x32_f16 takes 16.5 cycles, 16.9 with two packed
// subtractions beside it, and four more for every further packed instruction; the kernel takes about 26.
// Measured at M = K = 8192, N = 512, O = 16: 1.94 ms with 0.18 ms of gradient_signs_prepare (3.65 ms for the kernel that
// flipped the sign into both pieces of A: three products and 2.5 vector instructions per term), O = 32 3.75 ms (5.55).  W from
// pieces of A and C under a scale per row each, which loses bits as said above, took 1.94 and 3.70.
// Up to 8 outputs leave half of the columns unused: there the columns 8 .. 15 take the second pieces (PIECES_IN_COLUMNS),
// one matrix instruction instead of two.  Everything a step reads arrives in LDS by global_load_lds, a stage of 64 k in
// one of two buffers while the other is worked on; the copies are inline instructions for the reason given in
// gram_f16_wide.hpp.
#pragma once

#include "gram_f16_wide.hpp"
#include "norm_gradient.hpp"

namespace kmc {

typedef float ngf_float4 __attribute__((ext_vector_type(4)));

constexpr int NGF_STEP_K = 32;
constexpr int NGF_STAGE_K = 64;                // two steps
constexpr int NGF_WAVES = 8;
constexpr int NGF_TILE_M = 2 * NGF_WAVES;
constexpr int NGF_TILE_O = 16;
constexpr int NGF_THREADS = 64 * NGF_WAVES;
constexpr int NGF_N_PAD = 256;
constexpr int NGF_CORRECT_STAGES = 4;          // 1/2 sum W is taken off every so many stages
constexpr int NGF_PREPARE_THREADS = 256;
constexpr int NGF_PREPARE_GROUP = 256;
constexpr int NGF_M_PAD = 64;
constexpr int NGF_COPY_M = 128;                // tile of the copy of A: m, and k per workgroup at most and at least
constexpr int NGF_COPY_MAX_K = 512;
constexpr int NGF_COPY_MIN_K = 64;
constexpr int NGF_COPY_DEPTH = 16;             // k per lane at a time
constexpr int NGF_COPY_C_PITCH = 4 * NGF_TILE_O + 4;   // words of LDS per eight k of 16 o
constexpr int NGF_COPY_C_WORDS = NGF_COPY_MAX_K / 8 * NGF_COPY_C_PITCH;
constexpr int NGF_EXPONENT_W = 14;             // bound of a result's W in [2^14, 2^15.2): fp16 ends at 2^16
constexpr int NGF_EXPONENT_C = 14;             // largest C of a row as it is copied, in [2^14, 2^15): A, which takes the rest of W's scale, is
                                               // then brought to 1 or a little more
constexpr int NGF_MAX_CHUNK = 14272;           // k per sorted chunk: whole stages, counts up to 14334 (signs_half)

struct NormGradientF16Args {
    NormGradientArgs g;                        // extents, d, e, strides, o_chunks; a, b, c are not read
    int o_begin;                               // the launch covers the outputs from here on
    const unsigned short *positions;           // [batch][k / 8][n_pad][8]: of b in its sorted row
    const unsigned short *counts;              // [batch][chunk][n_pad][m_pad]: b not above d
    i64 positions_bs, counts_bs;               // in halves
    const float *a_copy; i64 a_copy_bs;        // [batch][m_pad / 2][k_pad / 32][4][2][8]: 8 k of each of 2 m, 4 times
    const float *a_magnitudes; i64 a_magnitudes_bs;    // [batch][ranges][m_pad]
    const unsigned short *products; i64 products_bs;   // [batch][ranges][o_pad / 16][m_pad][16 o]: sums of |a c|, bfloat16
    const float *c_copy; i64 c_copy_bs;        // [batch][o_pad / 16][k_pad / 4][16 o][4 k], times 2^c_exponents
    const int *c_exponents; i64 c_exponents_bs;        // [batch][o_pad]
    int n_pad, m_pad, k_pad, o_pad, ranges;
    int chunk_stages, stages;                  // length of the sorted chunks (the last may be shorter), all stages
};

struct GradientPrepareArgs {
    int m, n, o, k;
    const float *a; i64 a_ld, a_bs;
    const float *b; i64 b_ld, b_bs;
    const float *c; i64 c_ld, c_bs;
    const float *d; i64 d_ld, d_bs;
    unsigned short *positions, *counts; i64 positions_bs, counts_bs;
    float *a_copy; i64 a_copy_bs;
    float *a_magnitudes; i64 a_magnitudes_bs;
    unsigned short *products; i64 products_bs;
    float *c_copy; i64 c_copy_bs;
    int *c_exponents; i64 c_exponents_bs;
    int n_pad, m_pad, k_pad, o_pad, copy_k, ranges, chunk_k;
    int sort_d;                                // the rows of D are sorted, not those of B
    int sort_blocks, copy_blocks;              // rows to sort, tiles of A times blocks of 16 o, ...
    int sort_groups, copy_groups;              // ... and how many groups of NGF_PREPARE_GROUP that makes; blockIdx.x also has the rows of C
    int sort_batches, a_batches, c_batches, product_batches;       // blockIdx.y
    int a_vec;
};

// The integer count - 7167, count in 0 .. 14334, as an fp16 number: itself up to 2048, and beyond that the next larger
// fp16 numbers in turn, which lie 2, 4, .. 32 apart.  Larger counts give larger numbers, at least 1 larger.
__device__ __forceinline__ unsigned signs_half(int count)
{
    const int centred = count - 7167;
    const unsigned magnitude = (unsigned)abs(centred);
    const unsigned exact = __builtin_bit_cast(unsigned short, (_Float16)(float)magnitude);
    const unsigned bits = magnitude < 1024 ? exact : 0x6000 + magnitude;      // 1024 is 0x6400
    return bits | (centred < 0 ? 0x8000u : 0u);
}

// Unsigned integers in the order of copysign(1, d - b): -0 below +0, everything else as the floats
__device__ __forceinline__ unsigned signs_key(float x)
{
    const int bits = __float_as_int(x);
    return (unsigned)(bits ^ ((bits >> 31) & 0x7fffffff)) ^ 0x80000000u;
}

// LDS word of element i of the sorted row: a word of padding in 32, or lanes that own consecutive runs meet in few banks
__device__ __forceinline__ int signs_word(int i)
{
    return i + (i >> 5);
}

// Bitonic sort of 256 << LOG_R keys by 256 threads, LOG_R strides per pass through LDS: the 1 << LOG_R keys that a
// thread holds differ in the bits lo .. lo + LOG_R - 1 of their index.  (8192 keys: 19 passes instead of 91.)
template <int LOG_R>
__device__ __forceinline__ void signs_sort(unsigned (&key)[1 << LOG_R], unsigned *sorted, int tid)
{
    constexpr int R = 1 << LOG_R;
    constexpr int LOG_N = 8 + LOG_R;
    auto compare = [&](int low, int high, bool descending) {
        const unsigned smaller = min(key[low], key[high]), larger = max(key[low], key[high]);
        key[low] = descending ? larger : smaller;
        key[high] = descending ? smaller : larger;
    };
    // the keys arrive as consecutive runs of R: the first LOG_R levels need no exchange
#pragma unroll
    for (int level = 1; level <= LOG_R; level++)
#pragma unroll
        for (int bit = level - 1; bit >= 0; bit--)
#pragma unroll
            for (int e = 0; e < R; e++)
                if (!(e >> bit & 1)) compare(e, e | 1 << bit, level == LOG_R ? (tid & 1) : (e >> level & 1));
#pragma unroll
    for (int e = 0; e < R; e++) sorted[signs_word(tid * R + e)] = key[e];
    for (int level = LOG_R + 1; level <= LOG_N; level++) {
        for (int high = level - 1; high >= 0;) {
            const int lo = max(high - LOG_R + 1, 0);
            const int first = (tid & ((1 << lo) - 1)) | (tid >> lo) << (lo + LOG_R);
            const bool descending = first >> level & 1;
            __syncthreads();
#pragma unroll
            for (int e = 0; e < R; e++) key[e] = sorted[signs_word(first + (e << lo))];
#pragma unroll
            for (int bit = LOG_R - 1; bit >= 0; bit--) {
                if (bit > high - lo) continue;
#pragma unroll
                for (int e = 0; e < R; e++)
                    if (!(e >> bit & 1)) compare(e, e | 1 << bit, descending);
            }
#pragma unroll
            for (int e = 0; e < R; e++) sorted[signs_word(first + (e << lo))] = key[e];
            high = lo - 1;
        }
    }
    __syncthreads();
}

// How many of the 256 << LOG_R sorted keys are below x (NOT_ABOVE: not above x), for eight x side by side
template <int LOG_R, bool NOT_ABOVE>
__device__ __forceinline__ void signs_search(const unsigned *sorted, const unsigned (&x)[8], int (&count)[8])
{
#pragma unroll
    for (int j = 0; j < 8; j++) count[j] = 0;
    for (int half = 128 << LOG_R; half >= 1; half >>= 1) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const unsigned key = sorted[signs_word(count[j] + half - 1)];
            if (NOT_ABOVE ? key <= x[j] : key < x[j]) count[j] += half;
        }
    }
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const unsigned key = sorted[signs_word(count[j])];       // at most the last one
        if (NOT_ABOVE ? key <= x[j] : key < x[j]) count[j]++;
    }
}

__device__ __forceinline__ gram_chunk signs_pack(const int (&count)[8])
{
    gram_chunk packed;
#pragma unroll
    for (int j = 0; j < 4; j++) packed[j] = signs_half(count[2 * j]) | signs_half(count[2 * j + 1]) << 16;
    return packed;
}

// A row n of B and of D; the shorter one is sorted, the other one (and the sorted one itself) searched in it.  With b
// sorted: position = how many b are below b[k], count = how many b are not above d[m].  With d sorted: position = how
// many d are below b[k], count = 1 + how many d are below d[m].  Both ways count > position exactly if d >= b, equal keys
// included.  Bound by LDS (the sort, then log2 of its length dependent reads per element searched).
template <int LOG_R>
__device__ __forceinline__ void signs_rank_row(const GradientPrepareArgs &args, int block, int batch, unsigned *sorted)
{
    constexpr int R = 1 << LOG_R;
    const int tid = threadIdx.x;
    const int n = block % args.n, chunk = block / args.n;
    const int k0 = chunk * args.chunk_k;
    const int ks = min(args.chunk_k, args.k - k0);
    const int span = min(args.chunk_k, args.k_pad - k0);
    const float *b_row = args.b + batch * args.b_bs + (i64)n * args.b_ld + k0;
    const float *d_row = args.d + batch * args.d_bs + (i64)n * args.d_ld;
    const float *sorted_row = args.sort_d ? d_row : b_row;
    const int keys = args.sort_d ? args.m : ks;
    {
        unsigned key[R];
#pragma unroll
        for (int e = 0; e < R; e++) key[e] = tid * R + e < keys ? signs_key(sorted_row[tid * R + e]) : ~0u;
        signs_sort<LOG_R>(key, sorted, tid);
    }
    gram_chunk *positions = reinterpret_cast<gram_chunk *>(args.positions + batch * args.positions_bs) + (i64)(k0 / 8) * args.n_pad + n;
    for (int k = 8 * tid; k < span; k += 8 * NGF_PREPARE_THREADS) {
        unsigned x[8];
        int position[8];
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = k + j < ks ? signs_key(b_row[k + j]) : ~0u;
        signs_search<LOG_R, false>(sorted, x, position);
#pragma unroll
        for (int j = 0; j < 8; j++) position[j] = min(position[j], keys);         // what lies beyond K meets W = 0
        positions[(i64)(k / 8) * args.n_pad] = signs_pack(position);
    }
    unsigned short *counts = args.counts + batch * args.counts_bs + ((i64)chunk * args.n_pad + n) * args.m_pad;
    for (int m = 8 * tid; m < args.m_pad; m += 8 * NGF_PREPARE_THREADS) {
        unsigned x[8];
        int count[8];
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = m + j < args.m ? signs_key(d_row[m + j]) : 0u;
        if (args.sort_d) {
            signs_search<LOG_R, false>(sorted, x, count);
#pragma unroll
            for (int j = 0; j < 8; j++) count[j]++;
        } else {
            signs_search<LOG_R, true>(sorted, x, count);
        }
#pragma unroll
        for (int j = 0; j < 8; j++) count[j] = min(count[j], keys);               // the padding of the sort is not B's
        *reinterpret_cast<gram_chunk *>(counts + m) = signs_pack(count);
    }
}

typedef unsigned short ngf_ushort8 __attribute__((ext_vector_type(8)));

typedef short ngf_short4 __attribute__((ext_vector_type(4)));

// |x0| and |x1| as bfloat16, rounded down
__device__ __forceinline__ unsigned signs_magnitudes(float x0, float x1)
{
    return __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u) & 0x7fff7fffu;
}

// Chunk j of a lane becomes its chunk of the four that lane j of its group of four holds
__device__ __forceinline__ void signs_transpose_quad(float4 (&chunk)[4], int lane)
{
#pragma unroll
    for (int bit = 1; bit <= 2; bit *= 2) {
        const bool upper = lane & bit;
        auto exchange = [&](float &low, float &high) {
            const int sent = __float_as_int(upper ? low : high);
            const float received = __int_as_float(bit == 1 ? __builtin_amdgcn_update_dpp(0, sent, 0xB1, 0xF, 0xF, true)      // quad_perm 1, 0, 3, 2
                                                           : __builtin_amdgcn_update_dpp(0, sent, 0x4E, 0xF, 0xF, true));    // quad_perm 2, 3, 0, 1
            low = upper ? received : low;
            high = upper ? high : received;
        };
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j & bit) continue;
            exchange(chunk[j].x, chunk[j + bit].x);
            exchange(chunk[j].y, chunk[j + bit].y);
            exchange(chunk[j].z, chunk[j + bit].z);
            exchange(chunk[j].w, chunk[j + bit].w);
        }
    }
}

// Half word of LDS of the sum of row m and output 0 of a tile: 4 words of padding per 8 rows, or lanes that own them meet in one bank
__device__ __forceinline__ int signs_sum_at(int m)
{
    return 16 * m + 8 * (m >> 3);
}

// 128 m x copy_k k of A into the order of the product's waves, the largest magnitude per m, and for one block of 16 outputs (the blocks after
// the first only that) sum_k |a c| per m and o, the largest of four quarters of the k.  No |a c| is above its sum, and the sum, unlike a
// maximum, is work for the matrix instruction: v_mfma_f32_4x4x4_16B_bf16 takes 4 k of a lane's own row with 4 outputs, which are read as broadcasts
// of LDS.  (bfloat16 has the range of fp32; rounded down, |a|, |c| and the sum are up to 2.4 % too small.)  A lane holds 2 m and 16 k at a time,
// which are 128 bytes of the copy; a wave takes a quarter of the k.  Memory-bound together with the sorts beside it.  The launch with the maxima on the
// vector ALU and stores of 16 bytes per lane / now, us: 8192 x 512 x 16 x 8192 197 / 179, 2 x 3200 x 32 x 10 x 10432 154 / 119, 4000 x 32 x 128 x 4000 126 / 67.
__device__ __forceinline__ void signs_copy_tile(const GradientPrepareArgs &args, int block, int batch, unsigned *shared)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int o_blocks = args.o_pad / NGF_TILE_O, m_tiles = (args.m_pad + NGF_COPY_M - 1) / NGF_COPY_M;
    // the blocks of outputs of a tile run one behind the other on one XCD, whose L2 then holds the tile for all but the first
    const int o_block = block / BK_XCDS % o_blocks, at = block / BK_XCDS / o_blocks * BK_XCDS + block % BK_XCDS;
    const int m0 = at % m_tiles * NGF_COPY_M, range = at / m_tiles;
    if (range >= args.ranges) return;
    const int o_count = min(args.o - NGF_TILE_O * o_block, NGF_TILE_O);
    const int k_first = range * args.copy_k, k_count = min(args.copy_k, args.k_pad - k_first);
    const bool copies = o_block == 0 && batch < args.a_batches;

    const int m = m0 + 2 * lane;
    const float *a = args.a + batch * args.a_bs;
    const bool aligned = args.a_vec && m0 + NGF_COPY_M <= args.m;
    float2 v[NGF_COPY_DEPTH];
    auto load = [&](int k0) {
        if (aligned && k0 + NGF_COPY_DEPTH <= args.k) {
#pragma unroll
            for (int j = 0; j < NGF_COPY_DEPTH; j++) v[j] = *reinterpret_cast<const float2 *>(a + (i64)(k0 + j) * args.a_ld + m);
        } else {
            const int at0 = min(m, args.m - 1), at1 = min(m + 1, args.m - 1);
#pragma unroll
            for (int j = 0; j < NGF_COPY_DEPTH; j++) {
                const float *row = a + (i64)min(k0 + j, args.k - 1) * args.a_ld;
                v[j] = make_float2(row[at0], row[at1]);
            }
#pragma unroll
            for (int j = 0; j < NGF_COPY_DEPTH; j++) {
                v[j].x = k0 + j < args.k && m < args.m ? v[j].x : 0.0f;
                v[j].y = k0 + j < args.k && m + 1 < args.m ? v[j].y : 0.0f;
            }
        }
    };
    float magnitude[2] = {0.0f, 0.0f};
    const int k_wave = k_first + wave * (k_count / 4), k_end = k_wave + k_count / 4;        // k_count: a multiple of 64
    load(k_wave);
    // C while these are under way: four outputs per wave, two k per lane.  Loads of what does not exist, of C and of A, go to the
    // last element that does and are dropped: with a branch for each they would be waited for one by one
    {
        constexpr int ROWS = NGF_TILE_O / 4;
        const float *c = args.c + batch * args.c_bs + (i64)NGF_TILE_O * o_block * args.c_ld;
        constexpr int TIMES = 2;
        for (int first = 0; first < k_count / 2; first += 64 * TIMES) {
            float x[TIMES][ROWS][2];
#pragma unroll
            for (int t = 0; t < TIMES; t++) {
                const int k = k_first + 2 * (first + 64 * t + lane), at0 = min(k, args.k - 1), at1 = min(k + 1, args.k - 1);
#pragma unroll
                for (int j = 0; j < ROWS; j++) {
                    const float *row = c + (i64)min(ROWS * wave + j, o_count - 1) * args.c_ld;
                    x[t][j][0] = row[at0];
                    x[t][j][1] = row[at1];
                }
            }
#pragma unroll
            for (int t = 0; t < TIMES; t++) {
                const int pair = first + 64 * t + lane, k = k_first + 2 * pair;
#pragma unroll
                for (int j = 0; j < ROWS; j++) {
                    const int o = ROWS * wave + j;
                    if (pair < k_count / 2)
                        shared[pair / 4 * NGF_COPY_C_PITCH + 4 * o + pair % 4] =
                            signs_magnitudes(o < o_count && k < args.k ? x[t][j][0] : 0.0f, o < o_count && k + 1 < args.k ? x[t][j][1] : 0.0f);
                }
            }
        }
    }
    // sums[i][o4][j]: m = m0 + 8 (lane / 4) + 2 j + i, the row of lane 4 (lane / 4) + j, o = 4 o4 + lane % 4
    ngf_float4 sums[2][NGF_TILE_O / 4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int o4 = 0; o4 < NGF_TILE_O / 4; o4++) sums[i][o4] = ngf_float4{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();
    for (int k0 = k_wave; k0 < k_end; k0 += NGF_COPY_DEPTH) {
        uint2 magnitudes[2][NGF_COPY_DEPTH / 4];           // 4 k
#pragma unroll
        for (int j = 0; j < NGF_COPY_DEPTH / 4; j++) {
            magnitudes[0][j] = make_uint2(signs_magnitudes(v[4 * j].x, v[4 * j + 1].x), signs_magnitudes(v[4 * j + 2].x, v[4 * j + 3].x));
            magnitudes[1][j] = make_uint2(signs_magnitudes(v[4 * j].y, v[4 * j + 1].y), signs_magnitudes(v[4 * j + 2].y, v[4 * j + 3].y));
        }
        if (copies) {
#pragma unroll
            for (int j = 0; j < NGF_COPY_DEPTH; j++) {     // skips NaNs, whose products are not numbers at any scale
                magnitude[0] = fmaxf(magnitude[0], fabsf(v[j].x));
                magnitude[1] = fmaxf(magnitude[1], fabsf(v[j].y));
            }
            // 8 k of a lane's two m are 64 bytes of the copy: four lanes exchange theirs and store 64 bytes side by side (a lane's own stores, 16
            // bytes of 64 lines each, take half as long again as the memory)
#pragma unroll
            for (int eight = 0; eight < NGF_COPY_DEPTH; eight += 8) {
                float4 chunk[4];
#pragma unroll
                for (int j = 0; j < 8; j += 4) {
                    chunk[j / 4] = make_float4(v[eight + j].x, v[eight + j + 1].x, v[eight + j + 2].x, v[eight + j + 3].x);
                    chunk[2 + j / 4] = make_float4(v[eight + j].y, v[eight + j + 1].y, v[eight + j + 2].y, v[eight + j + 3].y);
                }
                signs_transpose_quad(chunk, lane);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int pair = m0 / 2 + (lane & ~3) + j;
                    if (2 * pair < args.m_pad)
                        *reinterpret_cast<float4 *>(args.a_copy + batch * args.a_copy_bs + ((i64)pair * args.k_pad + k0 + eight) * 2 + 4 * (lane & 3)) = chunk[j];
                }
            }
        }
        if (k0 + NGF_COPY_DEPTH < k_end) load(k0 + NGF_COPY_DEPTH);
        // (outputs that do not exist are zeros: a branch for them would have their reads waited for one by one)
#pragma unroll
        for (int eight = 0; eight < NGF_COPY_DEPTH / 8; eight++) {
            uint4 c8[NGF_TILE_O / 4];
#pragma unroll
            for (int o4 = 0; o4 < NGF_TILE_O / 4; o4++)
                c8[o4] = *reinterpret_cast<const uint4 *>(shared + ((k0 - k_first) / 8 + eight) * NGF_COPY_C_PITCH + 16 * o4 + 4 * (lane & 3));
#pragma unroll
            for (int four = 0; four < 2; four++)
#pragma unroll
                for (int o4 = 0; o4 < NGF_TILE_O / 4; o4++)
#pragma unroll
                    for (int i = 0; i < 2; i++)
                        sums[i][o4] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(
                            __builtin_bit_cast(ngf_short4, magnitudes[i][2 * eight + four]),
                            __builtin_bit_cast(ngf_short4, four == 0 ? make_uint2(c8[o4].x, c8[o4].y) : make_uint2(c8[o4].z, c8[o4].w)), sums[i][o4], 0, 0, 0);
        }
    }
    // the four waves' sums, as bfloat16, and behind them the magnitudes
    constexpr int WAVE_WORDS = NGF_COPY_M * NGF_TILE_O / 2 + NGF_COPY_M / 2;
    unsigned short *const wave_sums = reinterpret_cast<unsigned short *>(shared);
    float *const magnitudes = reinterpret_cast<float *>(shared + 4 * WAVE_WORDS);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; i++) {
#pragma unroll
        for (int o4 = 0; o4 < NGF_TILE_O / 4; o4++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                wave_sums[2 * wave * WAVE_WORDS + signs_sum_at(8 * (lane >> 2) + 2 * j + i) + 4 * o4 + (lane & 3)] =
                    (unsigned short)(__float_as_uint(sums[i][o4][j]) >> 16 & 0x7fff);
        magnitudes[(wave * 2 + i) * 64 + lane] = magnitude[i];
    }
    __syncthreads();
    const int to = m0 + (tid >> 1), i = tid >> 1 & 1;      // half of the outputs of one m per thread
    if (to >= args.m_pad) return;
    if (batch < args.product_batches) {
        ngf_ushort8 largest = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int part = 0; part < 4; part++)
            largest = __builtin_elementwise_max(
                largest, *reinterpret_cast<const ngf_ushort8 *>(wave_sums + 2 * part * WAVE_WORDS + signs_sum_at(tid >> 1) + 8 * (tid & 1)));
        unsigned short *products = args.products + batch * args.products_bs + (((i64)range * o_blocks + o_block) * args.m_pad + to) * NGF_TILE_O;
        reinterpret_cast<ngf_ushort8 *>(products)[tid & 1] = largest;
    }
    if (copies && !(tid & 1)) {
        float x = 0.0f;
#pragma unroll
        for (int part = 0; part < 4; part++) x = fmaxf(x, magnitudes[(part * 2 + i) * 64 + (tid >> 2)]);
        args.a_magnitudes[batch * args.a_magnitudes_bs + (i64)range * args.m_pad + to] = x;
    }
}

// Exponent of the first bit of a number (of its scale, which the largest value of a row is)
__device__ __forceinline__ int signs_exponent(float magnitude)
{
    return ((int)(__float_as_uint(magnitude) >> 23) & 0xff) - 127;
}

// One row o of C times the power of two that brings its largest magnitude to [2^14, 2^15), zeros beyond K and O
__device__ __forceinline__ void signs_scale_row(const GradientPrepareArgs &args, int o, int batch, float *shared)
{
    const int tid = threadIdx.x;
    const float *row = args.c + batch * args.c_bs + (i64)o * args.c_ld;
    const bool live = o < args.o;
    float magnitude = 0.0f;
    if (live)
        for (int k = tid; k < args.k; k += 4 * NGF_PREPARE_THREADS)
#pragma unroll
            for (int j = 0; j < 4; j++) magnitude = fmaxf(magnitude, fabsf(row[min(k + j * NGF_PREPARE_THREADS, args.k - 1)]));
#pragma unroll
    for (int bit = 1; bit < 64; bit *= 2) magnitude = fmaxf(magnitude, __shfl_xor(magnitude, bit));
    if ((tid & 63) == 0) shared[tid >> 6] = magnitude;
    __syncthreads();
#pragma unroll
    for (int wave = 0; wave < NGF_PREPARE_THREADS / 64; wave++) magnitude = fmaxf(magnitude, shared[wave]);
    const int exponent = NGF_EXPONENT_C - signs_exponent(magnitude);
    if (tid == 0) args.c_exponents[batch * args.c_exponents_bs + o] = exponent;
    float4 *copy = reinterpret_cast<float4 *>(args.c_copy + batch * args.c_copy_bs) + (i64)(o / NGF_TILE_O) * args.k_pad / 4 * NGF_TILE_O + o % NGF_TILE_O;
    for (int k = 4 * tid; k < args.k_pad; k += 4 * NGF_PREPARE_THREADS) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = live ? row[min(k + j, args.k - 1)] : 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = k + j < args.k ? __builtin_ldexpf(v[j], exponent) : 0.0f;
        copy[(i64)(k / 4) * NGF_TILE_O] = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// Rows to sort keep LDS busy, tiles of A the memory and the vector ALU, so the two are dealt out in turn, in groups of one workgroup per
// CU, spread evenly over the launch (all sorts within its first half: 214 us in the place of 200 at 8192 x 512 x 16 x 8192).  The rows of C, few
// and slow, come first.
template <int LOG_R>
__global__ __launch_bounds__(NGF_PREPARE_THREADS, LOG_R < 5 ? 4 : LOG_R < 6 ? 3 : 2) void gradient_signs_prepare(const GradientPrepareArgs args)
{
    constexpr int WORDS = (256 << LOG_R) + (8 << LOG_R);
    // C of a tile, then the waves' sums and magnitudes
    constexpr int SUM_WORDS = 4 * (NGF_COPY_M * (NGF_TILE_O + 1) / 2 + NGF_COPY_M);
    constexpr int TILE_WORDS = NGF_COPY_C_WORDS > SUM_WORDS ? NGF_COPY_C_WORDS : SUM_WORDS;
    __shared__ __attribute__((aligned(16))) unsigned words[WORDS > TILE_WORDS ? WORDS : TILE_WORDS];
    const int batch = blockIdx.y, block_behind_c = (int)blockIdx.x - args.o_pad;
    if (block_behind_c < 0) {
        if (batch < args.c_batches) signs_scale_row(args, blockIdx.x, batch, reinterpret_cast<float *>(words));
        return;
    }
    const i64 groups = args.sort_groups + args.copy_groups, group = block_behind_c / NGF_PREPARE_GROUP;
    const int within = block_behind_c % NGF_PREPARE_GROUP;
    const int sorts_before = (int)((group * args.sort_groups + groups - 1) / groups);
    const int sorts_behind = (int)(((group + 1) * args.sort_groups + groups - 1) / groups);
    if (sorts_behind > sorts_before) {
        const int block = sorts_before * NGF_PREPARE_GROUP + within;
        if (block < args.sort_blocks && batch < args.sort_batches) signs_rank_row<LOG_R>(args, block, batch, words);
    } else {
        const int block = ((int)group - sorts_before) * NGF_PREPARE_GROUP + within;
        if (block < args.copy_blocks && batch < max(args.a_batches, args.product_batches)) signs_copy_tile(args, block, batch, words);
    }
}

typedef _Float16 ngf_half2 __attribute__((ext_vector_type(2)));

// (by value: a bit cast of an element of a vector, in place, takes the first element)
__device__ __forceinline__ ngf_half2 signs_halves(unsigned x)
{
    return __builtin_bit_cast(ngf_half2, x);
}

// 1 where count > position and 0 where not, in both halves: one v_pk_add_f16 with clamp
__device__ __forceinline__ unsigned signs_compare(_Float16 count, unsigned positions)
{
    ngf_half2 x = ngf_half2{count, count} - signs_halves(positions);
    x = __builtin_elementwise_min(__builtin_elementwise_max(x, ngf_half2{(_Float16)0, (_Float16)0}), ngf_half2{(_Float16)1, (_Float16)1});
    return __builtin_bit_cast(unsigned, x);
}

template <int BLOCKS>
struct GradientF16Tile {
    static constexpr int TILE_N = 16 * BLOCKS;
    static constexpr int POSITION_CHUNKS = 8 * TILE_N;                  // of 16 bytes, per stage
    static constexpr int C_CHUNKS = NGF_STAGE_K * NGF_TILE_O / 4;
    static constexpr int A_CHUNKS = NGF_STAGE_K * NGF_TILE_M / 4;
    static constexpr int PASS_BLOCKS = BLOCKS < 4 ? BLOCKS : 2;         // of 16 n, per pass of the epilogue
    static constexpr int RESULT_PITCH = NGF_TILE_M + 4;
    static constexpr int PASS_CHUNKS = PASS_BLOCKS * 256 * RESULT_PITCH / 4;
    // two stages of everything: 80 KB at 256 n
    static constexpr int STAGE_CHUNKS = 2 * (POSITION_CHUNKS + C_CHUNKS + A_CHUNKS);
    static constexpr int CHUNKS = STAGE_CHUNKS > PASS_CHUNKS ? STAGE_CHUNKS : PASS_CHUNKS;
};

template <int BLOCKS, bool PIECES_IN_COLUMNS>
__global__ __launch_bounds__(NGF_THREADS, BLOCKS >= 8 ? 2 : 4) void norm_gradient_l1_f16(const NormGradientF16Args args)
{
    using Tile = GradientF16Tile<BLOCKS>;
    constexpr int COLUMN_PIECES = PIECES_IN_COLUMNS ? 1 : GW_PIECES;
    __shared__ gram_chunk lds[Tile::CHUNKS];

    const NormGradientArgs &g = args.g;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4;     // 8 k of a step (operands), row quad (result)
    const int r = lane & 15;     // row n (S) / column (W, result)
    const int batch = blockIdx.z / g.o_chunks;
    const int o0 = args.o_begin + (blockIdx.z % g.o_chunks) * NGF_TILE_O;
    // the tiles of an XCD (every eighth workgroup) lie side by side, so that two of them fill a line of E in its L2
    const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3, longer = gridDim.x & 7;
    const int m0 = (xcd * per_xcd + min(xcd, longer) + (int)(blockIdx.x >> 3)) * NGF_TILE_M;
    const int n0 = blockIdx.y * Tile::TILE_N;

    typedef const __attribute__((address_space(1))) void *global_address;
    typedef __attribute__((address_space(3))) void *lds_address;
    // Copies of 64 chunks per stage and wave, the same in every wave.  Positions: 8 runs (8 k each) of TILE_N chunks; a copy
    // is a part of a run, or, of 32 n, two runs.  C: 256 chunks in a row.  A: the 512 bytes of the wave's own two m, as two copies of 4
    // bytes per lane.
    constexpr int POSITION_COPIES = 2 * BLOCKS / NGF_WAVES > 0 ? 2 * BLOCKS / NGF_WAVES : 1;
    constexpr int COPIES_PER_RUN = BLOCKS >= 4 ? BLOCKS / 4 : 1;
    const gram_chunk *position_src[POSITION_COPIES];
    int position_dst[POSITION_COPIES];
#pragma unroll
    for (int j = 0; j < POSITION_COPIES; j++) {
        const int copy = (wave * POSITION_COPIES + j) % (2 * BLOCKS);
        const int run = BLOCKS >= 4 ? copy / COPIES_PER_RUN : 2 * copy + (lane >> 5);
        position_src[j] = reinterpret_cast<const gram_chunk *>(args.positions + batch * args.positions_bs) + (i64)run * args.n_pad + n0 +
                          (BLOCKS >= 4 ? 64 * (copy % COPIES_PER_RUN) + lane : lane & 31);
        position_dst[j] = 64 * copy;
    }
    const gram_chunk *c_src = reinterpret_cast<const gram_chunk *>(args.c_copy + batch * args.c_copy_bs) +
                              (i64)(o0 / NGF_TILE_O) * args.k_pad / 4 * NGF_TILE_O + 64 * (wave & 3) + lane;
    const float *a_src = args.a_copy + batch * args.a_copy_bs + (i64)(m0 / 2 + wave) * (args.k_pad / NGF_STEP_K) * 64 + lane;
    auto copy16 = [&](const gram_chunk *src, gram_chunk *dst) {
        const unsigned lds_byte = (unsigned)(unsigned long)(lds_address)dst;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"((global_address)src), "s"(lds_byte) : "memory", "m0");
    };
    auto copy4 = [&](const float *src, gram_chunk *dst) {
        const unsigned lds_byte = (unsigned)(unsigned long)(lds_address)dst;
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"((global_address)src), "s"(lds_byte) : "memory", "m0");
    };
    gram_chunk *const lds_c = lds + 2 * Tile::POSITION_CHUNKS;
    gram_chunk *const lds_a = lds_c + 2 * Tile::C_CHUNKS;
    auto copy_stage = [&](int into) {
#pragma unroll
        for (int j = 0; j < POSITION_COPIES; j++) {
            copy16(position_src[j], lds + into * Tile::POSITION_CHUNKS + position_dst[j]);
            position_src[j] += (i64)8 * args.n_pad;
        }
        copy16(c_src, lds_c + into * Tile::C_CHUNKS + 64 * (wave & 3));
        c_src += Tile::C_CHUNKS;
#pragma unroll
        for (int j = 0; j < 2; j++) copy4(a_src + 64 * j, lds_a + into * Tile::A_CHUNKS + 32 * wave + 16 * j);
        a_src += 128;
    };

    // The lane's column, and the power of two for A of each of the wave's two m, which with the scale of C makes W's largest value 2^14 or a
    // little more.  A stays finite with it (one that would not meets a C of zero, or of less than 2^-100 of its row).
    const int column = PIECES_IN_COLUMNS ? (r & 7) : r;
    float scale[2];
    int unscale[2];
    {
        const float *magnitudes = args.a_magnitudes + batch * args.a_magnitudes_bs + m0 + 2 * wave;
        const unsigned short *products = args.products + batch * args.products_bs + ((i64)(o0 / NGF_TILE_O) * args.m_pad + m0 + 2 * wave) * NGF_TILE_O + column;
        float magnitude[2] = {0.0f, 0.0f};
        int product[2] = {0, 0};
        for (int first = q; first < args.ranges; first += 16)
#pragma unroll
            for (int j = 0; j < 4; j++) {                  // loads side by side; beyond the end the last one again
                const i64 range = min(first + 4 * j, args.ranges - 1);
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    magnitude[i] = fmaxf(magnitude[i], magnitudes[range * args.m_pad + i]);
                    product[i] = max(product[i], (int)products[range * args.o_pad * args.m_pad + NGF_TILE_O * i]);
                }
            }
        const int c_exponent = args.c_exponents[batch * args.c_exponents_bs + o0 + column];
#pragma unroll
        for (int i = 0; i < 2; i++) {
#pragma unroll
            for (int bit : {16, 32}) {
                magnitude[i] = fmaxf(magnitude[i], __shfl_xor(magnitude[i], bit));
                product[i] = max(product[i], __shfl_xor(product[i], bit));
            }
            const int exponent = min(min(NGF_EXPONENT_W - ((product[i] >> 7) - 127) - c_exponent, 126 - signs_exponent(magnitude[i])), 126);
            scale[i] = __builtin_ldexpf(1.0f, exponent);
            unscale[i] = 1 - exponent - c_exponent;          // doubled: 2 S - 1 is summed as S - 1/2
        }
    }
    // counts of the lane's rows n for the wave's two m, one dword per block
    const unsigned short *counts = args.counts + batch * args.counts_bs + (i64)(n0 + r) * args.m_pad + m0 + 2 * wave;
    unsigned count[BLOCKS];
    auto load_counts = [&](int chunk) {
#pragma unroll
        for (int block = 0; block < BLOCKS; block++)
            count[block] = *reinterpret_cast<const unsigned *>(counts + ((i64)chunk * args.n_pad + 16 * block) * args.m_pad);
    };
    load_counts(0);
    // the copies are not counted by the compiler: nothing it loads may be under way beside them
    __builtin_amdgcn_s_waitcnt(0x0F70);

    ngf_float4 acc[2][BLOCKS];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int block = 0; block < BLOCKS; block++) acc[i][block] = ngf_float4{0.0f, 0.0f, 0.0f, 0.0f};
    float sum_w[2] = {0.0f, 0.0f};

    auto step = [&](int from, int half) {
        const gram_chunk *positions = lds + from * Tile::POSITION_CHUNKS + (4 * half + q) * Tile::TILE_N + r;
        float c[8];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float4 x = reinterpret_cast<const float4 *>(lds_c)[from * Tile::C_CHUNKS + (4 * half + q) * 32 + 16 * j + column];
            c[4 * j] = x.x; c[4 * j + 1] = x.y; c[4 * j + 2] = x.z; c[4 * j + 3] = x.w;
        }
        gram_half8 w[2][COLUMN_PIECES];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            float a[8];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float4 x = reinterpret_cast<const float4 *>(lds_a)[from * Tile::A_CHUNKS + 32 * wave + 16 * half + 4 * q + 2 * i + j];
                a[4 * j] = x.x; a[4 * j + 1] = x.y; a[4 * j + 2] = x.z; a[4 * j + 3] = x.w;
            }
            gram_chunk first, second;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float a0 = a[2 * j] * scale[i], a1 = a[2 * j + 1] * scale[i];
                const float w0 = a0 * c[2 * j], w1 = a1 * c[2 * j + 1];
                sum_w[i] += w0;
                sum_w[i] += w1;
                // What a pair of W costs is its instructions: 2.4 cycles for one of fp32, 4.6 for a packed or mixed one or a conversion, 8.3
                // for one that rounds into half a register (which the compiler takes for a difference that is rounded at once)
                gram_half2 h1 = __builtin_convertvector(gram_float2{w0, w1}, gram_half2);
                asm("" : "+v"(h1));
                // columns with the first pieces take nothing off: what is left is then W, and its rounding the first piece
                if constexpr (PIECES_IN_COLUMNS) h1 = __builtin_bit_cast(gram_half2, __builtin_bit_cast(unsigned, h1) & (r < 8 ? 0u : ~0u));
                float left0 = __builtin_fmaf(a0, c[2 * j], -(float)h1.x), left1 = __builtin_fmaf(a1, c[2 * j + 1], -(float)h1.y);
                asm("" : "+v"(left0), "+v"(left1));
                const unsigned left = __builtin_bit_cast(unsigned, __builtin_convertvector(gram_float2{left0, left1}, gram_half2));
                first[j] = PIECES_IN_COLUMNS ? left : __builtin_bit_cast(unsigned, h1);
                second[j] = left;
            }
            w[i][0] = __builtin_bit_cast(gram_half8, first);
            if constexpr (!PIECES_IN_COLUMNS) w[i][1] = __builtin_bit_cast(gram_half8, second);
            // where 128 registers are all, W is summed here: left to itself the sum runs beside the matrix instructions, which is faster (8192 x
            // 512 x 16 x 8192 2 %) but keeps a and c until then
            if constexpr (PIECES_IN_COLUMNS && BLOCKS == 4) asm volatile("" : "+v"(sum_w[i]));
        }
        gram_chunk p[3], s[2][2];
        auto compare = [&](int block, const gram_chunk &at, gram_chunk (&into)[2]) {
            const ngf_half2 pair = signs_halves(count[block]);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) into[i][j] = signs_compare(pair[i], at[j]);
        };
#pragma unroll
        for (int block = 0; block < 3 && block < BLOCKS; block++) p[block] = positions[16 * block];
        compare(0, p[0], s[0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int block = 0; block < BLOCKS; block++) {
            if (block + 3 < BLOCKS) p[block % 3] = positions[16 * (block + 3)];
            if (block + 1 < BLOCKS) compare(block + 1, p[(block + 1) % 3], s[(block + 1) % 2]);
#pragma unroll
            for (int piece = COLUMN_PIECES - 1; piece >= 0; piece--)
#pragma unroll
                for (int i = 0; i < 2; i++)
                    acc[i][block] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gram_half8, s[block % 2][i]), w[i][piece], acc[i][block], 0, 0, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
            for (int j = 0; j < 2 * COLUMN_PIECES; j++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 4 / COLUMN_PIECES, 0);
            }
        }
    };
    // the sums over k of the four row quads, half of them off the results of the column (with the pieces in the
    // columns: off the first piece's)
    auto correct = [&]() {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            float total = sum_w[i];
            total += __shfl_xor(total, 16);
            total += __shfl_xor(total, 32);
            const float off = PIECES_IN_COLUMNS && r >= 8 ? 0.0f : 0.5f * total;
#pragma unroll
            for (int block = 0; block < BLOCKS; block++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][block][j] -= off;
            sum_w[i] = 0.0f;
        }
    };

    // Copies go one stage ahead.  (Three buffers and copies two and three stages ahead: the same time; the copies' latency is not
    // what bounds a stage.)
    copy_stage(0);
    int chunk = 0, chunk_left = args.chunk_stages;
    for (int stage = 0; stage < args.stages; stage++) {
        // the wave's own copies have arrived; behind the barrier everybody's have, and the other buffer is free
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        if (chunk_left == 0) {
            load_counts(++chunk);
            chunk_left = args.chunk_stages;
            __builtin_amdgcn_s_waitcnt(0x0F70);
        }
        chunk_left--;
        const int here = stage & 1, other = here ^ 1;
        if (stage + 1 < args.stages) copy_stage(other);
        step(here, 0);
        step(here, 1);
        if (stage % NGF_CORRECT_STAGES == NGF_CORRECT_STAGES - 1 || stage + 1 == args.stages) correct();
    }

    // acc[i][block][j]: m = m0 + 2 wave + i, n = n0 + 16 block + 4 q + j, o = o0 + column.  Through LDS, so that the 16 m
    // of the workgroup are stored together.
    if constexpr (PIECES_IN_COLUMNS) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int block = 0; block < BLOCKS; block++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][block][j] += __shfl_xor(acc[i][block][j], 8);
    }
    float *results = reinterpret_cast<float *>(lds);
    constexpr int PITCH = Tile::RESULT_PITCH;
#pragma unroll
    for (int pass = 0; pass < BLOCKS / Tile::PASS_BLOCKS; pass++) {
        __syncthreads();
#pragma unroll
        for (int within = 0; within < Tile::PASS_BLOCKS; within++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int block = pass * Tile::PASS_BLOCKS + within;
                *reinterpret_cast<float2 *>(results + ((16 * within + 4 * q + j) * 16 + r) * PITCH + 2 * wave) =
                    make_float2(__builtin_ldexpf(acc[0][block][j], unscale[0]), __builtin_ldexpf(acc[1][block][j], unscale[1]));
            }
        __syncthreads();
        constexpr int QUADS = NGF_TILE_M / 4;
        const int quad = tid % QUADS;
        const int m = m0 + 4 * quad;
#pragma unroll
        for (int row = tid / QUADS; row < 256 * Tile::PASS_BLOCKS; row += NGF_THREADS / QUADS) {
            const int o = o0 + (row & 15), n = n0 + 16 * Tile::PASS_BLOCKS * pass + (row >> 4);
            if (o >= g.o || n >= g.n || (PIECES_IN_COLUMNS && (row & 8))) continue;
            const float4 v = *reinterpret_cast<const float4 *>(results + row * PITCH + 4 * quad);
            float *dst = g.e + batch * g.e_bs + (i64)o * g.e_ld_o + (i64)n * g.e_ld_n + m;
            if (g.e_vec && m + 3 < g.m) {
                *reinterpret_cast<float4 *>(dst) = v;
            } else {
                if (m < g.m) dst[0] = v.x;
                if (m + 1 < g.m) dst[1] = v.y;
                if (m + 2 < g.m) dst[2] = v.z;
                if (m + 3 < g.m) dst[3] = v.w;
            }
        }
    }
}

}  // namespace kmc
