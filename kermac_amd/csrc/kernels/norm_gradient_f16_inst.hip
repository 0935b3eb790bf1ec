// Host side of the L1 kernel gradient on the fp16 matrix instruction (norm_gradient_f16.hpp): when
// it applies, how the caller's workspace is divided, and the launches.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <type_traits>

#include "../host/host_common.hpp"
#include "../host/dispatch_rules.hpp"
#include "launch.hpp"
#include "norm_gradient_f16.hpp"

namespace kmc_host {

namespace {

constexpr int64_t REGION_ALIGN = 256;

struct GradientLayout {
    int stages, n_pad, m_pad, k_pad, o_pad, ranges;
    int chunks, chunk_k, keys, copy_k, copy_blocks;
    bool sort_d;
    int sort_batches, a_batches, c_batches, product_batches;
    int64_t positions_bs, counts_bs, a_copy_bs, a_magnitudes_bs, products_bs, c_copy_bs;      // in elements
    int64_t positions, counts, a_copy, a_magnitudes, products, c_copy, c_exponents;           // byte offsets into the workspace
    int64_t bytes;
};

int64_t place(int64_t &cursor, int64_t bytes)
{
    const int64_t at = cursor;
    cursor = (cursor + bytes + REGION_ALIGN - 1) / REGION_ALIGN * REGION_ALIGN;
    return at;
}

int64_t round_up(int64_t value, int64_t multiple) { return (value + multiple - 1) / multiple * multiple; }

// The route pays where the fp32 kernels are bound by their matrix or vector instructions: enough
// terms to carry the extra launch and the ranking, and more than two outputs (a workgroup costs the same for 1 .. 8 and for
// 9 .. 16 outputs; the vector kernel for one or two is cheap).  Few outputs make the fp32 kernels cheaper nearly in proportion and not the
// route, so the terms are asked for in proportion: 4e8 at 16 outputs, 1.6e9 at 4.  Its smallest tile holds 32 n.
// The limits are those of a slower kernel with five more launches.  Of 57 shapes that they send down the route the present one is 1.55 times as fast as the fp32
// kernels or more (11200 x 112 x 16 x 320 1.55, 4000 x 32 x 16 x 4000 1.80, 6862 x 105 x 24 x 417 1.96): they lose nothing, and leave calls to
// the fp32 kernels that the route would win; the Python layer takes those by models of both times (cdist_grad.py).
// KERMAC_AMD_GRADIENT_F16_MIN_TERMS replaces the conditions by a number of terms (read on every
// call, so that a test can send small shapes down the route).
bool f16_pays(const kmc_norm_gradient_params *p)
{
    const char *text = std::getenv("KERMAC_AMD_GRADIENT_F16_MIN_TERMS");
    const double forced = text ? std::atof(text) : 0.0;
    const double terms = static_cast<double>(p->m) * p->n * p->k * p->l;
    if (forced > 0.0) return terms >= forced;
    if (p->flags & KMC_FLAG_GRAM_WORKSPACE_ANY_SIZE) return true;
    // more than 16 outputs: the ranking serves all blocks of outputs, while the fp32 kernels go to their 32-column tiles (fp32 / route, us:
    // 704 x 48 x 32 x 1024, 3.5e7 terms, 102 / 59; 832 x 352 x 128 x 320, 9.4e7, 250 / 122; 576 x 48 x 64 x 2816, 7.8e7, 218 / 131)
    namespace r = kmc_rules;
    if (p->o > 16) return p->n >= r::GRADIENT_F16_MIN_N && terms >= static_cast<double>(r::GRADIENT_F16_MANY_OUTPUTS_MIN_TERMS);
    return p->o >= r::GRADIENT_F16_MIN_OUTPUTS && p->n >= r::GRADIENT_F16_MIN_N &&
           terms * p->o >= static_cast<double>(r::GRADIENT_F16_MIN_TERMS_TIMES_OUTPUTS);
}

bool gradient_layout(const kmc_norm_gradient_params *p, GradientLayout *layout)
{
    if (p->norm_type != KMC_NORM_L1 || p->m < 1 || p->n < 1 || p->o < 1 || p->k < 1 || p->l < 1) return false;
    if (!f16_pays(p)) return false;
    // a row n is a row of blockIdx.y in other kernels of its size: the fp32 kernels keep what they had
    if (round_up(p->n, 32) > 65535 || static_cast<int64_t>(p->l) * (p->o / 64 + 1) > 65535) return false;
    const int64_t k_pad = round_up(p->k, kmc::NGF_STAGE_K), m_pad = round_up(p->m, kmc::NGF_M_PAD);
    const int64_t n_pad = round_up(p->n, kmc::NGF_N_PAD), o_pad = round_up(p->o, kmc::NGF_TILE_O);
    // a dimension of a grid holds fewer than 2^32 threads
    const int64_t threads = int64_t{1} << 32;
    // the shorter row of a pair is sorted; rows of B longer than the sort takes are cut into chunks
    layout->sort_d = p->m < p->k && p->m <= kmc::NGF_MAX_CHUNK;
    layout->chunks = layout->sort_d ? 1 : (p->k + kmc::NGF_MAX_CHUNK - 1) / kmc::NGF_MAX_CHUNK;
    layout->chunk_k = static_cast<int>(round_up((p->k + layout->chunks - 1) / layout->chunks, kmc::NGF_STAGE_K));
    layout->chunks = (p->k + layout->chunk_k - 1) / layout->chunk_k;
    layout->keys = layout->sort_d ? p->m : layout->chunk_k;
    // fewer k per tile of A where that leaves fewer tiles than two per CU
    const int64_t tiles_m = (m_pad + kmc::NGF_COPY_M - 1) / kmc::NGF_COPY_M, tiles = tiles_m * (o_pad / kmc::NGF_TILE_O);
    layout->copy_k = kmc::NGF_COPY_MAX_K;
    while (layout->copy_k > kmc::NGF_COPY_MIN_K && tiles * p->l * ((k_pad + layout->copy_k - 1) / layout->copy_k) < 1024) layout->copy_k /= 2;
    layout->ranges = static_cast<int>((k_pad + layout->copy_k - 1) / layout->copy_k);
    const int64_t copy_blocks = round_up(tiles_m * layout->ranges, kmc::BK_XCDS) * (o_pad / kmc::NGF_TILE_O);
    const int64_t prepare_blocks = static_cast<int64_t>(p->n) * layout->chunks + copy_blocks + o_pad + 2 * kmc::NGF_PREPARE_GROUP;
    if (prepare_blocks * kmc::NGF_PREPARE_THREADS >= threads || m_pad / kmc::NGF_TILE_M * kmc::NGF_THREADS >= threads || k_pad > INT32_MAX ||
        m_pad > INT32_MAX || o_pad > INT32_MAX)
        return false;
    layout->copy_blocks = static_cast<int>(copy_blocks);
    layout->stages = static_cast<int>(k_pad / kmc::NGF_STAGE_K);
    layout->n_pad = static_cast<int>(n_pad); layout->m_pad = static_cast<int>(m_pad);
    layout->k_pad = static_cast<int>(k_pad); layout->o_pad = static_cast<int>(o_pad);
    layout->sort_batches = p->b_bs == 0 && p->d_bs == 0 ? 1 : p->l;
    layout->a_batches = p->a_bs == 0 ? 1 : p->l;
    layout->c_batches = p->c_bs == 0 ? 1 : p->l;
    layout->positions_bs = k_pad * n_pad;
    layout->counts_bs = static_cast<int64_t>(layout->chunks) * n_pad * m_pad;
    layout->a_copy_bs = m_pad * k_pad;
    layout->a_magnitudes_bs = static_cast<int64_t>(layout->ranges) * m_pad;
    layout->product_batches = layout->a_batches > 1 || layout->c_batches > 1 ? p->l : 1;
    layout->products_bs = layout->ranges * o_pad * m_pad;
    layout->c_copy_bs = o_pad * k_pad;
    int64_t cursor = 0;
    layout->positions = place(cursor, layout->sort_batches * layout->positions_bs * 2);
    layout->counts = place(cursor, layout->sort_batches * layout->counts_bs * 2);
    layout->a_copy = place(cursor, layout->a_batches * layout->a_copy_bs * 4);
    layout->a_magnitudes = place(cursor, layout->a_batches * layout->a_magnitudes_bs * 4);
    layout->products = place(cursor, layout->product_batches * layout->products_bs * 2);
    layout->c_copy = place(cursor, layout->c_batches * layout->c_copy_bs * 4);
    layout->c_exponents = place(cursor, layout->c_batches * o_pad * 4);
    layout->bytes = cursor;
    return true;
}

// Tile of the product in n: 16, 12, 8, 4 or 2 blocks of 16, as blocks and the cost of a workgroup, the second with the pieces in the
// columns, in us of two rounds of the 256 CUs at K = 8192 for those that have a CU to themselves.  A step costs about as much as 8 blocks beside its
// blocks, W above all, so wide tiles are cheaper per result, unless they are too few for the CUs or their last round is nearly empty.  Up to 4 blocks
// two workgroups share a CU and hide each other's ends: their cost is fitted to 120 shapes with every tile, K = 250 .. 5000.  12 / 4 blocks, us:
// 3264 x 304 x 16 x K, K = 800 119 / 106, K = 5000 482 / 461; 6000 x 147 x 16 x 5000 502 / 561; 16 / 4 blocks: 9000 x 200 x 16 x 5000 882 / 965.  (Below about 500 k
// the ends weigh more than this counts: K = 250 there 120 / 102.)
// 12 is for n that fill little of the second half of a larger tile: with the others only / with
// 12, us: 3000 x 147 x 64 x 4000 714 / 577, 2000 x 300 x 20 x 2000 301 / 212, 4000 x 147 x 32 x 4000 481 / 399.
constexpr struct { int blocks, cost, cost_in_columns; } PRODUCT_TILES[] = {{16, 936, 743}, {12, 772, 642}, {8, 621, 536}, {4, 355, 295}, {2, 255, 225}};

struct ProductTile {
    int blocks;
    int64_t cost;
};

ProductTile tile_for(const kmc_norm_gradient_params *p, int o_chunks, bool pieces_in_columns)
{
    ProductTile best = {0, o_chunks ? INT64_MAX : 0};
    for (const auto &tile : PRODUCT_TILES) {
        const int tile_n = 16 * tile.blocks;
        // 12 where its last tile ends inside the padded rows
        if (tile.blocks == 12 && round_up(p->n, tile_n) > round_up(p->n, kmc::NGF_N_PAD)) continue;
        const int64_t workgroups = static_cast<int64_t>((p->n + tile_n - 1) / tile_n) * ((p->m + kmc::NGF_TILE_M - 1) / kmc::NGF_TILE_M) * p->l * o_chunks;
        const int64_t cost = round_up(workgroups, 256) / 256 * (pieces_in_columns ? tile.cost_in_columns : tile.cost);
        if (cost < best.cost) best = {tile.blocks, cost};
    }
    return best;
}

template <int BLOCKS, bool PIECES_IN_COLUMNS>
hipError_t launch_product(kmc::NormGradientF16Args &args, int o_begin, int o_chunks, hipStream_t stream)
{
    using Tile = kmc::GradientF16Tile<BLOCKS>;
    const int per_launch = 65535 / args.g.l;         // blockIdx.z = batch entry x block of 16 outputs
    for (int first = 0; first < o_chunks; first += per_launch) {
        const int chunks = o_chunks - first < per_launch ? o_chunks - first : per_launch;
        args.o_begin = o_begin + first * kmc::NGF_TILE_O;
        args.g.o_chunks = chunks;
        const dim3 grid((args.g.m + kmc::NGF_TILE_M - 1) / kmc::NGF_TILE_M, (args.g.n + Tile::TILE_N - 1) / Tile::TILE_N,
                        static_cast<unsigned>(args.g.l) * chunks);
        const hipError_t status = launch(kmc::norm_gradient_l1_f16<BLOCKS, PIECES_IN_COLUMNS>, grid, dim3(kmc::NGF_THREADS), stream, args);
        if (status != hipSuccess) return status;
    }
    return hipSuccess;
}

template <bool PIECES_IN_COLUMNS>
hipError_t launch_products(int blocks, kmc::NormGradientF16Args &args, int o_begin, int o_chunks, hipStream_t stream)
{
    switch (blocks) {
    case 16: return launch_product<16, PIECES_IN_COLUMNS>(args, o_begin, o_chunks, stream);
    case 12: return launch_product<12, PIECES_IN_COLUMNS>(args, o_begin, o_chunks, stream);
    case 8: return launch_product<8, PIECES_IN_COLUMNS>(args, o_begin, o_chunks, stream);
    case 4: return launch_product<4, PIECES_IN_COLUMNS>(args, o_begin, o_chunks, stream);
    default: return launch_product<2, PIECES_IN_COLUMNS>(args, o_begin, o_chunks, stream);
    }
}

}  // namespace

int64_t norm_gradient_f16_bytes(const kmc_norm_gradient_params *p)
{
    GradientLayout layout;
    return gradient_layout(p, &layout) ? layout.bytes : 0;
}

// `*taken` says whether the route applied (and the launches were made); if not, nothing was launched.
hipError_t launch_norm_gradient_f16(const kmc_norm_gradient_params *p, bool a_vec, bool e_vec, hipStream_t stream, bool *taken)
{
    *taken = false;
    GradientLayout layout;
    if (!p->workspace || !gradient_layout(p, &layout) || p->workspace_bytes < layout.bytes ||
        (reinterpret_cast<uintptr_t>(p->workspace) & (REGION_ALIGN - 1)) != 0)
        return hipSuccess;
    char *workspace = static_cast<char *>(p->workspace);
    kmc::GradientPrepareArgs prepare = {};
    prepare.m = p->m; prepare.n = p->n; prepare.o = p->o; prepare.k = p->k;
    prepare.a = p->a; prepare.a_ld = p->a_ld; prepare.a_bs = p->a_bs; prepare.a_vec = a_vec;
    prepare.b = p->b; prepare.b_ld = p->b_ld; prepare.b_bs = p->b_bs;
    prepare.c = p->c; prepare.c_ld = p->c_ld; prepare.c_bs = p->c_bs;
    prepare.d = p->d; prepare.d_ld = p->d_ld; prepare.d_bs = p->d_bs;
    prepare.positions = reinterpret_cast<unsigned short *>(workspace + layout.positions); prepare.positions_bs = layout.positions_bs;
    prepare.counts = reinterpret_cast<unsigned short *>(workspace + layout.counts); prepare.counts_bs = layout.counts_bs;
    prepare.a_copy = reinterpret_cast<float *>(workspace + layout.a_copy); prepare.a_copy_bs = layout.a_copy_bs;
    prepare.a_magnitudes = reinterpret_cast<float *>(workspace + layout.a_magnitudes); prepare.a_magnitudes_bs = layout.a_magnitudes_bs;
    prepare.products = reinterpret_cast<unsigned short *>(workspace + layout.products); prepare.products_bs = layout.products_bs;
    prepare.c_copy = reinterpret_cast<float *>(workspace + layout.c_copy); prepare.c_copy_bs = layout.c_copy_bs;
    prepare.c_exponents = reinterpret_cast<int *>(workspace + layout.c_exponents); prepare.c_exponents_bs = layout.o_pad;
    prepare.n_pad = layout.n_pad; prepare.m_pad = layout.m_pad; prepare.k_pad = layout.k_pad; prepare.o_pad = layout.o_pad;
    prepare.sort_d = layout.sort_d;
    prepare.copy_k = layout.copy_k; prepare.ranges = layout.ranges; prepare.chunk_k = layout.chunk_k;
    prepare.sort_blocks = p->n * layout.chunks;
    prepare.copy_blocks = layout.copy_blocks;
    prepare.sort_batches = layout.sort_batches; prepare.a_batches = layout.a_batches; prepare.c_batches = layout.c_batches;
    prepare.product_batches = layout.product_batches;
    const int batches = layout.sort_batches > 1 || layout.a_batches > 1 || layout.c_batches > 1 ? p->l : 1;
    prepare.sort_groups = (prepare.sort_blocks + kmc::NGF_PREPARE_GROUP - 1) / kmc::NGF_PREPARE_GROUP;
    prepare.copy_groups = (prepare.copy_blocks + kmc::NGF_PREPARE_GROUP - 1) / kmc::NGF_PREPARE_GROUP;
    const dim3 prepare_grid((prepare.sort_groups + prepare.copy_groups) * kmc::NGF_PREPARE_GROUP + layout.o_pad, batches);
    const dim3 prepare_threads(kmc::NGF_PREPARE_THREADS);
    hipError_t status;
    if (layout.keys <= 1024) status = launch(kmc::gradient_signs_prepare<2>, prepare_grid, prepare_threads, stream, prepare);
    else if (layout.keys <= 2048) status = launch(kmc::gradient_signs_prepare<3>, prepare_grid, prepare_threads, stream, prepare);
    else if (layout.keys <= 4096) status = launch(kmc::gradient_signs_prepare<4>, prepare_grid, prepare_threads, stream, prepare);
    else if (layout.keys <= 8192) status = launch(kmc::gradient_signs_prepare<5>, prepare_grid, prepare_threads, stream, prepare);
    else status = launch(kmc::gradient_signs_prepare<6>, prepare_grid, prepare_threads, stream, prepare);
    if (status != hipSuccess) return status;

    kmc::NormGradientF16Args args = {};
    args.g.m = p->m; args.g.n = p->n; args.g.o = p->o; args.g.k = p->k; args.g.l = p->l;
    args.g.e = p->e; args.g.e_ld_n = p->e_ld_n; args.g.e_ld_o = p->e_ld_o; args.g.e_bs = p->e_bs;
    args.g.e_vec = e_vec;
    args.positions = prepare.positions; args.counts = prepare.counts;
    args.positions_bs = layout.sort_batches > 1 ? layout.positions_bs : 0;
    args.counts_bs = layout.sort_batches > 1 ? layout.counts_bs : 0;
    args.a_copy = prepare.a_copy; args.a_copy_bs = layout.a_batches > 1 ? layout.a_copy_bs : 0;
    args.a_magnitudes = prepare.a_magnitudes; args.a_magnitudes_bs = layout.a_batches > 1 ? layout.a_magnitudes_bs : 0;
    args.products = prepare.products; args.products_bs = layout.product_batches > 1 ? layout.products_bs : 0;
    args.c_copy = prepare.c_copy; args.c_copy_bs = layout.c_batches > 1 ? layout.c_copy_bs : 0;
    args.c_exponents = prepare.c_exponents; args.c_exponents_bs = layout.c_batches > 1 ? layout.o_pad : 0;
    args.n_pad = layout.n_pad; args.m_pad = layout.m_pad; args.k_pad = layout.k_pad; args.o_pad = layout.o_pad; args.ranges = layout.ranges;
    args.chunk_stages = layout.chunk_k / kmc::NGF_STAGE_K; args.stages = layout.stages;
    // Blocks of 16 outputs; what is left up to 8 in the first half of the columns, its second pieces in the other, in a launch behind the
    // first, with a tile of its own, unless one launch with a block of 16 for them fills its rounds better: 2794 x 344 x 24 x 838, 350
    // tiles of 192 n, 244 us in two launches and 196 in one
    const int left = p->o % kmc::NGF_TILE_O, all_chunks = (p->o + kmc::NGF_TILE_O - 1) / kmc::NGF_TILE_O;
    const bool may_split = left > 0 && left <= 8;
    const ProductTile whole = tile_for(p, all_chunks, false), full = tile_for(p, all_chunks - 1, false), rest = tile_for(p, 1, true);
    if (may_split && full.cost + rest.cost < whole.cost) {
        if (all_chunks > 1) status = launch_products<false>(full.blocks, args, 0, all_chunks - 1, stream);
        if (status == hipSuccess) status = launch_products<true>(rest.blocks, args, p->o - left, 1, stream);
    } else {
        status = launch_products<false>(whole.blocks, args, 0, all_chunks, stream);
    }
    if (status == hipSuccess) *taken = true;
    return status;
}

}  // namespace kmc_host
