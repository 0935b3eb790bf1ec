// Host side of the two-piece fp16 matrix-core path for large squared-difference problems
// (gram_f16_wide.hpp): when it applies, how the caller's workspace is divided, and the launches.
// One instantiation per kernel: the layout of an operand in memory is a run-time property of the
// two row kernels and does not reach the product kernel at all.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <mutex>
#include <unordered_map>

#include "../host/host_common.hpp"
#include "../host/dispatch_rules.hpp"
#include "launch.hpp"
#include "../host/contraction.hpp"
#include "gram_f16_wide.hpp"
#include "norm_gradient_l2_wide.hpp"

namespace kmc_host {

namespace {

constexpr int64_t REGION_ALIGN = 256;

struct OperandRegions {
    int rows_pad, batches;
    int slices_per_range, ranges;    // of the partial sums of squares
    bool once;               // gram_rows_once makes the pieces
    int64_t pieces_bs;       // chunks per batch entry
    int64_t stats_bs;        // floats per batch entry, for the squares and for the magnitudes
    int64_t pieces, squares, magnitudes, unscale;   // byte offsets into the workspace
};

struct WideLayout {
    int slices;
    int tiles_m, tiles_n;       // of GW_TILE x GW_TILE
    OperandRegions a, b;
    int64_t sample;         // byte offset of the words of gram_probe_operands
    int64_t centre = 0, centre_floats = 0;      // byte offset of the centre that the route takes for itself, floats per batch entry (0: it takes none)
    int centre_batches = 1;
    int64_t products = 0, stamps = 0;           // byte offsets of a contraction's products and stamps
    int64_t bytes;
};

// Whether the route pays for its extra launches, for a caller who leaves that to the library.  (With KMC_FLAG_GRAM_WORKSPACE_ANY_SIZE the caller has decided: the Python
// layer's default mode does for nearly all squared differences from K = 128 on and for products with coefficients, by the rules and figures in
// build_a_kernel.py and kernel_coefficients.py.)  Tiles are counted in 256 x 256, the rows that an operand is padded to.
// The lines for squared differences stand where the one-step kernels and a slower product kernel, one workgroup of 256 x 256 per CU, crossed: tiles over the batch and tiles * k; tiles
// in both directions of an entry, since the split is paid per row and earned back per tile the row meets; little padding.  The present kernel is
// faster almost everywhere, so that they keep some calls on a slower kernel and send hardly any to one.  One-step / route, us, of calls that they leave to
// the one-step kernel: k contiguous 1500 x 1500 x 784 102 / 50, 2000 x 2000 x 256 60 / 41, 8 x 512 x 512 x 784 64 / 53, 100 x 50000 x 784 185 / 142; rows contiguous 3000 x 3000 x 784
// 140 / 98, 1000 x 30000 x 256 161 / 111; the other way round, 16 x 512 x 512 x 2048 with k contiguous, 144 / 171.
// KERMAC_AMD_WIDE_MIN_TILES = t replaces the rule by "at least t tiles" (read on every call, so that
// a test can send small shapes down the route).
// Sums of products have no one-step matrix-core kernel to fall back to: the alternative is the direct
// kernel, which the route beats much earlier (direct / route time: 64 tiles 1.04 .. 1.42 at K = 1024,
// 0.82 .. 1.04 at K = 512; 256 tiles 1.25 at K = 256, 0.86 at K = 128; 1024 tiles 1.17 .. 1.35 at K = 128,
// 0.91 .. 1.02 at K = 64; 64 batch entries of 2 x 2 tiles 1.5, 118 x 2 tiles 1.9).  From K = 256 on it is
// taken from 32 tiles and tiles * k = 24576 on whatever the padding (8 entries of 512 x 512 x 784 1.3 .. 1.4, at
// K = 3072 1.7 .. 1.9; 4 of 1000 x 1000 x 784 1.7; 144 tiles at K = 256 1.2 .. 1.3; 300 x 30000, 41 % of the tiles
// padding, 1.1 .. 1.2 at K = 256 and 1.7 .. 1.9 beyond; at K = 256 with 64 tiles 0.8 .. 0.9), but a single problem
// only from 64 tiles on: the direct path cuts such a call over k (1500 x 1500, 36 tiles: 0.77 .. 0.84).
//
// Operands with k contiguous (row-major, as torch allocates them): the one-step kernels stage such operands
// more slowly, the route splits them once and walks pieces whose layout is its own, so it pays earlier
// and whatever the shape of a batch entry.  Not for a dimension that half a tile holds, where the 128 x 128 tiles of the
// one-step kernels waste half as much.
//
// A set against itself (the tiles of one triangle): one round of workgroups either way, whose walk is the route's faster one
// (one-step split kernel / route, us, k contiguous: 1400 points, 21 tiles, at K = 784 77 / 63; 2000 at K = 256 66 / 52, at
// K = 784 152 / 65; rows contiguous: 2400 at K = 1024 106 / 90; 3000 at K = 128 46 / 70).
bool wide_pays(int64_t m, int64_t n, int64_t tiles_m, int64_t tiles_n, int64_t tiles, int k, bool products, bool k_contiguous,
               bool batched, bool symmetric)
{
    const char *text = std::getenv("KERMAC_AMD_WIDE_MIN_TILES");
    const int forced = text ? std::atoi(text) : 0;
    if (forced > 0) return tiles >= forced && k >= 1;
    namespace r = kmc_rules;
    if (k_contiguous && !products && k >= r::WIDE_K_CONTIGUOUS_MIN_K && tiles >= r::WIDE_K_CONTIGUOUS_MIN_TILES &&
        tiles * k >= r::WIDE_K_CONTIGUOUS_MIN_TILES_TIMES_K && m >= r::WIDE_K_CONTIGUOUS_MIN_ROWS && n >= r::WIDE_K_CONTIGUOUS_MIN_ROWS)
        return true;
    if (symmetric && !products &&
        (k_contiguous ? k >= r::WIDE_SYMMETRIC_K_CONTIGUOUS_MIN_K && tiles >= r::WIDE_SYMMETRIC_K_CONTIGUOUS_MIN_TILES &&
                            tiles * k >= r::WIDE_SYMMETRIC_K_CONTIGUOUS_MIN_TILES_TIMES_K
                      : tiles >= r::WIDE_SYMMETRIC_MIN_TILES && tiles * k >= r::WIDE_SYMMETRIC_MIN_TILES_TIMES_K))
        return true;
    const bool little_padding = 100 * m * n >= (100 - r::WIDE_MAX_PADDING_PERCENT) * (tiles_m * kmc::GW_TILE) * (tiles_n * kmc::GW_TILE);
    if (products && k >= r::DOT_LONG_K && tiles * k >= r::DOT_LONG_MIN_TILES_TIMES_K &&
        tiles >= (batched ? r::DOT_LONG_MIN_TILES_BATCHED : r::DOT_LONG_MIN_TILES_SINGLE))
        return true;
    if (products) return k >= r::DOT_MIN_K && tiles >= r::DOT_MIN_TILES && tiles * k >= r::DOT_MIN_TILES_TIMES_K && little_padding;
    // (from 768 tiles on the route is as fast as the one-step kernel also for the shortest contractions
    // it takes, 8192 x 8192 x 64 180 us against 187, and ahead of the direct kernel, 236)
    // (long contractions of few tiles, one-step / route, us: 1500 x 1500 x 2048 129 / 75, 2048 x 2048 x 2048 173 / 88, 1800 x 1500 x 4000 294 / 126)
    const bool long_walk = k >= r::WIDE_LONG_MIN_K && ((m + 127) / 128) * ((n + 127) / 128) >= r::WIDE_LONG_MIN_TILES && !k_contiguous && !symmetric;
    if (!long_walk && (k < r::WIDE_MIN_K || tiles < r::WIDE_MIN_TILES || (tiles * k < r::WIDE_MIN_TILES_TIMES_K && tiles < r::WIDE_TILES_FOR_ANY_K))) return false;
    if (2 * tiles_m * tiles_n < r::WIDE_MIN_TILES_PER_SIDE_X2 * (tiles_m + tiles_n)) return false;
    return little_padding;
}

int64_t place(int64_t &cursor, int64_t bytes)
{
    const int64_t at = cursor;
    cursor = (cursor + bytes + REGION_ALIGN - 1) / REGION_ALIGN * REGION_ALIGN;
    return at;
}

void place_operand(OperandRegions &r, int rows, bool broadcast, int l, bool once, const WideLayout &layout, int64_t &cursor)
{
    // at most 8 ranges of K per row (9 by the rounding): enough workgroups for the row kernels, few partial sums
    r.once = once;
    r.slices_per_range = once ? layout.slices : layout.slices / 8 > 8 ? (layout.slices + 7) / 8 : 8;
    r.ranges = (layout.slices + r.slices_per_range - 1) / r.slices_per_range;
    static_assert(kmc::GW_MAX_RANGES == 9, "the two lines above");
    r.rows_pad = (rows + kmc::GW_TILE - 1) / kmc::GW_TILE * kmc::GW_TILE;
    r.batches = broadcast ? 1 : l;
    r.pieces_bs = static_cast<int64_t>(2 * ((layout.slices + 1) / 2)) * kmc::GW_SEGMENTS * r.rows_pad;      // whole steps of the walk
    r.stats_bs = static_cast<int64_t>(r.ranges) * r.rows_pad;
    r.pieces = place(cursor, r.batches * r.pieces_bs * 16);
    r.squares = place(cursor, r.batches * r.stats_bs * 4);
    r.magnitudes = place(cursor, r.batches * r.stats_bs * 4);
    r.unscale = place(cursor, static_cast<int64_t>(r.batches) * r.rows_pad * 4);
}

// Grid, slices and the regions of both operands in the workspace; tiles_m and tiles_n are set.
// a_shared, b_shared: one operand for all batch entries.  a_once, b_once: one launch makes its pieces (made_once).
// repair_tiles: the list of the repair launch, as long as all tiles of the result.
bool place_wide(int m, int n, int k, int l, bool a_shared, bool b_shared, bool a_once, bool b_once, bool symmetric, int64_t repair_tiles, WideLayout *layout)
{
    // room for any tile of the product kernel in a grid, n tiles padded to the XCDs
    if (static_cast<int64_t>(layout->tiles_m) * (layout->tiles_n + kmc::BK_XCDS) * 4 > 0x7fffffff) return false;
    layout->slices = (k + kmc::BK_TILE_K - 1) / kmc::BK_TILE_K;
    int64_t cursor = 0;
    place_operand(layout->a, m, a_shared, l, a_once, *layout, cursor);
    // behind the region of a, where it stays when b grows or shrinks: the split of a may be kept
    layout->centre = layout->centre_floats ? place(cursor, 4 * layout->centre_floats * layout->centre_batches) : 0;
    if (symmetric) layout->b = layout->a;      // one panel, split once
    else place_operand(layout->b, n, b_shared, l, b_once, *layout, cursor);
    layout->sample = place(cursor, kmc::BK_SAMPLE_BYTES + 4 * (kmc::BK_REPAIR_WORDS + repair_tiles));
    layout->bytes = cursor;
    return true;
}

bool rows_vec(const float *x, int64_t ld, int64_t bs, int majorness, bool scalar_only)
{
    return majorness == KMC_ROW_MAJOR && !scalar_only && aligned16(x) && ld % 4 == 0 && bs % 4 == 0;
}

// Whether gram_rows_once or gram_columns_once makes the pieces of an operand: up to 2048 k its values, in chunks up to 1024, stay in registers; longer ones are read twice by
// the same workgroup (LONG), which is ahead of two launches for rows that lie apart or cannot be read 16 bytes at a time, and behind for others, whose k
// the two launches share among nine workgroups.  Two launches / LONG, us of a call: rows contiguous 197 x 7052 x 3328 166 / 154, 3000 x 3000 x 8000 637 / 547, 8000 x 8000 x 3000
// 1018 / 980, 20000 x 20000 x 2304 4490 / 4414; k contiguous, not aligned, 4 x 3840 x 347 x 2767 767 / 317, 2 x 192 x 7002 x 3730 683 / 345; aligned 197 x 7052 x 3328
// 167 / 184, 3000 x 3000 x 8000 631 / 656, 8000 x 8000 x 3000 1060 / 1059, 20000 x 20000 x 2304 4552 / 4718.  Two launches / one pass of 2048 k: 2000 x 2000 x 2048 109 / 84,
// 8000 x 8000 x 1300 504 / 476, 200 x 60000 x 1030 793 / 295.
bool made_once(const float *x, int64_t ld, int64_t bs, int majorness, int flags, int k)
{
    return k <= 2 * kmc::GRO_HELD_K || (k <= kmc::GRO_MAX_K && !rows_vec(x, ld, bs, majorness, (flags & KMC_FLAG_FORCE_SCALAR_ACCESS) != 0));
}

bool wide_layout(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, WideLayout *layout)
{
    const bool squared_differences = (p->flags & KMC_FLAG_L2_GRAM_BF16) && p->inner_operator == KMC_OP_DIFF && p->inner_power == KMC_POW_SQUARE;
    const bool products = (p->flags & KMC_FLAG_DOT_PIECES) && p->inner_operator == KMC_OP_DOT && p->inner_power == KMC_POW_NOOP;
    if (!squared_differences && !products) return false;
    if (args.m < 1 || args.n < 1 || args.l < 1) return false;
    layout->tiles_m = (args.m + kmc::GW_TILE - 1) / kmc::GW_TILE;
    layout->tiles_n = (args.n + kmc::GW_TILE - 1) / kmc::GW_TILE;
    // a panel against itself: the tiles on and below the diagonal
    const int64_t tiles = args.symmetric ? static_cast<int64_t>(layout->tiles_m) * (layout->tiles_m + 1) / 2
                                         : static_cast<int64_t>(layout->tiles_m) * layout->tiles_n;
    const bool k_contiguous = p->a_majorness == KMC_ROW_MAJOR && p->b_majorness == KMC_ROW_MAJOR;
    const bool asked_for = (p->flags & KMC_FLAG_GRAM_WORKSPACE_ANY_SIZE) && args.k >= 1;
    if (!asked_for && !wide_pays(args.m, args.n, layout->tiles_m, layout->tiles_n, tiles * args.l, args.k, products, k_contiguous, args.l > 1, args.symmetric)) return false;
    // an operand that is the same for every batch entry is split once, unless the centre differs
    // (products have no centre: the caller's parameter block carries none into `args`)
    const bool own_centre = squared_differences && (p->flags & KMC_FLAG_GRAM_OWN_CENTRE);
    layout->centre_batches = own_centre && args.a_bs != 0 ? args.l : 1;
    layout->centre_floats = own_centre ? 2 * ((args.k + kmc::GRAM_CENTRE_PAD - 1) / kmc::GRAM_CENTRE_PAD * kmc::GRAM_CENTRE_PAD) + kmc::GRAM_CENTRE_PAD : 0;
    const int64_t ids = static_cast<int64_t>(args.grid_width) * args.l;
    const bool one_centre = products || (own_centre ? layout->centre_batches == 1 : !args.centre || args.centre_bs == 0);
    return place_wide(args.m, args.n, args.k, args.l, args.a_bs == 0 && one_centre, args.b_bs == 0 && one_centre,
                      made_once(args.a, args.a_ld, args.a_bs, p->a_majorness, p->flags, args.k), made_once(args.b, args.b_ld, args.b_bs, p->b_majorness, p->flags, args.k),
                      args.symmetric, squared_differences && ids >= kmc::BK_REPAIR_MIN_TILES && ids <= kmc::BK_REPAIR_MAX_TILES ? ids : 0, layout);
}

kmc::GramRowsArgs rows_args(const float *x, int64_t ld, int64_t bs, int rows, int majorness, bool scalar_only,
                            const kmc::BuildKernelArgs &args, const WideLayout &layout, const OperandRegions &r, char *workspace,
                            int centre_pairs = 0)
{
    kmc::GramRowsArgs rows_of = {};
    rows_of.x = x; rows_of.ld = ld; rows_of.bs = bs;
    rows_of.rows = rows; rows_of.k = args.k;
    rows_of.row_major = majorness == KMC_ROW_MAJOR;
    rows_of.vec = rows_vec(x, ld, bs, majorness, scalar_only);
    rows_of.centre = args.centre; rows_of.centre_bs = args.centre_bs;
    rows_of.centre_pairs = centre_pairs;
    rows_of.pieces = reinterpret_cast<kmc::gram_chunk *>(workspace + r.pieces); rows_of.pieces_bs = r.pieces_bs;
    rows_of.squares = reinterpret_cast<float *>(workspace + r.squares);
    rows_of.magnitudes = reinterpret_cast<float *>(workspace + r.magnitudes);
    rows_of.unscale = reinterpret_cast<float *>(workspace + r.unscale);
    rows_of.stats_bs = r.stats_bs; rows_of.unscale_bs = r.rows_pad;
    rows_of.rows_pad = r.rows_pad; rows_of.slices = layout.slices;
    rows_of.slices_per_range = r.slices_per_range; rows_of.ranges = rows_of.magnitude_ranges = r.ranges;
    rows_of.zero_slices = layout.slices & 1;      // the walk takes two slices per step
    return rows_of;
}

// What the split of `a` in a workspace was made from, kept on the host per workspace address: a call with
// KMC_FLAG_GRAM_A_KEPT skips the split only when this record says that the previous split through this
// workspace was of the same operand, shape, centre and layout; anything else (another operand, a call
// that did not take this route in between and left no record, a workspace seen for the first time)
// makes the split again.  What the host cannot see is whether the memory itself was overwritten since.
struct SplitRecord {
    const float *a; int64_t ld, bs; int majorness, m, k, l, slices, rows_pad;
    const float *centre; int64_t centre_bs;
};

std::mutex split_records_mutex;
std::unordered_map<const void *, SplitRecord> split_records;

SplitRecord record_of(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, const WideLayout &layout)
{
    SplitRecord record;
    std::memset(&record, 0, sizeof record);          // padding too: the records are compared as bytes
    record.a = p->a; record.ld = p->a_ld; record.bs = p->a_bs; record.majorness = p->a_majorness;
    record.m = p->m; record.k = p->k; record.l = layout.a.batches; record.slices = layout.slices; record.rows_pad = layout.a.rows_pad;
    record.centre = args.centre; record.centre_bs = args.centre_bs;
    return record;
}

// true: the split of `a` in this workspace is the one this call needs; either way the record is this call's afterwards
bool split_of_a_is_kept(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, const WideLayout &layout)
{
    const SplitRecord wanted = record_of(p, args, layout);
    std::lock_guard<std::mutex> lock(split_records_mutex);
    auto found = split_records.find(p->gram_workspace);
    const bool kept = (p->flags & KMC_FLAG_GRAM_A_KEPT) && found != split_records.end() &&
                      std::memcmp(&found->second, &wanted, sizeof wanted) == 0;
    if (split_records.size() > 4096) split_records.clear();      // addresses of freed workspaces pile up otherwise
    split_records[p->gram_workspace] = wanted;
    return kept;
}

}  // namespace

// A route other than this one is about to write into `workspace`: whatever split it held is gone.
void forget_split_in(const void *workspace)
{
    std::lock_guard<std::mutex> lock(split_records_mutex);
    split_records.erase(workspace);
}

// Statistics and split of one operand (also used by the gradient's fp16 route).
hipError_t launch_gram_probe(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, unsigned *sample, int centre_pairs, int queues, hipStream_t stream);   // gram_probe.hip
kmc::GramProbeArgs gram_probe_args(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, unsigned *sample, int centre_pairs, int queues);                 // gram_probe.hip
hipError_t launch_route_centre(const float *x, int majorness, int rows, int k, int64_t ld, int64_t bs, int l, float *mean, int64_t mean_bs, hipStream_t stream);   // sample_mean.hip
int route_centre_pairs(int majorness, int rows, int k, int l);                                                                                                    // sample_mean.hip

hipError_t launch_gram_rows(const kmc::GramRowsArgs &rows_of, int batches, hipStream_t stream)
{
    const dim3 grid(rows_of.rows_pad / kmc::GW_ROW_THREADS, rows_of.ranges, batches);
    hipError_t status = launch(kmc::gram_row_stats<0>, grid, dim3(kmc::GW_ROW_THREADS), stream, rows_of);
    if (status != hipSuccess) return status;
    return launch(kmc::gram_f16_split<0>, grid, dim3(kmc::GW_ROW_THREADS), stream, rows_of);
}

// The same for both operands of a call, in two launches instead of four.
hipError_t launch_gram_rows_pair(const kmc::GramRowsArgs &first, int first_batches, const kmc::GramRowsArgs &second, int second_batches,
                                 hipStream_t stream)
{
    if (first.ranges != second.ranges) {
        hipError_t status = launch_gram_rows(first, first_batches, stream);
        return status != hipSuccess ? status : launch_gram_rows(second, second_batches, stream);
    }
    kmc::GramRowsPair pair;
    pair.first = first; pair.second = second;
    pair.first_blocks = first.rows_pad / kmc::GW_ROW_THREADS;
    pair.first_batches = first_batches; pair.second_batches = second_batches;
    const dim3 grid(pair.first_blocks + second.rows_pad / kmc::GW_ROW_THREADS, first.ranges, first_batches > second_batches ? first_batches : second_batches);
    hipError_t status = launch(kmc::gram_row_stats_pair<0>, grid, dim3(kmc::GW_ROW_THREADS), stream, pair);
    if (status != hipSuccess) return status;
    return launch(kmc::gram_f16_split_pair<0>, grid, dim3(kmc::GW_ROW_THREADS), stream, pair);
}

// The pieces of the operands that are not null and of one storage order, and in front of them the sample if there is one, in one launch.
hipError_t launch_gram_once(const kmc::GramRowsArgs *first, int first_batches, const kmc::GramRowsArgs *second, int second_batches,
                            const kmc::GramProbeArgs &probe, bool take_sample, hipStream_t stream)
{
    const bool rows = (first ? first : second)->row_major;
    const int rows_per_block = rows ? kmc::GRO_ROWS : kmc::GCO_ROWS;
    kmc::GramRowsOnceArgs args = {};
    args.probe = probe;
    args.samples = take_sample ? kmc::BK_SAMPLE_TILES : 0;
    int blocks = args.samples, k = 0, batches = 1;
    if (first) {
        args.first = *first; args.first_batches = batches = first_batches;
        args.first_blocks = first->rows_pad / rows_per_block;
        blocks += args.first_blocks;
        k = first->k;
    }
    if (second) {
        args.second = *second; args.second_batches = second_batches;
        if (second_batches > batches) batches = second_batches;
        blocks += second->rows_pad / rows_per_block;
        k = second->k;
    }
    const dim3 grid(blocks, 1, batches), threads(kmc::GW_ROW_THREADS);
    // registers for 256, 512 or 1024 k: the smallest that holds a row
    if (k > kmc::GRO_HELD_K) {
        if (!rows) return launch(kmc::gram_columns_once<16, true>, grid, threads, stream, args);
        return k <= 2 * kmc::GRO_HELD_K ? launch(kmc::gram_rows_once<32>, grid, threads, stream, args) : launch(kmc::gram_rows_once<32, true>, grid, threads, stream, args);
    }
    if (rows)
        return k <= 256 ? launch(kmc::gram_rows_once<4>, grid, threads, stream, args)
             : k <= 512 ? launch(kmc::gram_rows_once<8>, grid, threads, stream, args) : launch(kmc::gram_rows_once<16>, grid, threads, stream, args);
    return k <= 256 ? launch(kmc::gram_columns_once<4>, grid, threads, stream, args)
         : k <= 512 ? launch(kmc::gram_columns_once<8>, grid, threads, stream, args) : launch(kmc::gram_columns_once<16>, grid, threads, stream, args);
}

// Both operands, in one launch if they are stored alike; the sample in the first.
hipError_t launch_gram_once_both(const kmc::GramRowsArgs *first, int first_batches, const kmc::GramRowsArgs *second, int second_batches,
                                 const kmc::GramProbeArgs &probe, bool take_sample, hipStream_t stream)
{
    if (!first || !second || first->row_major == second->row_major)
        return launch_gram_once(first, first_batches, second, second_batches, probe, take_sample, stream);
    const hipError_t status = launch_gram_once(first, first_batches, nullptr, 0, probe, take_sample, stream);
    return status != hipSuccess ? status : launch_gram_once(nullptr, 0, second, second_batches, probe, false, stream);
}

// The product kernel in tiles of TILE; extents, batch entries and operands of `wide` are set.
template <typename Tile, bool SYMMETRIC, int EPILOGUE>
hipError_t launch_product_in(kmc::GramWideArgs &wide, hipStream_t stream)
{
    wide.wide_tiles_m = (wide.kernel.m + Tile::TILE_M - 1) / Tile::TILE_M;
    wide.wide_tiles_n = (wide.kernel.n + Tile::TILE_N - 1) / Tile::TILE_N;
    int padded = (wide.wide_tiles_n + kmc::BK_XCDS - 1) / kmc::BK_XCDS * kmc::BK_XCDS;
    if ((padded - wide.wide_tiles_n) * 8 > wide.wide_tiles_n) padded = wide.wide_tiles_n;
    // ... nor where a launch that fits the chip at once would no longer, since the padding's idle ids fall to some of the XCDs (2 x 2816 x 2816
    // of K = 4096, 22 large tiles in n, 66 of them on 64 places: 604 -> 488 us)
    const int64_t places = 32 * Tile::PER_CU, rows_of_tiles = static_cast<int64_t>(wide.wide_tiles_m) * wide.kernel.l;
    if (rows_of_tiles * (padded / kmc::BK_XCDS) > places && rows_of_tiles * wide.wide_tiles_n <= places * kmc::BK_XCDS) padded = wide.wide_tiles_n;
    wide.wide_tiles_n_padded = padded;
    const int64_t blocks = (wide.kernel.m + kmc::GW_TILE - 1) / kmc::GW_TILE;
    const int64_t width = SYMMETRIC ? blocks * (blocks + 1) / 2 * (kmc::GW_TILE / Tile::TILE_M) * (kmc::GW_TILE / Tile::TILE_N)
                                    : static_cast<int64_t>(wide.wide_tiles_m) * padded;
    if (width > 0x7fffffff) return hipErrorInvalidValue;
    // An entry of a batch on one XCD / spread over all of them, us: 64 x 300 x 300 x 4096, products, 866 / 1009; 16 x 1280 x 1280 x 4096 1010 / 1174;
    // 10 x 1100 x 1100 x 4096 637 / 733; 64 x 600 x 600 x 4096 1593 / 1993; 500 x 300 x 300 x 784 1207 / 1408; 40 sets of 900 points of K = 784
    // against themselves 224 / 251; 10 x 1500 x 100 x 8 x 4000, the gradient, 738 / 836.  Larger entries keep an XCD's L2 busy by themselves
    // and gain nothing: 20 x 2000 x 2000 (256 tiles each) 248 / 236 at K = 256, 536 / 535 at K = 784; 8 x 4096 x 4096 x 784 752 / 702.
    wide.entry_per_xcd = wide.kernel.l >= kmc::BK_XCDS &&
                         static_cast<int64_t>((wide.kernel.m + 127) / 128) * ((wide.kernel.n + 127) / 128) <= kmc_rules::WIDE_ENTRY_PER_XCD_MAX_TILES;
    return launch(kmc::gram_f16_wide<Tile, SYMMETRIC, EPILOGUE>, dim3(static_cast<unsigned>(width), wide.kernel.l, 1), dim3(Tile::THREADS), stream, wide);
}

// Tiles of 128 x 128 unless there are many: three of them share a CU and share the chip out more evenly, tiles of 256 x 128 ask
// the L2 for three quarters of the bytes per multiply-add.  Time of a call in the small tiles over the large ones: 32 large
// tiles 0.94 at K = 128, 0.75 at K = 2048; 288 tiles 0.92, 0.90; 512 tiles 0.99, 1.03; 800 tiles 0.97, 0.96; 1128 tiles
// 0.89, 0.97; 2048 tiles 0.96, 1.03; 3160 tiles 0.91, 1.00; 8192 tiles 1.02 at K = 128, 1.01 at K = 512.
//
// Above one round of small tiles (three on each of 256 CUs) the few of the second round have the chip to themselves; where the large
// tiles are one round (two per CU) they are taken instead, as long as the second round of small ones is little or the contraction long.
// Not for a set against itself, whose rounds are of unequal tiles.  Small / large, us, k contiguous: 800 small tiles, 8 x 1280 x 1280 of
// K = 784 129.4 / 127.5, of K = 4096 644 / 617; 840, 28 x 640 x 768 of
// K = 784 210 / 185, of K = 4096 1072 / 934; 784, 3584 x 3584 of K = 784 100 / 96, of K = 4096 395 / 371; 938, 200 x 60000 of K = 784 194.4 / 197.5,
// of K = 2048 568 / 561; 1024, 4096 x 4096 of K = 784 103.1 / 103.8, of K = 4096 432 / 421; more than one round of either: 1156,
// 4352 x 4352 of K = 2048 276 / 306.  A set against itself: 780, 4900 points of K = 784 110 / 120; 990, 5632 of K = 784 130 / 127.
//
// A contraction stays with the small tiles: the large one's sums and products leave no registers for its operands, and it has no stores to save on
// (large / small, us: 4 x 16384 x 16384 x 256, 32 columns 3073 / 2967, 10 columns 2477 / 2407; 30000 x 30000 x 1024, 16 columns 5012 / 5054, 32
// columns 5418 / 5406; 16384 x 16384 x 128, 32 columns 622 / 613).
constexpr int64_t SMALL_TILES_PER_ROUND = kmc::WideTileSmall::PER_CU * 256, LARGE_TILES_PER_ROUND = kmc::WideTileLarge::PER_CU * 256;
constexpr int64_t LITTLE_OF_A_ROUND = SMALL_TILES_PER_ROUND / 6;
constexpr int LONG_CONTRACTION_SLICES = 2048 / kmc::BK_TILE_K;
// Two small tiles per CU: up to there a tile by 8 waves, beyond it three by 4 each.  By 4 / 8 waves, us of a call, k contiguous: 192 tiles,
// 3000 x 1000 x 784 49.4 / 45.8; 256, 2000 x 2000 of K = 784 51.5 / 48.9, of K = 3072 152.6 / 149.2; 324, 2200 x 2200 x 784 63.5 / 63.1; 484,
// 2700 x 2700 x 784 77.7 / 71.5, products 2800 x 2800 of K = 256 31.9 / 29.3, of K = 4096 272 / 228; 480, 20 x 500 x 700 x 784 102.2 / 102.5; beyond:
// 529, 2880 x 2880 x 784 78.6 / 81.2; 676, 3300 x 3300 x 784 88.1 / 93.1.  A set against itself: 128, 2000 points of K = 784 63.0 / 52.5; 288,
// 3000 of K = 512 67.1 / 61.1; 392, 3500 of K = 784 79.0 / 73.2; 480, 3900 of K = 784 93.5 / 92.7; 544, 4200 102.0 / 99.6.
constexpr int64_t FEW_TILES = 2 * 256;

template <bool SYMMETRIC, int EPILOGUE>
hipError_t launch_product(kmc::GramWideArgs &wide, hipStream_t stream)
{
    using Large = kmc::WideTileLarge;
    using Small = kmc::WideTileSmall;
    auto tiles_of = [&](int tile_m, int tile_n) {
        return static_cast<int64_t>((wide.kernel.m + tile_m - 1) / tile_m) * ((wide.kernel.n + tile_n - 1) / tile_n) * wide.kernel.l / (SYMMETRIC ? 2 : 1);
    };
    const int64_t large = tiles_of(Large::TILE_M, Large::TILE_N), small = tiles_of(Small::TILE_M, Small::TILE_N);
    const bool one_round = !SYMMETRIC && small > SMALL_TILES_PER_ROUND && large <= LARGE_TILES_PER_ROUND &&
                           (small <= SMALL_TILES_PER_ROUND + LITTLE_OF_A_ROUND || wide.slices >= LONG_CONTRACTION_SLICES);
    // KERMAC_AMD_WIDE_LARGE_TILE_MIN_TILES=n replaces the number (read on every call, so that a test can send small shapes to the large tiles)
    const char *text = std::getenv("KERMAC_AMD_WIDE_LARGE_TILE_MIN_TILES");
    if constexpr (EPILOGUE < kmc::GW_CONTRACT_16) {
        if (large >= (text ? std::atoi(text) : kmc_rules::WIDE_LARGE_TILE_MIN_TILES) || one_round) return launch_product_in<Large, SYMMETRIC, EPILOGUE>(wide, stream);
    } else if (text && std::atoi(text) > 0) {
        return launch_product_in<Small, SYMMETRIC, EPILOGUE>(wide, stream);
    }
    if (small <= FEW_TILES) return launch_product_in<kmc::WideTileFew, SYMMETRIC, EPILOGUE>(wide, stream);
    return launch_product_in<Small, SYMMETRIC, EPILOGUE>(wide, stream);
}

// Room for the products of a contraction's tiles, behind everything else; false where the kernels behind it could not take the problem.
bool place_contraction(const kmc::BuildKernelArgs &args, int outputs, WideLayout *layout)
{
    if (outputs < 1 || outputs > CONTRACTION_MAX_OUTPUTS || args.tiles_n > 65535) return false;
    int64_t cursor = layout->bytes;
    layout->products = place(cursor, static_cast<int64_t>(args.tiles_n) * args.l * args.m * ((outputs + 3) / 4 * 4) * 4);
    layout->stamps = place(cursor, static_cast<int64_t>(args.l) * args.tiles_m * args.tiles_n * 4);
    layout->bytes = cursor;
    return true;
}

// Bytes of workspace for the matrix times coefficients by this path; 0 when it does not apply.
int64_t gram_f16_wide_contraction_bytes(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args, int outputs)
{
    WideLayout layout;
    return wide_layout(p, args, &layout) && place_contraction(args, outputs, &layout) ? layout.bytes : 0;
}

// Bytes of workspace the path needs for this problem; 0 when it does not apply.
int64_t gram_f16_wide_bytes(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &args)
{
    WideLayout layout;
    return wide_layout(p, args, &layout) ? layout.bytes : 0;
}

// Row statistics and split of both operands, then the product kernel.  `*taken` says whether the
// path applied (and the launches were made); if not, nothing was launched.
hipError_t launch_gram_f16_wide(const kmc_build_kernel_params *p, const kmc::BuildKernelArgs &as_given, hipStream_t stream, bool *taken,
                                const unsigned **sample_taken, Contraction *contraction)
{
    kmc::BuildKernelArgs args = as_given;
    *taken = false;
    if (sample_taken) *sample_taken = nullptr;
    WideLayout layout;
    if (!p->gram_workspace || !wide_layout(p, args, &layout) || (contraction && !place_contraction(args, contraction->outputs, &layout)) || p->gram_workspace_bytes < layout.bytes ||
        (reinterpret_cast<uintptr_t>(p->gram_workspace) & (REGION_ALIGN - 1)) != 0)
        return hipSuccess;
    char *workspace = static_cast<char *>(p->gram_workspace);
    const bool scalar_only = (p->flags & KMC_FLAG_FORCE_SCALAR_ACCESS) != 0;
    const bool own_centre = layout.centre_floats != 0;
    if (own_centre) {
        args.centre = reinterpret_cast<float *>(workspace + layout.centre);
        args.centre_bs = layout.centre_batches > 1 ? layout.centre_floats : 0;
    }
    const int centre_pairs = own_centre ? route_centre_pairs(p->a_majorness, args.m, args.k, layout.centre_batches) : 0;
    const kmc::GramRowsArgs rows_a = rows_args(args.a, args.a_ld, args.a_bs, args.m, p->a_majorness, scalar_only, args, layout, layout.a, workspace, centre_pairs);
    const kmc::GramRowsArgs rows_b = rows_args(args.b, args.b_ld, args.b_bs, args.n, p->b_majorness, scalar_only, args, layout, layout.b, workspace, centre_pairs);
    // The caller's trust rule grows with sqrt(k) (the error of a sum of k terms against the norms) and
    // passes 1 near k = 18000, where it would send every part to the repair launch -- whose own
    // fp32 sum over k is no better by then (measured at k = 20000 .. 200000: products of pieces, rounded once
    // per 16 k, 4e-7 .. 2e-6 of d for points as far apart as their norms, the direct kernel 5e-6 .. 4e-5; the present walk, once per
    // 32 k, as that one: largest error 5.7e-7 at k = 20000, 9.3e-7 at k = 60000).
    // With a product worth half the norms the two are equally good, so that is where the rule stops.
    kmc::GramWideArgs wide = {};
    wide.kernel = args;
    if (wide.kernel.gram_trust > 0.5f) wide.kernel.gram_trust = 0.5f;
    const bool products = p->inner_operator == KMC_OP_DOT;
    // Squared differences: a sample of the result first, so that data the trust rule would reject wholesale
    // (sets of near-duplicates) costs the direct kernel's time and little more, instead of both.
    // KMC_FLAG_NO_PROBE leaves it out.
    unsigned *sample = !products && !(p->flags & KMC_FLAG_NO_PROBE) ? reinterpret_cast<unsigned *>(workspace + layout.sample) : nullptr;
    // the region of a lies first in the workspace and its size does not depend on b
    const bool a_is_kept = split_of_a_is_kept(p, args, layout);
    const bool split_a = !a_is_kept, split_b = !args.symmetric;
    bool sampled = false;
    hipError_t status = hipSuccess;
    // (a kept split of a was made around the centre that is still there)
    if (own_centre && split_a)
        status = launch_route_centre(args.a, p->a_majorness, args.m, args.k, args.a_ld, args.a_bs, layout.centre_batches,
                                     reinterpret_cast<float *>(workspace + layout.centre), layout.centre_floats, stream);
    if (status != hipSuccess) return status;
    if ((split_a && layout.a.once) || (split_b && layout.b.once)) {
        status = launch_gram_once_both(split_a && layout.a.once ? &rows_a : nullptr, layout.a.batches, split_b && layout.b.once ? &rows_b : nullptr,
                                       layout.b.batches, sample ? gram_probe_args(p, wide.kernel, sample, centre_pairs, kmc::BK_REPAIR_WORDS) : kmc::GramProbeArgs{}, sample != nullptr, stream);
        sampled = true;
    }
    if (status == hipSuccess && split_a && split_b && !layout.a.once && !layout.b.once) {
        status = launch_gram_rows_pair(rows_a, layout.a.batches, rows_b, layout.b.batches, stream);
    } else {
        if (status == hipSuccess && split_a && !layout.a.once) status = launch_gram_rows(rows_a, layout.a.batches, stream);
        if (status == hipSuccess && split_b && !layout.b.once) status = launch_gram_rows(rows_b, layout.b.batches, stream);
    }
    if (status == hipSuccess && sample && !sampled) status = launch_gram_probe(p, wide.kernel, sample, centre_pairs, kmc::BK_REPAIR_WORDS, stream);
    if (status != hipSuccess) return status;
    if (sample) {
        wide.kernel.sample = sample;
        if (sample_taken) *sample_taken = sample;
    }

    wide.pieces_a = rows_a.pieces; wide.pieces_b = rows_b.pieces;
    wide.pieces_a_bs = layout.a.batches > 1 ? layout.a.pieces_bs : 0;
    wide.pieces_b_bs = layout.b.batches > 1 ? layout.b.pieces_bs : 0;
    wide.squares_a = rows_a.squares; wide.squares_b = rows_b.squares;
    wide.stats_a_bs = layout.a.batches > 1 ? layout.a.stats_bs : 0;
    wide.stats_b_bs = layout.b.batches > 1 ? layout.b.stats_bs : 0;
    wide.unscale_a = rows_a.unscale; wide.unscale_b = rows_b.unscale;
    wide.unscale_a_bs = layout.a.batches > 1 ? layout.a.rows_pad : 0;
    wide.unscale_b_bs = layout.b.batches > 1 ? layout.b.rows_pad : 0;
    wide.rows_pad_a = layout.a.rows_pad; wide.rows_pad_b = layout.b.rows_pad;
    wide.slices = layout.slices; wide.ranges_a = layout.a.ranges; wide.ranges_b = layout.b.ranges;
    if (contraction) {
        wide.coef = contraction->coef; wide.coef_ld = contraction->coef_ld; wide.coef_bs = contraction->coef_bs;
        wide.outputs = contraction->outputs;
        wide.products = contraction->products = reinterpret_cast<float *>(workspace + layout.products);
        wide.products_ld = (contraction->outputs + 3) / 4 * 4;
        wide.products_bs = wide.products_ld * args.m;
        wide.products_tile = wide.products_bs * args.l;
        wide.stamps = contraction->stamps = reinterpret_cast<int *>(workspace + layout.stamps);
        wide.stamps_m = args.tiles_m; wide.stamps_n = args.tiles_n;
        const bool few = contraction->outputs <= 16;
        if (products)
            status = few ? launch_product<false, kmc::GW_EPILOGUE_DOT + kmc::GW_CONTRACT_16>(wide, stream) : launch_product<false, kmc::GW_EPILOGUE_DOT + kmc::GW_CONTRACT_32>(wide, stream);
        else
            status = few ? launch_product<false, kmc::GW_EPILOGUE_DISTANCE + kmc::GW_CONTRACT_16>(wide, stream) : launch_product<false, kmc::GW_EPILOGUE_DISTANCE + kmc::GW_CONTRACT_32>(wide, stream);
        if (status == hipSuccess) *taken = true;
        return status;
    }
    if (args.symmetric)
        status = products ? launch_product<true, kmc::GW_EPILOGUE_DOT>(wide, stream) : launch_product<true, kmc::GW_EPILOGUE_DISTANCE>(wide, stream);
    else
        status = products ? launch_product<false, kmc::GW_EPILOGUE_DOT>(wide, stream) : launch_product<false, kmc::GW_EPILOGUE_DISTANCE>(wide, stream);
    if (status == hipSuccess) *taken = true;
    return status;
}

// ---- the gradient of the L2 norm as one product of pieces (norm_gradient_l2_wide.hpp) ----

bool matrix_coefficients_by_rows4(const kmc_matrix_coefficients_params *p);                            // matrix_times_coefficients.hip
int matrix_times_coefficients(const kmc_matrix_coefficients_params *p, float *magnitudes, int64_t magnitudes_bs, int64_t magnitudes_split_stride,
                              hipStream_t stream);                                                   // matrix_times_coefficients.hip

namespace {

struct GradientL2Layout {
    WideLayout wide;                 // a: the columns m of a; b: the rows (o, n) of the products
    int g_parts;                     // ranges of k that g is summed in (partial products, then their sum)
    int64_t shift, c_transposed, g, g_partial, magnitudes;      // byte offsets behind the regions of `wide`
    int64_t bytes;
};

// The route pays where a model of both times says so by 15 %, in microseconds, fitted to sweeps with the kernels of the route before the present
// ones (which make the pieces of the products straight from b and c and walk faster, so the rule leaves a few calls to the fp32 kernels
// that the route would win, and takes none that it loses):
//   fp32 kernels   30 + terms * t(o) with terms = m n k l and t(o) = 0.077, 0.10, 0.126, 0.137 ps for 1 .. 4
//                  outputs, 0.028 o up to 8 (vector kernels), 0.27 up to 16, 0.56 up to 32, 0.0175 o beyond
//                  (matrix-core kernels: a run of outputs costs what its 16 or 32 columns cost);
//   this route     200 + 1.5e-6 (o n + m) k l for the products in fp32 and the two splits, and for the walk
//                  6.3e-9 per multiply-add of the padded tiles but not less than 0.056 k (1.7 us per 256 x 256 x 16 step of a CU
//                  with the chip full, 0.9 us alone; the present kernel takes 4.7e-9 with the chip full).
// Examples (fp32 / this route, measured with the present kernel): 8192 x 512 x 16 x 8192 3.0; o = 1 4.3, o = 32 3.2; n = 64 1.65;
// m = 1024 1.6; k = 512 1.8, k = 256 1.2; 10000 x 1000 x 10 x 784 3.4.  Calls below stay on the fp32 kernels, which
// are more exact where the rows of a and c have opposite scales (cdist_grad.py).  KERMAC_AMD_GRADIENT_L2_MIN_TERMS replaces the rule by a number of terms
// (read on every call, so that a test can send small shapes down the route).
bool gradient_l2_pays(const kmc_norm_gradient_params *p, int64_t tiles_m, int64_t tiles_n)
{
    const char *text = std::getenv("KERMAC_AMD_GRADIENT_L2_MIN_TERMS");
    const double forced = text ? std::atof(text) : 0.0;
    const double terms = static_cast<double>(p->m) * p->n * p->k * p->l;
    if (forced > 0.0) return terms >= forced;
    if (p->flags & KMC_FLAG_GRAM_WORKSPACE_ANY_SIZE) return true;
    const int o = p->o;
    const double per_term = o == 1 ? 0.077 : o == 2 ? 0.10 : o == 3 ? 0.126 : o == 4 ? 0.137 : o <= 8 ? 0.028 * o
                          : o <= 16 ? 0.27 : o <= 32 ? 0.56 : 0.0175 * o;
    const double fp32_us = 30.0 + terms * per_term * 1e-6;
    const double padded = static_cast<double>(tiles_m) * tiles_n * kmc::GW_TILE * kmc::GW_TILE * p->k * p->l;
    const double walk_us = padded * 6.3e-9 > 0.056 * p->k ? padded * 6.3e-9 : 0.056 * p->k;
    const double route_us = 200.0 + 1.5e-6 * (static_cast<double>(o) * p->n + p->m) * p->k * p->l + walk_us;
    return (100 + kmc_rules::GRADIENT_L2_ADVANTAGE_PERCENT) * route_us < 100 * fp32_us;
}

bool gradient_l2_layout(const kmc_norm_gradient_params *p, GradientL2Layout *layout)
{
    if (p->norm_type != KMC_NORM_L2 || p->m < 1 || p->n < 1 || p->o < 1 || p->k < 1 || p->l < 1) return false;
    // row r = o * n_rows + n of the product is row n of plane o of e
    if (p->o > 1 && p->e_ld_o != static_cast<int64_t>(p->n) * p->e_ld_n) return false;
    const int64_t rows = static_cast<int64_t>(p->o) * p->n;
    if (rows > 0x7fffffff - kmc::GW_TILE || (p->o + kmc::GL2_OUTPUTS - 1) / kmc::GL2_OUTPUTS > 65535) return false;
    WideLayout &wide = layout->wide;
    wide.tiles_m = (p->m + kmc::GW_TILE - 1) / kmc::GW_TILE;
    wide.tiles_n = static_cast<int>((rows + kmc::GW_TILE - 1) / kmc::GW_TILE);
    if (!gradient_l2_pays(p, wide.tiles_m, wide.tiles_n)) return false;
    if (!place_wide(p->m, static_cast<int>(rows), p->k, p->l, p->a_bs == 0, false, false, false, false, 0, &wide)) return false;
    int64_t cursor = wide.bytes;
    layout->shift = place(cursor, static_cast<int64_t>(p->l) * p->n * 4);
    layout->c_transposed = place(cursor, static_cast<int64_t>(p->l) * p->k * p->o * 4);
    layout->g = place(cursor, static_cast<int64_t>(p->l) * p->m * p->o * 4);
    // kmc_matrix_times_coefficients wants a workgroup per CU: 256 columns m and 32 outputs each (of 128: 287 us where these take 269)
    const int64_t workgroups = static_cast<int64_t>((p->m + 255) / 256) * ((p->o + 31) / 32) * p->l;
    int parts = workgroups >= 256 ? 1 : static_cast<int>((256 + workgroups - 1) / workgroups);
    if (parts > p->k / 512) parts = p->k / 512 > 1 ? p->k / 512 : 1;
    if (static_cast<int64_t>(parts) * p->l > 65535) parts = 1;
    layout->g_parts = parts;
    layout->g_partial = parts > 1 ? place(cursor, static_cast<int64_t>(parts) * p->l * p->m * p->o * 4) : 0;
    layout->magnitudes = place(cursor, static_cast<int64_t>(parts) * wide.a.batches * wide.a.rows_pad * 4);
    layout->bytes = cursor;
    return true;
}

}  // namespace

int64_t norm_gradient_l2_wide_bytes(const kmc_norm_gradient_params *p)
{
    GradientL2Layout layout;
    return gradient_l2_layout(p, &layout) ? layout.bytes : 0;
}

// `*taken` says whether the route applied (and the launches were made); if not, nothing was launched.
int launch_norm_gradient_l2_wide(const kmc_norm_gradient_params *p, hipStream_t stream, bool *taken)
{
    *taken = false;
    GradientL2Layout layout;
    if (!p->workspace || !gradient_l2_layout(p, &layout) || p->workspace_bytes < layout.bytes ||
        (reinterpret_cast<uintptr_t>(p->workspace) & (REGION_ALIGN - 1)) != 0)
        return KMC_OK;
    char *workspace = static_cast<char *>(p->workspace);
    const WideLayout &wide = layout.wide;
    const int rows = p->o * p->n;
    const bool scalar_only = (p->flags & KMC_FLAG_FORCE_SCALAR_ACCESS) != 0;

    kmc::GradientL2PrepareArgs prepare = {};
    prepare.b = p->b; prepare.b_ld = p->b_ld; prepare.b_bs = p->b_bs;
    prepare.c = p->c; prepare.c_ld = p->c_ld; prepare.c_bs = p->c_bs;
    prepare.shift = reinterpret_cast<float *>(workspace + layout.shift); prepare.shift_bs = p->n;
    prepare.c_transposed = reinterpret_cast<float *>(workspace + layout.c_transposed);
    prepare.c_transposed_ld = p->o; prepare.c_transposed_bs = static_cast<int64_t>(p->k) * p->o;
    prepare.n = p->n; prepare.o = p->o; prepare.k = p->k;
    hipError_t status = launch(kmc::gradient_l2_prepare, dim3(p->n + (p->k + kmc::GL2_THREADS - 1) / kmc::GL2_THREADS, p->l), dim3(kmc::GL2_THREADS), stream, prepare);
    if (status != hipSuccess) return fail_hip(status, "gradient_l2_prepare launch");

    // g[m][o] = sum_k a[k][m] c[o][k]: a is a stored panel with m contiguous
    float *g = reinterpret_cast<float *>(workspace + layout.g);
    kmc_matrix_coefficients_params weights = {};
    weights.m = p->m; weights.n = p->k; weights.o = p->o; weights.l = p->l;
    weights.matrix = p->a; weights.matrix_ld = p->a_ld; weights.matrix_bs = p->a_bs;
    weights.coef = prepare.c_transposed; weights.coef_ld = prepare.c_transposed_ld; weights.coef_bs = prepare.c_transposed_bs;
    weights.out = g; weights.out_ld = p->o; weights.out_bs = static_cast<int64_t>(p->m) * p->o;
    if (layout.g_parts > 1) {
        weights.out = reinterpret_cast<float *>(workspace + layout.g_partial);
        weights.n_splits = layout.g_parts;
        weights.out_split_stride = static_cast<int64_t>(p->l) * weights.out_bs;
    }
    // the largest magnitudes of a's columns come with it (of a broadcast a from every batch entry, the same words)
    const bool with_magnitudes = matrix_coefficients_by_rows4(&weights);
    float *magnitudes = reinterpret_cast<float *>(workspace + layout.magnitudes);
    const int64_t magnitudes_bs = static_cast<int64_t>(layout.g_parts) * wide.a.rows_pad;
    const int contracted = matrix_times_coefficients(&weights, with_magnitudes ? magnitudes : nullptr, wide.a.batches > 1 ? magnitudes_bs : 0, wide.a.rows_pad, stream);
    if (contracted != KMC_OK) return contracted;
    if (layout.g_parts > 1) {
        kmc::GradientL2SumArgs sum = {};
        sum.partial = weights.out; sum.sum = g;
        sum.count = static_cast<int64_t>(p->l) * weights.out_bs; sum.stride = weights.out_split_stride;
        sum.parts = layout.g_parts;
        status = launch(kmc::gradient_l2_sum_parts, dim3(static_cast<unsigned>((sum.count + kmc::GL2_THREADS - 1) / kmc::GL2_THREADS)),
                        dim3(kmc::GL2_THREADS), stream, sum);
        if (status != hipSuccess) return fail_hip(status, "gradient_l2_sum_parts launch");
    }

    // no centre: the shift of b is in the products already
    kmc::BuildKernelArgs walk = {};
    walk.m = p->m; walk.n = rows; walk.k = p->k; walk.l = p->l;
    const kmc::GramRowsArgs rows_a = rows_args(p->a, p->a_ld, p->a_bs, p->m, KMC_COL_MAJOR, scalar_only, walk, wide, wide.a, workspace);
    const kmc::GramRowsArgs rows_b = rows_args(nullptr, 0, 0, rows, KMC_ROW_MAJOR, scalar_only, walk, wide, wide.b, workspace);
    kmc::GradientL2PiecesArgs pieces = {};
    pieces.a = rows_a; pieces.p = rows_b;
    // the columns that pad a hold zeros whatever their scale, of which the workspace may hold any
    pieces.a_blocks = with_magnitudes ? 0 : rows_a.rows_pad / kmc::GW_ROW_THREADS; pieces.a_batches = wide.a.batches;
    pieces.from = prepare;
    // four outputs share a read of b, unless that leaves p fewer workgroups than three per CU
    const int ranges = rows_a.ranges > rows_b.ranges ? rows_a.ranges : rows_b.ranges, blocks_n = (p->n + kmc::GL2_ROWS - 1) / kmc::GL2_ROWS;
    pieces.outputs = kmc::GL2_OUTPUTS;
    while (pieces.outputs > 1 && static_cast<int64_t>(blocks_n) * ((p->o + pieces.outputs - 1) / pieces.outputs) * ranges * p->l < 768) pieces.outputs /= 2;
    dim3 grid(pieces.a_blocks + blocks_n * ((p->o + pieces.outputs - 1) / pieces.outputs), ranges, p->l);
    static_assert(kmc::GW_ROW_THREADS == kmc::GL2_THREADS, "one launch for both operands");
    status = launch(kmc::gradient_l2_pieces_stats, grid, dim3(kmc::GL2_THREADS), stream, pieces);
    if (with_magnitudes) {
        pieces.a.magnitudes = magnitudes;
        pieces.a.stats_bs = magnitudes_bs;
        pieces.a.magnitude_ranges = layout.g_parts;
        pieces.a_blocks = rows_a.rows_pad / kmc::GW_ROW_THREADS;
        grid.x += pieces.a_blocks;
    }
    if (status == hipSuccess) status = launch(kmc::gradient_l2_pieces_split, grid, dim3(kmc::GL2_THREADS), stream, pieces);
    if (status != hipSuccess) return fail_hip(status, "gradient_l2_pieces launches");

    kmc::GramWideArgs product = {};
    product.kernel = walk;
    product.kernel.c = p->e; product.kernel.c_ld = p->e_ld_n; product.kernel.c_bs = p->e_bs;
    product.kernel.c_vec = !scalar_only && aligned16(p->e) && p->e_ld_n % 4 == 0 && p->e_bs % 4 == 0;
    product.pieces_a = rows_a.pieces; product.pieces_b = rows_b.pieces;
    product.pieces_a_bs = wide.a.batches > 1 ? wide.a.pieces_bs : 0;
    product.pieces_b_bs = wide.b.batches > 1 ? wide.b.pieces_bs : 0;
    product.squares_a = rows_a.squares; product.squares_b = rows_b.squares;
    product.stats_a_bs = wide.a.batches > 1 ? wide.a.stats_bs : 0;
    product.stats_b_bs = wide.b.batches > 1 ? wide.b.stats_bs : 0;
    product.unscale_a = rows_a.unscale; product.unscale_b = rows_b.unscale;
    product.unscale_a_bs = wide.a.batches > 1 ? wide.a.rows_pad : 0;
    product.unscale_b_bs = wide.b.batches > 1 ? wide.b.rows_pad : 0;
    product.rows_pad_a = wide.a.rows_pad; product.rows_pad_b = wide.b.rows_pad;
    product.slices = wide.slices; product.ranges_a = wide.a.ranges; product.ranges_b = wide.b.ranges;
    product.gradient_d = p->d; product.gradient_d_ld = p->d_ld; product.gradient_d_bs = p->d_bs;
    product.gradient_g = g; product.gradient_g_ld = p->o; product.gradient_g_bs = weights.out_bs;
    product.gradient_shift = prepare.shift; product.gradient_shift_bs = prepare.shift_bs;
    product.gradient_n = p->n;
    status = launch_product<false, kmc::GW_EPILOGUE_GRADIENT_L2>(product, stream);
    if (status != hipSuccess) return fail_hip(status, "gram_f16_wide (gradient) launch");
    *taken = true;
    return KMC_OK;
}

}  // namespace kmc_host
