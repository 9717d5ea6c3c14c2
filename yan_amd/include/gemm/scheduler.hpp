// Workgroup -> output-tile mapping for a 256-CU, 8-XCD part.
// Replaces the reference's persistent tile Scheduler (yan/include/gemm/scheduler.cuh:15-58: block count
// ceil(m/BLOCK_M)*ceil(N/BLOCK_N), grouped swizzle of 16 blocks for L2 reuse). The mapping is the same for all
// three GemmTypes; what a group changes (operand bases, valid rows) is applied by the kernel on top of the tile.
#pragma once

#include "utils.hpp"

namespace yan {

enum class GemmType { Normal, GroupedContiguous, GroupedMasked };

struct TileCoord {
    int  m_idx;
    int  n_idx;
    bool valid;
};

// The hardware hands consecutive workgroup ids to the 8 XCDs round-robin, and each XCD has a private L2.
// Workgroup `bid` therefore runs on XCD `bid % 8`, and the 32 tiles an XCD has in flight should form a compact
// GROUP_M x 4 patch whose A and B panels are shared through that L2. Two arrangements do that; both have the same
// number of slots and give every XCD the same number of tiles.
//
// Band order (the default): every XCD gets one contiguous range of a tile sequence that walks bands of GROUP_M
// tile-rows column by column.
//
// Region order (chosen when the operands together do not fit the 256 MB memory-side cache; the caller passes
// `row_bytes`, the bytes of one operand row = K * element size): the 8 patches that run at the
// same time form one region of R x (256 / R) tiles, R = 16, 32, 8 or 64, and the regions are walked along one dimension
// first, so that the panels of the other dimension stay in the cache while those of the first stream through. Band
// order keeps up to 8 x 8 + 4 x 8 different panels in flight chip-wide and re-reads a whole operand from HBM for every
// round once they outgrow the cache; here the region shape and the direction are the ones a small traffic model rates
// cheapest (ties go to the squarer region). Measured on bf16 with 256 x 256 tiles: 12288^3 3067 -> 2737 us,
// 8192 x 4096 x 14336 735 -> 683, 16384^2 x 8192 3195 -> 2995; no change where the model picks what band order amounts
// to (8192^2 x 12288). FP8: 16384^3 3627 -> 3506 us.
template <int GROUP_M = 8>
struct XcdTileScheduler {
    static constexpr int PATCH_COLS = 4, PATCH = GROUP_M * PATCH_COLS, ROUND = PATCH * kNumXCD;
    static constexpr long long kCacheBytes = 256ll << 20;

    int  tiles_m, tiles_n, total, per_xcd;
    int  band_height;                     // tile-rows of a band: GROUP_M, or fewer when the caller's groups hold fewer (below)
    int  region_rows, region_cols;        // 0: band order
    bool rows_outer;                      // region order: all column blocks of a row block before the next row block

    __host__ __device__ XcdTileScheduler(int m, int n, int block_m, int block_n, long long row_bytes = 0) {
        tiles_m = ceil_div(m, block_m);
        tiles_n = ceil_div(n, block_n);
        total   = tiles_m * tiles_n;
        per_xcd = ceil_div(total, kNumXCD);
        band_height = GROUP_M;
        region_rows = region_cols = 0;
        rows_outer = true;
        const long long panel_a = row_bytes * block_m, panel_b = row_bytes * block_n;
        const long long all_a = panel_a * tiles_m, all_b = panel_b * tiles_n;
        if (row_bytes <= 0 || total < ROUND || all_a + all_b <= kCacheBytes) return;
        long long best = -1;
        static_assert(GROUP_M == 8 && ROUND == 256);
        const int candidates[4] = {16, 32, 8, 64};          // region rows; ties go to the earlier (squarer) one
        for (int i = 0; i < 4; ++i) {
            const int r = candidates[i], c = ROUND / r;
            if (r > ceil_div(tiles_m, GROUP_M) * GROUP_M || c > ceil_div(tiles_n, PATCH_COLS) * PATCH_COLS) continue;
            const int re = r < tiles_m ? r : tiles_m, ce = c < tiles_n ? c : tiles_n;
            const int row_blocks = ceil_div(tiles_m, r), col_blocks = ceil_div(tiles_n, c);
            const bool block_fits = re * panel_a + ce * panel_b <= kCacheBytes;
            // rows outer: the A block stays while the column blocks pass; B is read once per row block unless all of it stays
            const long long a_outer = (block_fits ? all_a : all_a * col_blocks) +
                                      ((col_blocks == 1 && all_b + re * panel_a <= kCacheBytes) ? all_b : all_b * row_blocks);
            const long long b_outer = (block_fits ? all_b : all_b * row_blocks) +
                                      ((row_blocks == 1 && all_a + ce * panel_b <= kCacheBytes) ? all_a : all_a * col_blocks);
            if (best < 0 || a_outer < best) { best = a_outer; region_rows = r; region_cols = c; rows_outer = true; }
            if (b_outer < best)             { best = b_outer; region_rows = r; region_cols = c; rows_outer = false; }
        }
    }

    __host__ __device__ int grid_size() const { return per_xcd * kNumXCD; }

    __host__ __device__ TileCoord tile_of(int bid) const {
        if (region_rows) return region_tile_of(bid);
        const int t = (bid % kNumXCD) * per_xcd + bid / kNumXCD;
        if (t >= total) return {0, 0, false};
        return band_tile(t);
    }

    // Grouped layouts: the rows are `groups` stacked problems with their own weights. Bands no taller than a group keep the
    // 32 consecutive tiles an XCD runs at once inside one group where groups are aligned: h x (32 / h) tiles share h
    // activation panels and 32 / h weight panels of one group, instead of 8 and 4 per group touched (4 groups of 4 tile-rows:
    // 12 panels instead of 16).
    __host__ __device__ void fit_bands_to_groups(int tile_rows_per_group) {
        band_height = tile_rows_per_group < 1 ? 1 : (tile_rows_per_group < GROUP_M ? tile_rows_per_group : GROUP_M);
    }

    // Tile number t of the band-order sequence.
    __host__ __device__ TileCoord band_tile(int t) const {
        const int band      = band_height * tiles_n;
        const int first_m   = (t / band) * band_height;
        const int band_rows = (tiles_m - first_m) < band_height ? (tiles_m - first_m) : band_height;
        const int in_band   = t % band;
        return {first_m + in_band % band_rows, in_band / band_rows, true};
    }

    // Slot -> position in a tile sequence, dealt out in rounds: full rounds of 256 tiles hand XCD x the x-th run of 32
    // consecutive tiles; the tiles left after the full rounds are dealt out in 8 equal runs. -1: an empty slot.
    __host__ __device__ int dealt_position(int bid) const {
        const int x = bid % kNumXCD, q = bid / kNumXCD;
        const int full = total / ROUND, rest = total - full * ROUND;
        if (q < full * PATCH) return ((q / PATCH) * kNumXCD + x) * PATCH + q % PATCH;
        const int run = ceil_div(rest, kNumXCD), q_rest = q - full * PATCH;
        const int t = full * ROUND + x * run + q_rest;
        return (q_rest >= run || t >= total) ? -1 : t;
    }

    // Band order dealt out in rounds: an XCD's 32 concurrent tiles are still a patch of one band, but consecutive patches
    // go to different XCDs. For grids whose tiles differ in cost by position (the masked layout: a group may have few rows
    // or none), where a contiguous range per XCD would leave some XCDs with all the work.
    __host__ __device__ TileCoord dealt_band_tile_of(int bid) const {
        const int t = dealt_position(bid);
        if (t < 0) return {0, 0, false};
        return band_tile(t);
    }

    // Region order, dealt out in rounds (a run of 32 consecutive tiles is one patch when the region is whole). The sequence: region
    // by region; inside a region patch rows of GROUP_M, inside a patch row patches of 4 columns, inside a patch column by
    // column. Regions, patch rows and patches at the lower and right edges are smaller, which shifts the runs against
    // the patches but loses no tile.
    __host__ __device__ TileCoord region_tile_of(int bid) const {
        const int t = dealt_position(bid);
        if (t < 0) return {0, 0, false};
        int rb, cb, hh, ww, p;        // region (rb, cb) of hh x ww tiles, position p inside it
        if (rows_outer) {
            rb = t / (region_rows * tiles_n);
            hh = (tiles_m - rb * region_rows) < region_rows ? (tiles_m - rb * region_rows) : region_rows;
            const int in_block = t - rb * region_rows * tiles_n;
            cb = in_block / (hh * region_cols);
            ww = (tiles_n - cb * region_cols) < region_cols ? (tiles_n - cb * region_cols) : region_cols;
            p  = in_block - cb * hh * region_cols;
        } else {
            cb = t / (region_cols * tiles_m);
            ww = (tiles_n - cb * region_cols) < region_cols ? (tiles_n - cb * region_cols) : region_cols;
            const int in_block = t - cb * region_cols * tiles_m;
            rb = in_block / (ww * region_rows);
            hh = (tiles_m - rb * region_rows) < region_rows ? (tiles_m - rb * region_rows) : region_rows;
            p  = in_block - rb * ww * region_rows;
        }
        const int pr = p / (GROUP_M * ww);                                       // patch row
        const int ph = (hh - pr * GROUP_M) < GROUP_M ? (hh - pr * GROUP_M) : GROUP_M;
        const int in_row = p - pr * GROUP_M * ww;
        const int pc = in_row / (ph * PATCH_COLS);                               // patch
        const int in_patch = in_row - pc * ph * PATCH_COLS;
        return {rb * region_rows + pr * GROUP_M + in_patch % ph, cb * region_cols + pc * PATCH_COLS + in_patch / ph, true};
    }
};

// Slot numbering of the masked layout. Only the first masked_m[g] rows of a group exist, and the caller's `expected_m`
// says how many that usually is: the tile rows below it come first, all groups' stacked along m into one grid whose
// patches of 32 tiles (8 x 4, or as tall as a group where groups hold fewer tile-rows) are dealt out to the XCDs in turn (the
// 32 tiles an XCD runs at once share weight panels through its L2; consecutive patches go to different XCDs, so a group with few rows or none does not
// leave one XCD idle), the tile rows above it afterwards in a second grid of the same kind. A workgroup whose tile does not exist leaves at once, but
// it still takes a compute unit to start: numbered group by group, existing and empty tiles alternate and the existing
// ones start in ever smaller waves as the empty ones get out of their way (8 groups x 128 rows of which 64 exist: 58 us
// against 42 us when the rows are 64). Same on the host (slot count) and on the device (slot -> group, tile).
struct MaskedSlots {
    XcdTileScheduler<> likely, rest;
    int tiles_m, likely_rows, likely_slots;

    __host__ __device__ MaskedSlots(int num_groups, int m, int n, int block_m, int block_n, int expected_m)
        : likely(0, 0, block_m, block_n), rest(0, 0, block_m, block_n) {
        tiles_m = ceil_div(m, block_m);
        likely_rows = expected_m > 0 ? ceil_div(expected_m, block_m) : tiles_m;
        likely_rows = likely_rows < tiles_m ? likely_rows : tiles_m;
        likely = XcdTileScheduler<>(num_groups * likely_rows * block_m, n, block_m, block_n);
        rest   = XcdTileScheduler<>(num_groups * (tiles_m - likely_rows) * block_m, n, block_m, block_n);
        likely.fit_bands_to_groups(likely_rows);
        rest.fit_bands_to_groups(tiles_m - likely_rows);
        likely_slots = likely.grid_size();
    }

    __host__ __device__ long long num_slots() const { return (long long)likely_slots + rest.grid_size(); }

    // group and tile (within the group's [m, n] problem) of a slot
    __host__ __device__ TileCoord tile_of(int slot, int* group) const {
        const bool first = slot < likely_slots;
        const int rows = first ? likely_rows : tiles_m - likely_rows;
        TileCoord t = first ? likely.dealt_band_tile_of(slot) : rest.dealt_band_tile_of(slot - likely_slots);
        if (!t.valid) { *group = 0; return t; }
        *group = t.m_idx / rows;
        t.m_idx = t.m_idx % rows + (first ? 0 : likely_rows);
        return t;
    }
};

// The contiguous layout on tiles that follow the groups (fp8_gemm_contiguous_rows_kernel). A group is a run of 128-row blocks with
// one index; walked from its first block it is cut into tall tiles of two blocks and, where it has an odd number, a flat tile
// of one. Padding (negative indices) has neither. A wave looks at 64 blocks at a time, one per lane: this is what a lane
// knows of its block, and what follows from the ballot of `starts_run` and from the blocks in front of the 64.
struct ContiguousBlock {
    int group, behind;          // of this block and the next one; -1 past the end
    bool starts_run;

    __host__ __device__ ContiguousBlock(const int* grouped_layout, int blocks, int b) {
        const bool real = b < blocks;
        group = real ? grouped_layout[b * 128] : -1;
        const int before = real && b > 0 ? grouped_layout[(b - 1) * 128] : -1;
        behind = b + 1 < blocks ? grouped_layout[(b + 1) * 128] : -1;
        starts_run = b == 0 || group != before;
    }

    // How far into its run the block of lane `lane` is, counted from the last start of a run at or in front of it; `odd`: whether
    // the run that reaches the 64 blocks from in front is an odd number of blocks long there.
    __host__ __device__ static int into_run(unsigned long long starts, int lane, int odd) {
        const unsigned long long at_or_before = starts & (~0ull >> (63 - lane));
        return at_or_before ? lane - (63 - __builtin_clzll(at_or_before)) : lane + odd;
    }

    __host__ __device__ bool starts_tall(int into) const { return group >= 0 && (into & 1) == 0 && behind == group; }
    __host__ __device__ bool starts_flat(int into) const { return group >= 0 && (into & 1) == 0 && behind != group; }
};

// How many of a contiguous layout's tall tile rows run as two flat ones each: those of the tall tiles' last, partial round, where it
// is made of whole rows and all flat tiles then run at one time. A flat tile takes 0.7 to 0.8 of a tall one's time, so two flat
// rounds would take longer than the tall one, and so does a round in which some tall tiles are left: 8192 rows in 4 groups x
// 5120 x 7168, 128 tiles of 20 a row, 268 -> 279 us with six rows of them flat. With few k-tiles the flat tile's start weighs
// more. Whole rows, tall -> flat, 10240 rows in 6 groups x 4096: K = 512 39.7 -> 41.9 us, 1024 58.9 -> 60.2, 1536 79.3 -> 79.7, 2688 118.0 ->
// 117.5, 5120 213.5 -> 206.8; 6144 in 8 groups x 4096: K = 512 25.7 -> 26.9, 1536 52.3 -> 51.9, 2688 77.4 -> 75.4, 7168 180.1 -> 175.0.
__host__ __device__ inline int tall_rows_run_flat(int tall_rows, int flat_rows, int tiles_n, int compute_units, int k) {
    const long long tall = (long long)tall_rows * tiles_n, flat = (long long)flat_rows * tiles_n;
    const int over = int(tall % compute_units);
    if (k < 2048 || tall <= compute_units || over % tiles_n != 0) return 0;
    return flat + 2 * (long long)over <= compute_units ? over / tiles_n : 0;
}

// Workgroups to launch for `slots` units of work (tiles, or groups x tiles) under the caller's compute-unit cap, the
// `num_sms` of the reference's persistent kernels (yan/include/gemm/fp8_gemm.cuh:40 launches num_sms blocks,
// yan/jit_kernels/utils.py:6-29 holds the cap). No cap (0, or at least `device_cus`): one workgroup per slot, and the
// hardware hands them to compute units as they free up. A cap below the device's compute units: that many workgroups,
// rounded down to a multiple of the 8 XCDs so that slot b, b + grid, b + 2 grid, ... all fall to the same XCD and the
// scheduler's per-XCD ranges keep their meaning; workgroup b then walks those slots.
__host__ __device__ inline int capped_grid(int slots, int num_sms, int device_cus) {
    if (num_sms <= 0 || num_sms >= device_cus || num_sms >= slots) return slots;
    return num_sms >= kNumXCD ? num_sms / kNumXCD * kNumXCD : num_sms;
}

// Whether the plain FP8 GEMM on two LDS stages walks its tiles (fp8_gemm_walk) or runs a workgroup per tile: it walks, but for 3 to
// 17 k-tiles, an odd number, and outputs of up to 64 MB. A short tile leaves the walk little to hide its seam under, and tiles handed
// out as units fall free end more evenly: walk -> workgroup per tile, inputs changing, 7902 x 2624 x 640 26.8 -> 24.2 us, x 1152 38.3 ->
// 35.7, 8192 x 2560 x 1152 38.9 -> 36.0 (x 384 20.1 -> 21.3), 4096 x 7168 x 896 39.4 -> 36.6, x 1664 55.5 -> 53.9, 5222 x 1792 x 384 12.5 ->
// 11.7. Larger outputs gain by the walk at every K (8192 x 7168 x 384 42.6 -> 40.2 us, x 1152 78.2 -> 75.4), longer K gain at every
// size (4096 x 7168 x 9344 234 -> 230), and even numbers of k-tiles walk as they always have.
__host__ __device__ constexpr bool fp8_walk_pays(int k, uint64_t output_bytes) {
    return k % 256 == 0 || k > 17 * 128 || output_bytes > (uint64_t(64) << 20);
}

// Whether the persistent FP8 walk stores its output (`bytes`) with the non-temporal hint: outputs that would push the operands out of
// the 256 MB memory-side cache, from 64 MB on whatever K, from 32 MB on where the k-loop is long (operands many times the output).
// Plain -> hint, inputs changing: 8192 x 7168 x 768 57.4 -> 54.7 us, 4096 x 16384 x 3072 184.7 -> 175.2, 2048 x 12288 x 4096
// 100.8 -> 96.4, 4096 x 7168 x 7168 183.5 -> 177.3. Outputs of 32 to 64 MB behind a short K are quick to write and stay in that
// cache: 8192 x 2560 x 1024 27.1 -> 29.9, 4096 x 4608 x 768 21.8 -> 23.5, 2048 x 12288 x 2048 53.2 -> 54.7.
__host__ __device__ constexpr bool fp8_walk_streams_output(uint64_t bytes, int k) {
    return bytes > (uint64_t(k >= 3072 ? 32 : 64) << 20);
}

// Whether a ring tile's copies of the weights carry the non-temporal hint: so many weights that the 256 MB memory-side cache cannot
// hold them until their next use even in a program that goes round three such matrices, and each panel read once, by one tile
// row, or by a few that stay together because a row of K (`row_bytes`) is short. Such weights gain nothing from that cache, and left
// out of it they stream at 6.6 TB/s instead of 5.9: masked 32 groups x 8 rows x 4096 x 7168 158 -> 141 us, 8 x 30 rows 44 -> 40, contiguous
// 64 x 64 rows x 2048 x 4096 60.6 -> 57.7, FP8 64 x 16384 x 7168 26.8 -> 24.0, 16-bit 16 x 16384 x 4096 22.6 -> 19.6.
// Smaller ones may still be in the cache. From 32 MB on they gain as much where they are not (16-bit 32 x 8192 x 8192 31.1 -> 27.7, 37 x
// 4096 x 7168 15.1 -> 14.8) but lose more where they are (going round three: 16-bit 128 x 12288 x 2048 12.0 -> 17.6, FP8 16 x 16384 x
// 4096 13.4 -> 16.0, contiguous 32 x 64 rows x 2048 x 2048 14.7 -> 16.9). Tile rows drift apart along a long K, most of all where the last
// is ragged and runs ahead, and a panel that one has let go comes from HBM again for the next: FP8 300 x 8192 x 5120 28.3 -> 33.1,
// 16-bit 300 x 5000 x 7168 36.0 -> 44.9, where 256 rows, in step, gain 1 to 5 %; five tile rows and more are on two XCDs (900 x 3072 x
// 7168 on 64 x 192 62 -> 76.5). Rows of no whole 128-byte lines are read plainly: a k-tile ends inside a line, and the rest of it, wanted
// a k-tile later, is no longer there (fp16 26 x 12628 x 4760 35.7 -> 39.1).
__host__ __device__ constexpr bool streams_weights(int tile_rows, uint64_t weight_bytes, int row_bytes) {
    return (tile_rows <= 1 || (tile_rows <= 4 && row_bytes <= 4096)) && row_bytes % 128 == 0 && weight_bytes >= (uint64_t(96) << 20);
}

// Weights that a contiguous grouped launch reads at the most: of as many groups as it has blocks of 128 rows. (With 59 groups and ten
// blocks, 10 x 5184 x 1792, weights that the caches held were streamed for the sake of the 49 not read: 23.4 -> 26.2 us.)
__host__ __device__ constexpr uint64_t contiguous_weight_bytes(int num_groups, int m, int n, int k) {
    const int blocks = ceil_div(m, 128);
    return uint64_t(num_groups < blocks ? num_groups : blocks) * n * k;
}

// Whether four k-tiles of row-major scales a copy (Fp8ScaleCopies) are worth it in an unsplit plain FP8 GEMM of `tile_rows` rows of
// BLOCK_M x BLOCK_N tiles.
// On 64 x 64 tiles in a loop (K beyond 2048) they are not while a row's scales are at most one cache line (K = 4096), which stays in
// the caches from copy to copy where four tile rows and more read it: four a copy -> one, 300 x 2112 x 2560 11.0 -> 10.2 us, 395 x 1728 x
// 3072 12.7 -> 11.8, 500 x 1088 x 4096 15.3 -> 13.4, 256 x 4096 x 4096 17.0 -> 16.4. They are elsewhere: 64 x 64 with K = 1024 (256 x
// 3072 5.5 against 5.65), one tile row (62 x 16384 x 7168 30.0 against 33.4), 128 x 128 (1000 x 2112 x 4096 24.5 against 27.2).
__host__ __device__ constexpr bool fp8_scale_pieces_pay(int tile_rows, int block_m, int block_n, int k) {
    return block_m * block_n > 64 * 64 || tile_rows < 4 || k <= 2048 || k > 4096;
}

// Whether the tiles of a 16-bit ring launch start at different places along K (kSpreadStarts in bf16_gemm.hpp): rows a multiple
// of 16 KB apart, few tile rows, and
//   * weights of 48 MB and more. Smaller ones are often still in the 256 MB memory-side cache, whose channels do not mind, and
//     lose: going round three, 64 x 1024 x 16384 14.6 -> 15.3 us, 128 x 2048 x 8192 13.7 -> 14.3;
//   * activations that stay in an XCD's 4 MB of L2 while its tiles are all over the part's range of K (in step they stay whatever
//     their size): 400 x 8192 x 16384 141 -> 181 us, 256 x 16384 x 16384 176 -> 218, 128 x 45056 x 16384 269 -> 275 unsplit, but
//     256 x 8192 x 16384 in two parts 101 -> 96;
//   * at most two tile rows: with four nothing gains (200 x 1024 x 8192 14.5 -> 15.2 us, 400 x 4096 x 16384 77.8 -> 79.2).
// Where it spreads: 37 x 4096 x 8192 22.2 -> 18.4 us, 64 x 8192 x 16384 58.4 -> 50.8, 128 x 8192 x 16384 72.2 -> 59.0, 200 x 4096 x
// 16384 56.7 -> 51.7, 128 x 3072 x 8192 24.7 -> 24.1.
__host__ __device__ constexpr bool spreads_starts(int tile_rows, int m, uint64_t weight_bytes, int k, int split_k) {
    const uint64_t activations = uint64_t(m) * k * 2 / split_k, l2 = uint64_t(4) << 20;
    return k % 8192 == 0 && tile_rows <= 2 && weight_bytes >= (uint64_t(48) << 20) && (split_k > 1 ? activations <= l2 : activations < l2);
}

// Split-K workspaces (fp8_gemm.hpp, bf16_gemm.hpp): the arrival counters take the first kSplitKCounterBytes whatever the
// problem, so that launches of different shapes and kernels can share a workspace; the largest plan of the tile heuristics
// (256 workgroups of 128 x 128 partial sums) fits kSplitKWorkspaceBytes.
constexpr size_t kSplitKCounterBytes = 16 * 1024, kSplitKWorkspaceBytes = kSplitKCounterBytes + size_t(256) * 128 * 128 * 4;

} // namespace yan
