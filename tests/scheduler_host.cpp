// Host-side check of the workgroup -> tile mapping (gemm/scheduler.hpp is __host__ __device__): built and run by
// tests/test_host_cpu.py with `hipcc --cuda-host-only`, no device involved.
//
// For a range of (tiles_m, tiles_n) it asserts that
//   * tile_of over [0, grid_size()) visits every tile exactly once and marks the remaining slots invalid
//     (reference: yan/include/gemm/scheduler.cuh:39-41, num_blocks = ceil(m/BLOCK_M) * ceil(N/BLOCK_N));
//   * under every compute-unit cap, the walk b, b + grid, b + 2 grid, ... of capped_grid() workgroups covers every slot
//     exactly once and, for grids that are multiples of 8, never leaves the XCD residue b % 8;
//   * the masked layout's slot numbering (MaskedSlots) visits every (group, tile) once, likely tile rows first, and bands
//     fitted to the height of a group lose no tile and keep a patch inside one group;
//   * the contiguous layout cut along its groups (ContiguousBlock) covers every block of a group exactly once, no tile reaches
//     from one group into another, and the slots of the tall and flat tiles fit the launched ones and visit every tile once;
//   * the same holds in region order (operand rows long enough that the problem outgrows the memory-side cache), whose
//     choice of region is pinned for a few measured shapes.
#include "gemm/scheduler.hpp"

#include <cstdio>
#include <vector>

#define CHECK(cond)                                                                                   \
    do {                                                                                              \
        if (!(cond)) {                                                                                \
            std::printf("FAILED %s at %s:%d (m=%d n=%d bm=%d bn=%d)\n", #cond, __FILE__, __LINE__, m, n, bm, bn); \
            return 1;                                                                                 \
        }                                                                                             \
    } while (0)

int main() {
    int cases = 0, region_cases = 0, halved_cases = 0;
    const int blocks[][2] = {{256, 256}, {128, 256}, {64, 16}, {256, 224}};
    for (const auto& blk : blocks) {
        const int bm = blk[0], bn = blk[1];
        for (int tm = 1; tm <= 40; tm += (tm < 12 ? 1 : 7))
            for (int tn = 1; tn <= 70; tn += (tn < 10 ? 1 : 9)) {
                // ragged sizes: the last tile of each dimension holds a single row / column
                const int m = (tm - 1) * bm + 1, n = (tn - 1) * bn + 1;
                // bytes per operand row: 0 = band order; the others put problems of 256 tiles and more whose operands
                // outgrow the 256 MB cache into region order
                for (long long row_bytes : {0ll, 4096ll, 28672ll, 262144ll}) {
                const yan::XcdTileScheduler<> sched(m, n, bm, bn, row_bytes);
                if (row_bytes == 0 || tm * tn < 256) CHECK(sched.region_rows == 0);
                if (sched.region_rows) {
                    ++region_cases;
                    CHECK(sched.region_rows * sched.region_cols == 256 && sched.region_rows % 8 == 0 && sched.region_cols % 4 == 0);
                }
                CHECK(sched.tiles_m == tm && sched.tiles_n == tn && sched.total == tm * tn);
                const int slots = sched.grid_size();
                CHECK(slots >= sched.total && slots < sched.total + yan::kNumXCD && slots % yan::kNumXCD == 0);
                std::vector<int> seen(size_t(tm) * tn, 0);
                int invalid = 0;
                for (int bid = 0; bid < slots; ++bid) {
                    const yan::TileCoord t = sched.tile_of(bid);
                    if (!t.valid) { ++invalid; continue; }
                    CHECK(t.m_idx >= 0 && t.m_idx < tm && t.n_idx >= 0 && t.n_idx < tn);
                    ++seen[size_t(t.m_idx) * tn + t.n_idx];
                }
                CHECK(invalid == slots - sched.total);
                for (int v : seen) CHECK(v == 1);
                // walks under a cap
                for (int cap : {0, 1, 3, 8, 20, 64, 100, 255, 256, 300}) {
                    const int grid = yan::capped_grid(slots, cap, 256);
                    CHECK(grid >= 1 && grid <= slots);
                    if (cap <= 0 || cap >= 256 || cap >= slots) CHECK(grid == slots);
                    else CHECK(grid <= cap && (cap < yan::kNumXCD || grid % yan::kNumXCD == 0) && grid > cap - yan::kNumXCD);
                    std::vector<int> hit(slots, 0);
                    for (int b = 0; b < grid; ++b)
                        for (int slot = b; slot < slots; slot += grid) {
                            ++hit[slot];
                            if (grid % yan::kNumXCD == 0) CHECK(slot % yan::kNumXCD == b % yan::kNumXCD);
                        }
                    for (int v : hit) CHECK(v == 1);
                }
                ++cases;
                }
            }
    }
    // bands fitted to the tile-rows of a group (grouped layouts): still every tile exactly once, and with aligned groups the
    // 32 consecutive tiles of a patch stay inside one group
    for (int rows_per_group : {1, 2, 3, 4, 5, 8, 11})
        for (int groups : {1, 4, 9})
            for (int tn : {1, 7, 16, 40}) {
                const int bm = 256, bn = 256, tm = rows_per_group * groups, m = tm * bm, n = (tn - 1) * bn + 1;
                yan::XcdTileScheduler<> sched(m, n, bm, bn);
                sched.fit_bands_to_groups(rows_per_group);
                CHECK(sched.band_height == (rows_per_group < 8 ? rows_per_group : 8));
                std::vector<int> seen(size_t(tm) * tn, 0);
                for (int bid = 0; bid < sched.grid_size(); ++bid) {
                    const yan::TileCoord t = sched.tile_of(bid);
                    if (t.valid) { CHECK(t.m_idx >= 0 && t.m_idx < tm && t.n_idx >= 0 && t.n_idx < tn); ++seen[size_t(t.m_idx) * tn + t.n_idx]; }
                }
                for (int v : seen) CHECK(v == 1);
                if (rows_per_group <= 8 && 32 % rows_per_group == 0 && tn % (32 / rows_per_group) == 0)
                    for (int t0 = 0; t0 + 32 <= sched.total; t0 += 32) {
                        const int g0 = sched.band_tile(t0).m_idx / rows_per_group;
                        for (int t = t0; t < t0 + 32; ++t) CHECK(sched.band_tile(t).m_idx / rows_per_group == g0);
                    }
                ++cases;
            }
    // the masked layout's slot numbering: every (group, tile) exactly once, the tile rows below expected_m before the others
    for (int groups : {1, 3, 8, 17})
        for (int tm = 1; tm <= 9; tm += (tm < 3 ? 1 : 3))
            for (int tn : {1, 5, 16, 33})
                for (int expected : {0, 1, 100, 257, 100000}) {
                    const int bm = 128, bn = 256, m = (tm - 1) * bm + 1, n = (tn - 1) * bn + 1;
                    const yan::MaskedSlots slots(groups, m, n, bm, bn, expected);
                    CHECK(slots.num_slots() % yan::kNumXCD == 0 && slots.num_slots() < (long long)groups * tm * tn + 2 * yan::kNumXCD);
                    std::vector<int> seen(size_t(groups) * tm * tn, 0);
                    const int likely_rows = expected <= 0 ? tm : ((expected + bm - 1) / bm < tm ? (expected + bm - 1) / bm : tm);
                    bool rest_seen = false;
                    for (int s = 0; s < slots.num_slots(); ++s) {
                        int g = -1;
                        const yan::TileCoord t = slots.tile_of(s, &g);
                        if (!t.valid) continue;
                        CHECK(g >= 0 && g < groups && t.m_idx >= 0 && t.m_idx < tm && t.n_idx >= 0 && t.n_idx < tn);
                        ++seen[(size_t(g) * tm + t.m_idx) * tn + t.n_idx];
                        if (t.m_idx >= likely_rows) rest_seen = true;
                        else CHECK(!rest_seen);
                    }
                    for (int v : seen) CHECK(v == 1);
                    ++cases;
                }
    // the contiguous layout on tiles that follow the groups: layouts of up to 200 blocks in runs of 1 to 70, padding among them,
    // cut 64 blocks at a time as a wave does it
    unsigned rng = 1;
    auto random = [&](int below) { rng = rng * 1664525u + 1013904223u; return int((rng >> 8) % unsigned(below)); };
    for (int trial = 0; trial < 2000; ++trial) {
        const int bm = 256, bn = (trial / 4) % 2 ? 256 : 128, tn = (trial / 8) % 2 ? 1 << random(4) : 1 + random(20), n = (tn - 1) * bn + 4 + random(bn - 4);
        std::vector<int> group_of;
        const int blocks = 1 + random(200), longest = trial % 3 == 0 ? 70 : (trial % 3 == 1 ? 4 : 1);
        for (int g = 0; int(group_of.size()) < blocks;) {
            const int run = 1 + random(longest), group = random(5) == 0 ? -1 - random(2) : g++;
            for (int r = 0; r < run && int(group_of.size()) < blocks; ++r) group_of.push_back(group);
        }
        const int m = blocks * 128 - (trial % 5 == 0 ? random(127) : 0);
        std::vector<int> layout(size_t(blocks) * 128);
        for (int b = 0; b < blocks; ++b) for (int r = 0; r < 128; ++r) layout[b * 128 + r] = group_of[b];
        std::vector<int> covered(blocks, 0);
        int tall_rows = 0, flat_rows = 0, odd = 0;
        for (int chunk = 0; chunk * 64 < blocks; ++chunk) {
            unsigned long long starts = 0;
            for (int lane = 0; lane < 64; ++lane)
                if (yan::ContiguousBlock(layout.data(), blocks, chunk * 64 + lane).starts_run) starts |= 1ull << lane;
            for (int lane = 0; lane < 64; ++lane) {
                const int b = chunk * 64 + lane, into = yan::ContiguousBlock::into_run(starts, lane, odd);
                const yan::ContiguousBlock block(layout.data(), blocks, b);
                CHECK(!(block.starts_tall(into) && block.starts_flat(into)));
                if (block.starts_tall(into)) {
                    CHECK(b + 1 < blocks && group_of[b] >= 0 && group_of[b + 1] == group_of[b]);
                    ++covered[b], ++covered[b + 1], ++tall_rows;
                }
                if (block.starts_flat(into)) {
                    CHECK(b < blocks && group_of[b] >= 0);
                    ++covered[b], ++flat_rows;
                }
            }
            odd = (yan::ContiguousBlock::into_run(starts, 63, odd) + 1) & 1;
        }
        for (int b = 0; b < blocks; ++b) CHECK(covered[b] == (group_of[b] >= 0 ? 1 : 0));
        const long long launched = (long long)yan::XcdTileScheduler<>(m, n, 128, bn).grid_size() + yan::kNumXCD;
        const int cus[] = {1 << 30, 8, 40, 256};          // 2^30: no tall row ever runs flat
        const int halved = yan::tall_rows_run_flat(tall_rows, flat_rows, tn, cus[trial % 4], 2048);
        CHECK(halved >= 0 && halved <= tall_rows && (trial % 4 != 0 || halved == 0));
        CHECK(yan::tall_rows_run_flat(tall_rows, flat_rows, tn, cus[trial % 4], 1920) == 0);
        if (halved) {        // whole rounds of tall tiles, then all the rest at one time
            CHECK((tall_rows - halved) * tn % cus[trial % 4] == 0 && (flat_rows + 2 * halved) * tn <= cus[trial % 4]);
            ++halved_cases;
        }
        tall_rows -= halved;
        flat_rows += 2 * halved;
        yan::XcdTileScheduler<> tall(tall_rows * 256, n, 256, bn), flat(flat_rows * 128, n, 128, bn);
        tall.fit_bands_to_groups(tall_rows / 3);
        flat.fit_bands_to_groups(1);
        CHECK((long long)tall.grid_size() + flat.grid_size() <= launched);
        for (const auto* tiles : {&tall, &flat}) {
            const int rows = tiles == &tall ? tall_rows : flat_rows;
            std::vector<int> seen(size_t(rows) * tn, 0);
            for (int slot = 0; slot < tiles->grid_size(); ++slot) {
                const yan::TileCoord t = tiles->dealt_band_tile_of(slot);
                if (!t.valid) continue;
                CHECK(t.m_idx >= 0 && t.m_idx < rows && t.n_idx >= 0 && t.n_idx < tn);
                ++seen[size_t(t.m_idx) * tn + t.n_idx];
            }
            for (int v : seen) CHECK(v == 1);
        }
        ++cases;
    }
    // what the traffic model picks for shapes that were measured (bf16, 256 x 256 tiles)
    {
        const int m = 0, n = 0, bm = 256, bn = 256;
        const yan::XcdTileScheduler<> a(8192, 8192, 256, 256, 12288 * 2), b(8192, 4096, 256, 256, 14336 * 2),
            c(12288, 12288, 256, 256, 12288 * 2), d(8192, 8192, 256, 256, 8192 * 2), e(16384, 16384, 256, 256, 16384);
        CHECK(a.region_rows == 32 && a.rows_outer);          // the activation block stays: what band order amounts to
        CHECK(b.region_rows == 16 && c.region_rows == 32);
        CHECK(d.region_rows == 0);                           // 2 x 128 MiB of operands fit
        CHECK(e.region_rows == 32 && e.rows_outer);          // the FP8 16384^3 shape
        CHECK(region_cases > 100 && halved_cases > 10);
        CHECK(yan::tall_rows_run_flat(32, 0, 20, 256, 7168) == 0);          // 120 of 128 tiles would be flat, 8 stay tall
        CHECK(yan::tall_rows_run_flat(24, 0, 16, 256, 7168) == 8 && yan::tall_rows_run_flat(38, 4, 16, 256, 7168) == 6);
    }
    {
        // Outputs the walk stores with the non-temporal hint: from past 64 MB, behind a long K from past 32 MB.
        const int m = 0, n = 0, bm = 256, bn = 256;
        const uint64_t mb = uint64_t(1) << 20;
        // Launches whose tiles start at different places along K: (tile rows, m, n, k, parts)
        auto spreads = [](int rows, int m, int n, int k, int parts) { return yan::spreads_starts(rows, m, uint64_t(n) * k * 2, k, parts); };
        CHECK(spreads(1, 37, 4096, 8192, 4) && spreads(2, 128, 16384, 8192, 1) && spreads(2, 256, 8192, 16384, 2) && spreads(1, 37, 3072, 8192, 4));
        CHECK(!spreads(1, 64, 1024, 16384, 8) && !spreads(4, 200, 4096, 8192, 4) && !spreads(1, 37, 4096, 7168, 4));
        CHECK(!spreads(2, 256, 16384, 16384, 1) && !spreads(2, 256, 16384, 8192, 1) && !spreads(4, 400, 8192, 16384, 1) && !spreads(1, 128, 45056, 16384, 1));
        // Row-major scales four k-tiles at a time: not where many 64 x 64 tile rows loop over few of them.
        CHECK(!yan::fp8_scale_pieces_pay(5, 64, 64, 2560) && !yan::fp8_scale_pieces_pay(4, 64, 64, 4096) && yan::fp8_scale_pieces_pay(3, 64, 64, 2560));
        CHECK(yan::fp8_scale_pieces_pay(5, 64, 64, 2048) && yan::fp8_scale_pieces_pay(5, 64, 64, 4608) && yan::fp8_scale_pieces_pay(5, 64, 128, 2560));
        // Weights whose rows end inside a 128-byte line are not streamed.
        CHECK(!yan::streams_weights(1, 12628ull * 4760 * 2, 4760 * 2) && yan::streams_weights(1, 12672ull * 4736 * 2, 4736 * 2));
        // A contiguous layout of few blocks reads few groups' weights.
        CHECK(yan::contiguous_weight_bytes(59, 1280, 5184, 1792) == 10ull * 5184 * 1792 && yan::contiguous_weight_bytes(4, 1280, 512, 256) == 4ull * 512 * 256);
        CHECK(!yan::streams_weights(1, yan::contiguous_weight_bytes(59, 1280, 5184, 1792), 1792));
        // Problems that walk: not the odd numbers of up to 17 k-tiles, unless the output is large.
        CHECK(!yan::fp8_walk_pays(384, 64 * mb) && !yan::fp8_walk_pays(640, 2ull * 7902 * 2624) && !yan::fp8_walk_pays(2176, 0));
        CHECK(yan::fp8_walk_pays(384, 64 * mb + 8) && yan::fp8_walk_pays(2432, 0) && yan::fp8_walk_pays(256, 0) && yan::fp8_walk_pays(2048, 0));
        CHECK(!yan::fp8_walk_streams_output(2ull * 8192 * 2560, 1024) && !yan::fp8_walk_streams_output(2ull * 4096 * 7168, 512));
        CHECK(yan::fp8_walk_streams_output(2ull * 8192 * 7168, 512) && yan::fp8_walk_streams_output(2ull * 4096 * 7168, 7168));
        CHECK(!yan::fp8_walk_streams_output(64 * mb, 2944) && yan::fp8_walk_streams_output(64 * mb + 8, 2944));
        CHECK(!yan::fp8_walk_streams_output(32 * mb, 3072) && yan::fp8_walk_streams_output(32 * mb + 8, 3072));
    }
    std::printf("ok %d\n", cases);
    return 0;
}
