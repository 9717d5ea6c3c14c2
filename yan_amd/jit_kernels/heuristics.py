"""Macro-tile selection for a 256-CU part.

The reference leaves this open: its dense entry hard-codes one tile and an empty tuning space
(`yan/jit_kernels/cute_gemm.py:39-53`) and its FP8 template takes BLOCK_M / BLOCK_N as keys without saying who
picks them (`yan/jit_kernels/gemm.py:13-16`). Here a small cost model ranks the tiles the kernels support:
one workgroup per tile, one workgroup per CU at a time, so a launch costs
`ceil(tiles / num_cus)` rounds of one tile time, and a tile's time grows with its MFMA work but shrinks per
flop as the tile gets larger (fewer operand bytes fetched per flop).
"""
import functools
from typing import List, Optional, Tuple

from .utils import ceil_div, env_switch

# (BLOCK_M, BLOCK_N): relative time per unit of tile area. Bigger tiles reuse operands better.
# Dense tiles: 256 rows x {256, 224, 192, 160} columns run the persistent 4-wave kernel with a ring of five LDS units (the
# 8-wave kernel on two stages for short or ragged K), the others the 4-wave kernel with a ring of stages. Costs of the 256-row
# tiles are measured: time per output of a problem that fills four whole rounds of 256 compute units with the tile
# (8192 x 32 BLOCK_N x 8192), relative to 256 x 256 (1.02-1.04, 1.035-1.06, 1.07-1.10 over three boxes). The ring tiles measure
# 1.30-1.32 (256 x 128, 128 x 256) and 1.49 (128 x 128) there, but no problem of four rounds ever takes them: where they
# compete, in launches of one or two rounds, a tile pays its first loads and its epilogue in full, and 1.40 / 1.42 is what
# made the table's pick the fastest tile or within 1.2 % of it on all 67 shapes swept with every tile forced in turn (with
# 1.30, 128 x 256 took eight one-round shapes from 256 x 160, which is 4 to 17 % faster there). That was before the ring tiles
# had waves that only copy: over 70 shapes since then the pick is within 2 % of the fastest on 57, and 64 x 192 is 5 to 17 %
# behind 128 x 128 on seven (670 x 4416 x 3264 29.5 against 25.2 us).
# 128 x 192 and 64 x 192 (ring kernel, wave slabs 96 columns wide) are for problems that leave most compute units idle with
# 256-wide tiles and need two rounds with 128-wide ones (2048 x 2112 x 7168: 144 tiles of 128 x 256 run 85 us, 176 of 128 x 192 68 us).
_DENSE_TILES = {(256, 256): 1.00, (256, 224): 1.03, (256, 192): 1.05, (256, 160): 1.085, (256, 128): 1.42, (128, 256): 1.40,
                (128, 192): 1.43, (128, 128): 1.51, (64, 192): 1.96, (64, 128): 2.0, (64, 64): 2.78}
# FP8 tiles: measured over 74 shapes (m = 17 ... 8192, n = 2048 ... 32768, k = 512 ... 16384) with every tile forced in turn;
# with these costs the model's pick is within 1 % of the fastest tile on all of them. 256 x 192 and 256 x 160 are there for
# problems whose 256 x 256 tiles leave a round of compute units partly empty (4096 x 5120 x 5120: 320 tiles, against 512
# tiles of 256 x 160 = two full rounds, 13 % faster); 256 x 224 and 64 x 160 are supported by the kernel and never the
# cheapest (a round of 64 x 160 tiles takes longer than a round of 128 x 128 tiles, which run eight waves).
_FP8_TILES = {(256, 256): 1.00, (256, 192): 1.12, (256, 160): 1.28, (256, 128): 1.34, (128, 256): 1.34, (128, 128): 1.5,
              (64, 128): 2.3, (64, 64): 3.55, (64, 32): 4.8, (32, 32): 7.0}


def rank_tiles(m: int, n: int, num_cus: int, table, groups: int = 1) -> List[Tuple[float, Tuple[int, int]]]:
    ranked = []
    for (bm, bn), per_area in table.items():
        tiles = ceil_div(m, bm) * ceil_div(n, bn) * groups
        rounds = ceil_div(tiles, num_cus)
        ranked.append((rounds * bm * bn * per_area, (bm, bn)))
    return sorted(ranked)


def tuning_enabled() -> bool:
    """Empirical tile selection on the first call per shape (`YAN_TUNE_TILES=1`): the entry points hand the cost model's
    three best tiles to the tuner as its `space` and the fastest on the device wins, as the reference's tuner does with
    its candidate list (`yan/jit_kernels/cute_gemm.py:42-53`, `tuner.py:42-69`). Off by default: the first call of a
    shape then costs up to three compilations and sixty timed launches."""
    return env_switch(b'YAN_TUNE_TILES', False)


def get_dense_tile_space(m: int, n: int, k: int, num_cus: int, count: int = 3) -> List[Tuple[int, int]]:
    return [tile for _, tile in rank_tiles(m, n, num_cus, _DENSE_TILES)[:count]]


def get_fp8_tile_space(m: int, n: int, k: int, num_cus: int, count: int = 3) -> List[Tuple[int, int]]:
    return [tile for _, tile in rank_tiles(m, n, num_cus, _FP8_TILES)[:count]]


def get_best_dense_config(m: int, n: int, k: int, num_cus: int) -> Tuple[int, int]:
    return rank_tiles(m, n, num_cus, _DENSE_TILES)[0][1]


def get_best_fp8_config(m: int, n: int, k: int, num_cus: int) -> Tuple[int, int]:
    return rank_tiles(m, n, num_cus, _FP8_TILES)[0][1]


def get_dense_num_stages(block_m: int, block_n: int) -> int:
    """LDS stages of the dense kernel for a tile: 2 names the persistent kernels of the tiles with 256 rows and more than 128
    columns (8 waves on two stages, or 4 waves on a ring of five operand units for 256 x 256: the launcher chooses), else as
    many as the 160 KB LDS holds, at most 8 (`DenseTileConfig::MAX_STAGES` in bf16_gemm.hpp): 3 for 128 x 256, ... 8 for 64 x 64."""
    if block_m == 256 and block_n > 128:
        return 2            # the persistent kernels, whatever the width
    return min(8, 160 * 1024 // ((block_m + block_n) * 128))


def get_fp8_num_stages(block_m: int, block_n: int) -> int:
    """LDS stages of the tiled FP8 kernel for a tile: a ring as deep as the 160 KB LDS allows, at most 8, or 12 for the
    tiles of 32 weight rows that run the decode shapes (`Fp8TileConfig::MAX_RING_STAGES` in fp8_gemm.hpp): 2 for
    256 x 256, 3 for 256 x 128 and 128 x 256, 8 for 64 x 64, 12 for 64 x 32 and 32 x 32. Tiles below 256 x 256 are what the cost model picks when a problem is short on work per CU, i.e. bound by
    operand streaming, and there one k-tile of prefetch does not cover the memory latency."""
    waves = 4               # get_num_waves in mfma_utils.hpp
    if block_m * block_n >= 256 * 128 or (block_m * block_n >= 64 * 64 and block_m % 64 == 0 and block_n % 64 == 0):
        waves = 8
    capable = block_m % 32 == 0 and (block_m // 8) % waves == 0 and block_n % 16 == 0
    if not capable:
        return 2
    rows = ceil_div(block_m, 8 * waves) * 8 * waves + ceil_div(block_n, 8 * waves) * 8 * waves      # whole copy passes
    stage_bytes = rows * 128 + ceil_div(block_m * 4, 1024) * 1024
    return max(2, min(12 if block_n <= 32 else 8, 160 * 1024 // stage_bytes))


def get_best_grouped_fp8_config(m: int, n: int, k: int, num_cus: int, groups: int = 1, m_alignment: int = 0,
                                groups_in_m: int = 1) -> Tuple[int, int]:
    """Tile of a grouped FP8 GEMM, among the tiles 64, 128 or 256 columns wide. Contiguous layout: `m` is the total row count and
    `m_alignment` the padding of every group, which the tile's rows must divide. 256 x 128, whose tiles follow the `groups_in_m`
    groups as the 256 x 256 ones of `get_contiguous_rows_on_device` do, is offered when they average 1024 rows or more and the
    tiles are more than one round: 10 groups, 15104 x 2112 x 5760 244 us on 128 x 128 tiles, 220 on these; 3 groups, 8832 x 3648 x
    5632 231 and 203; 23 such shapes 0.88 to 1.03 times the time on 128 x 128, one 1.11. In one round it loses (4 groups,
    4352 x 1856 x 6912: 73 us on 128 x 128, 86 on these). Masked layout: `m` is the expected row count of one group and `groups` multiplies
    the tile count."""
    def allowed(bm, bn):
        if m_alignment == 0 or m_alignment % bm == 0:
            return True
        return (bm, bn) == (2 * m_alignment, 128) and m >= 1024 * groups_in_m and ceil_div(m, bm) * ceil_div(n, bn) > num_cus
    table = {t: c for t, c in _FP8_TILES.items() if t[1] in (64, 128, 256) and allowed(*t)}
    return rank_tiles(max(m, 1), n, num_cus, table, groups)[0][1]


def _tall_then_flat(tall: int, flat: int, num_cus: int) -> float:
    """When the last of `tall` tiles of 256 x 256 and, behind them, `flat` ones of 128 x 256 ends, in times of a tall tile, with every
    compute unit taking the next tile when it is done with one."""
    flat_time = _FP8_TILES[(128, 256)] / 2
    full, over = divmod(tall, num_cus)          # `over` units run one tall tile more than the others
    end = full + (1 if over else 0)
    early, late = full + flat_time, full + 1 + flat_time        # when the next flat tile ends on a unit of either kind
    while flat > 0:
        if over == 0 or early <= late:
            flat -= num_cus - over
            end = max(end, early)
            early += flat_time
        else:
            flat -= over
            end = max(end, late)
            late += flat_time
    return end


def get_contiguous_rows_on_device(m: int, n: int, k: int, num_cus: int, groups_in_m: int) -> bool:
    """Whether a contiguous grouped GEMM runs the kernel whose tiles follow the groups (`fp8_gemm_contiguous_rows_kernel`: 256 x
    256 tiles and, for the odd block of a group, 128 x 256): groups that average a block of 128 rows or more, for which the
    cost table, with 256-row tiles allowed, takes 256 x 256. Against 128 x 256 tiles and 256-row tiles on a fixed grid, which ran
    two passes over K where a tile held two groups: 16 groups of 128 to 768 rows x 4096 x 7168 220 -> 197 us, 4 of about 2500 290 ->
    276, 7 of about 2300 x 2112 x 5120 210 -> 197; level (0.5 %) for 4 of 8192.
    Groups that average less than 256 rows have no tile row of 256 rows to every 256: the table counts too few tiles there.
    They are priced by what runs if every second group has an odd number of blocks, tall tiles first. Next to 128 x 256 tiles a
    launch takes 750 k-rows of a tall tile more, for finding the tiles and filling three stages; next to 128 x 128 tiles, whose
    rounds each have a start of their own, 180 per round, and those cost 1.36 times what the table says (it comes from plain
    problems, where their panels are shared). Measured, 128-row tile that the table takes -> this kernel: 64 of about 130 x 7168 x
    2048 190 -> 175, 32 of about 190 x 4096 x 4096 142 -> 130, 24 of about 165 x 2880 x 2048 46 -> 41 (taken); 49 of about 200 x 1344 x
    1280 34.1 -> 40.1, 43 of about 165 x 2112 x 1152 32.7 -> 38.8, 46 of about 180 x 1344 x 1024 28.0 -> 31.9, 41 of about 205 x 1600 x
    1664 40.3 -> 46.4 (not taken). Over the 78 shapes the rule was made on its pick takes 0.90 of the time of the 128-row tile (1.04
    at worst), over 44 others 0.74 to 1.02. Same rule as `rows_on_device` in yan_amd/csrc/yan_gemm_capi.hip."""
    if groups_in_m <= 0 or m < 128 * groups_in_m:
        return False
    table = {t: c for t, c in _FP8_TILES.items() if t[1] in (64, 128, 256) and t[0] in (64, 128, 256)}
    if rank_tiles(m, n, num_cus, table)[0][1] != (256, 256):
        return False
    if m >= 256 * groups_in_m:
        return True
    blocks, tiles_n = ceil_div(m, 128), ceil_div(n, 256)
    tall_rows = (blocks - (groups_in_m + 1) // 2) // 2
    time = _tall_then_flat(tall_rows * tiles_n, (blocks - 2 * tall_rows) * tiles_n, num_cus)
    cost, tile = rank_tiles(m, n, num_cus, {t: c for t, c in table.items() if t[0] <= 128})[0]
    if tile == (128, 128):
        return time * (1 + 180 / max(k, 1)) * 65536 < cost * 1.36
    return (time + 750 / max(k, 1)) * 65536 < cost


def get_skinny_fp8_config(m: int, n: int, k: int, num_cus: int) -> int:
    """Number of 16-row activation atoms (1) when the weight-streaming kernel runs instead of the tiled one where K is not split,
    else 0: up to 16 activation rows, and few enough weight rows that n / 16 workgroups fit the chip in one round. There it is
    faster than the tiles whatever K is (16 rows x 1472 x 15104: 9.7 us). `get_weight_stream_fp8_config` says where it also goes
    before a split-K plan and which problems beyond these it takes."""
    if 0 < m <= 16 and 16 <= n <= 16 * num_cus:
        return 1
    return 0


def get_skinny_dense_config(m: int, n: int, k: int, num_cus: int) -> int:
    """The same for the dense 16-bit GEMM: 1 or 2 atoms, whole 128-byte K blocks. `get_weight_stream_dense_config` says where the
    kernel also goes before a split-K plan and which problems beyond these it takes."""
    if n < 16 or n > 16 * num_cus or n % 4 or k <= 0 or k % 64:
        return 0
    if 0 < m <= 16:
        return 1
    if 16 < m <= 32 and k >= 2048:
        return 2
    return 0


def _weight_stream_pull(m: int, n: int, k_bytes: int, num_cus: int) -> Tuple[int, int, int]:
    """Bytes a workgroup of the weight-streaming kernel pulls: its 8 to 32 or (up to 32 activation rows) 64 weight rows, as few as
    give one round of workgroups (`launch_weight_stream` in gemm/weight_stream.hpp), and all `m` activation rows; 0 when that takes
    more than a round, or beyond 32-bit offsets. Also those weight rows, and the number of workgroups."""
    if m <= 0 or m > 64 or n < 16 or n % 4 or k_bytes <= 0 or k_bytes % 128 or (n + 64) * k_bytes >= 1 << 31:
        return 0, 0, 0
    for rows in (8, 16, 24, 32, 40, 48, 64):
        if ceil_div(n, rows) <= num_cus and (rows <= 32 or m <= 32):
            return (rows + m) * k_bytes, rows, ceil_div(n, rows)
    return 0, 0, 0


@functools.lru_cache(maxsize=None)
def get_weight_stream_fp8_config(m: int, n: int, k: int, num_cus: int) -> int:
    """Number of 16-row activation atoms (1 to 4) when the weight-streaming kernel goes before split-K plans and tiles, else 0.

    Its time is 3.3 us + what a workgroup pulls at about 62 bytes/ns, or the weights at 6 to 7 TB/s; a split-K plan
    pays 2 us for the meeting of the parts, the tiles of a short K too few workgroups. Measured per call, weights cycling through
    more matrices than the caches hold, 60 shapes of n = 128 .. 16384, k = 512 .. 16384, up to ten m each (split-K plan or tiles -> this
    kernel): 1 x 2112 x 7168 8.7 -> 5.4 us, 1 x 4096 x 7168 9.8 -> 7.6, 16 x 1984 x 4608 6.7 -> 4.5, 32 x 2944 x 5632 10.3 -> 7.8,
    40 x 4096 x 16384 22.3 -> 19.8, 8 x 10240 x 7168 22.5 -> 15.0, 32 x 16384 x 16384 53.8 -> 47.5. It loses
    up to 40 rows only where a workgroup of 8 or 16 weight rows pulls more than 400 KB (8 weight rows from 17 rows on: 285 KB, 25 x 1856 x 9728
    8.1 -> 8.7) and they do not fill the chip (20 x 1472 x 15104 10.9 -> 11.3), and up to 16 rows on 64 weight rows beyond 800 KB (10 x 13184 x 11264
    30.0 -> 30.9); with 48 rows it is level from 300 KB on (4096 x 7168 11.1 -> 11.3), 400 KB on more weight rows
    (4100 x 7168 12.2 at 516 KB both ways, but 8192 x 4096 11.1 -> 10.1); with 64 from 130 KB on (4096 x 2048 4.7 -> 4.8;
    3072 x 1536 4.5 -> 4.2; 2112 x 7168 10.3 -> 12.2; 7168 x 2048 7.1 both ways), on 24 weight rows 365 KB (4224 x 4096
    10.5 -> 9.5; 5120 x 8192 14.2 -> 16.2 at 721 KB). Same rule as `weight_stream_fp8_atoms` in yan_amd/csrc/yan_gemm_capi.hip."""
    pull, rows, groups = _weight_stream_pull(m, n, k, num_cus)
    full, wide = rows >= 16 and groups * 8 >= num_cus * 7, rows >= 24
    if not pull:
        return 0
    if m <= 32:
        takes = pull <= (285_000 if rows == 8 and m > 16 else 400_000) or full or n >= 16 * num_cus
        if rows == 64 and m <= 16:
            takes = pull <= 800_000
    elif m <= 40:
        takes = pull <= 400_000 or full or wide
    elif m <= 48:
        takes = pull <= (400_000 if wide else 300_000) or (rows == 32 and full)
    else:
        takes = pull <= (365_000 if rows == 24 else 130_000)
    return ceil_div(m, 16) if takes else 0


@functools.lru_cache(maxsize=None)
def get_weight_stream_dense_config(m: int, n: int, k: int, num_cus: int) -> int:
    """The same for the dense 16-bit GEMM, whose smallest tile holds 64 weight rows: while a workgroup pulls no more than a limit that
    depends on its weight rows, on m and on how much of the chip they fill. The limits are from 2000 shapes of n = 1024 .. 16384, k = 1024 ..
    16384, weights cycling (time here : time of split-K plan or tiles): there and below it is 0.70 to 1.02 (0.81 on average over 700 other shapes in
    the upper half of the limits, three above 1.03), beyond, on 24 weight rows, 0.97 to 1.11 (14 x 4428 x 15360 26.0 -> 28.9 us, 17 x 4736 x 8832 19.6 ->
    21.8), on 32 1.0 to 1.12 (6 x 7992 x 15872 40.5 -> 45.6), on 48 0.86 to 1.10 (4 x 12288 x 8192 33.3 -> 36.5), on 64 1.04 to 1.10 (1 x 15116 x 4608
    23.0 -> 25.3, and from 17 rows on between K = 1024 and 2048, 30 x 13888 x 1408 9.9 -> 10.3), with 33 to 64 rows 1.03 to 1.09 (48 x 4096 x 4480 11.7 -> 12.8, 63 x 7872 x 2688 12.9 -> 13.6). Up to 16
    rows 8 and 16 weight rows go on any K (1 x 1024 x 7168 12.7 -> 5.5, 16 x 1472 x 15104 31.1 -> 16.7, 16 x 2112 x 7168 11.5 -> 11.6, the
    closest). Same rule as `weight_stream_dense_atoms` in yan_amd/csrc/yan_gemm_capi.hip."""
    pull, rows, groups = _weight_stream_pull(m, n, 2 * k, num_cus)
    full = groups * 8 >= num_cus * 7
    if not pull:
        return 0
    if rows <= 16:
        limit = 580_000 if rows == 16 and full and m <= 32 else 450_000
    elif rows == 24:
        limit = (850_000 if full else 700_000) if m <= 16 else (850_000 if full else 500_000) if m <= 32 else 450_000 if full else 350_000
    elif rows == 32:
        limit = 750_000 if m <= 16 else 450_000 if m > 48 else 780_000 if full else 600_000
    elif rows == 64:
        limit = 440_000 if m <= 16 else 600_000 if k >= 2048 or k <= 1024 else 0
    else:
        limit = 830_000 if rows == 48 and m <= 16 else 1_200_000
    return ceil_div(m, 16) if pull <= limit or (m <= 16 and rows <= 16) else 0


def get_cast_stream_rows(m: int, n: int, k: int, num_cus: int) -> int:
    """Activation rows (1, 2, 4 or 8) the weight-streaming kernel quantises itself when it takes bf16 activations, else 0: problems it
    takes with FP8 activations, up to 8 rows, whose quantising is shorter than the launch it saves. Every workgroup repeats it for
    all rows, four groups of 128 numbers a step, the waves a share of K each while their first weights are on the way. Measured per call, weights
    cycling, against quantiser and GEMM in two launches, same bits: 1 row: 2112 x 7168 7.9 -> 6.0 us, 1024 x 2048 6.0 -> 3.9, 5120 x 8192 11.6 -> 9.4,
    9152 x 16000 29.3 -> 26.9; 4 rows: 7 steps, 2112 x 7168 8.2 -> 7.8, 16384 x 2048 9.8 -> 7.8; 2 rows x 1472 x 15104, 8 steps on 8 weight rows a
    workgroup, 9.3 -> 9.5 (not taken); 8 rows: 4 steps, 7168 x 2048 7.6 -> 6.1, 8 steps, 3008 x 3328 6.3 -> 6.7 (not taken). `cast_rows` in
    gemm/weight_stream.hpp names the rows."""
    if not 0 < m <= 8 or not get_weight_stream_fp8_config(m, n, k, num_cus):
        return 0
    rows = 1 if m == 1 else 2 if m == 2 else 4 if m <= 4 else 8
    steps = ceil_div(ceil_div(k // 128, 8) * rows, 4)
    return rows if steps <= (4 if rows == 8 else 8 if n > 8 * num_cus else 7) else 0


def get_dense_tile(m: int, n: int, k: int, num_cus: int) -> Tuple[int, int]:
    """(BLOCK_M, BLOCK_N) of the dense kernel that runs: (16 * atoms, 16) for the weight-streaming kernel."""
    atoms = get_weight_stream_dense_config(m, n, k, num_cus) or get_skinny_dense_config(m, n, k, num_cus)
    return (16 * atoms, 16) if atoms else get_best_dense_config(m, n, k, num_cus)


def get_fp8_tile(m: int, n: int, k: int, num_cus: int) -> Tuple[int, int]:
    """(BLOCK_M, BLOCK_N) of the FP8 kernel that runs: (16 * atoms, 16) for the weight-streaming kernel."""
    atoms = get_weight_stream_fp8_config(m, n, k, num_cus) or get_skinny_fp8_config(m, n, k, num_cus)
    return (16 * atoms, 16) if atoms else get_best_fp8_config(m, n, k, num_cus)


# Split-K of the FP8 GEMM: microseconds a workgroup spends per k-tile on a ring tile when every compute unit runs one
# (measured: m x 4096 x 7168, sizes at run time, 56 k-tiles, one round of workgroups). Only used to weigh split-K plans
# against the unsplit pick of the cost table above.
_FP8_SPLIT_K_TILE_US = {(32, 32): 0.133, (64, 32): 0.192, (64, 64): 0.296, (64, 128): 0.395, (128, 128): 0.51}
# The same for the unsplit kernel, which pulls its weights with fewer workgroups at a time and, a workgroup per tile, runs
# without a loop around the tile: 0.88 to 0.975 of the figures above.
_FP8_UNSPLIT_TILE_US = {(32, 32): 0.117, (64, 32): 0.169, (64, 64): 0.275, (64, 128): 0.375, (128, 128): 0.497}
FP8_SPLIT_K_FACTORS = (2, 3, 4)


def get_split_k_fp8_config(m: int, n: int, k: int, num_cus: int) -> Optional[Tuple[int, int, int]]:
    """(BLOCK_M, BLOCK_N, SPLIT_K) when the plain FP8 GEMM should split K over SPLIT_K workgroups per tile, else None.

    A problem whose unsplit tiles fit the chip in one round is bound by what one compute unit can pull per k-tile
    (60-65 GB/s whatever the tile), and every workgroup pulls the activation rows of its tile over all of K. With K split,
    a larger tile on as many workgroups pulls fewer bytes per output; the price is a round trip of the partial sums
    through memory, paid by the part that arrives last. Modelled time of a plan: k-tiles per part x the tile's time per
    k-tile + 0.5 us + 12.5 ns per KB of partial sums the last part reads, never less than streaming the weights at 6 TB/s.
    A plan is taken when it fits one round (tile slots x SPLIT_K <= num_cus), leaves every part at least 14 k-tiles (24 when there are only two parts) and beats
    the unsplit pick (its own, slightly lower time per k-tile) by a tenth of its modelled time plus 3.5 us of launch. On 36 shapes (m = 32..256, n = 1536..24576,
    k = 1536..16384) swept with every tile and factor, weights cycling through more matrices than the caches hold, the
    plan taken is the fastest measured or within 1 % of it wherever one is taken (64 x 4096 x 7168: 64 x 64 tiles in four
    parts; 32 x 2112 x 7168: 32 x 32 in three); over 80 shapes with a plan (m = 17..1024, 13 (n, k)) it takes 0.47 to 1.04 of the
    unsplit time, median 0.83; k up to about 5000 in two parts, k = 2048 and n = 16384 or more stay unsplit.
    The weight-streaming kernel goes before a plan where
    `get_weight_stream_fp8_config` says so. Same rule as
    `pick_split_k` in yan_amd/csrc/yan_gemm_capi.hip (a CPU test keeps the two in step)."""
    if m <= 0 or n <= 0:
        return None
    k_tiles = k // 128
    unsplit = get_best_fp8_config(m, n, k, num_cus)
    if unsplit not in _FP8_SPLIT_K_TILE_US or ceil_div(m, unsplit[0]) * ceil_div(n, unsplit[1]) > num_cus:
        return None
    floor = n * k / 6.0e6
    base = max(k_tiles * _FP8_UNSPLIT_TILE_US[unsplit], floor)
    best, best_plan = None, None
    for (bm, bn), per_k_tile in _FP8_SPLIT_K_TILE_US.items():
        if bm > 32 and bm >= 2 * m:
            continue                # a tile more than twice as tall as the problem
        tiles = ceil_div(m, bm) * ceil_div(n, bn)
        for split in FP8_SPLIT_K_FACTORS:
            # a workgroup per part of every tile slot (tiles rounded up to the 8 XCDs); 256 also bounds the workspace
            # two parts save half the k-tiles at most: they pay from 24 k-tiles per part on, three and four from 14
            if ceil_div(tiles, 8) * 8 * split > min(num_cus, 256) or ceil_div(k_tiles, split) < (24 if split == 2 else 14):
                continue
            t = max(ceil_div(k_tiles, split) * per_k_tile + 0.5 + (split * bm * bn * 4) / 1024 * 0.0125, floor)
            if best is None or t < best:
                best, best_plan = t, (bm, bn, split)
    if best is not None and base - best >= 0.10 * (base + 3.5):
        return best_plan
    return None


# Split-K of the dense GEMM: microseconds per k-tile (64 deep) of a workgroup on a ring tile with the chip full (measured with
# weights cycling through more matrices than the caches hold), for every tile the unsplit pick can be; the first three are
# the tiles split-K plans use, with what their longer ring fill and larger partial sums add per launch.
_DENSE_SPLIT_K_TILE_US = {(64, 64): 0.248, (64, 128): 0.378, (128, 128): 0.51, (64, 192): 0.60, (128, 192): 0.80, (128, 256): 0.94,
                          (256, 128): 0.94}
_DENSE_SPLIT_K_EXTRA_US = {(64, 64): 0.0, (64, 128): 1.0, (128, 128): 2.5}
DENSE_SPLIT_K_FACTORS = (2, 3, 4, 6, 8)         # six and eight parts on 64 x 64 tiles only (few weight rows, long K)


def get_split_k_dense_config(m: int, n: int, k: int, num_cus: int) -> Optional[Tuple[int, int, int]]:
    """(BLOCK_M, BLOCK_N, SPLIT_K) when the dense 16-bit GEMM should split K over SPLIT_K workgroups per tile, else None.
    The rule of `get_split_k_fp8_config` with the dense tiles' numbers: the smallest dense tile holds 64 weight rows, so
    m = 64, n = 4096 puts 64 of 256 compute units to work and K = 7168 keeps each for 112 k-tiles; in four parts the same
    tiles fill the chip. A plan fits one round (tile slots x SPLIT_K <= num_cus), leaves every part at least 16 k-tiles and
    must beat the unsplit pick by 11 % of its modelled time plus 3.5 us. Measured (bf16, weights cycling, unsplit ->
    plan): 64 x 4096 x 7168 37.1 -> 16.2 us, 256 x 2048 x 7168 34.2 -> 20.3, 256 x 5120 x 5120 44.7 -> 33.9,
    64 x 2048 x 7168 36.1 -> 12.8 (six parts; four: 14.5), 64 x 1024 x 16384 69.3 -> 16.5 (eight parts; four: 24.1),
    256 x 7168 x 16384 113.4 -> 90.9, 512 x 4096 x 7168 53.4 -> 43.9 (hipBLASLt on the first five and the 256-row shapes: 22.7, 24.7, 49.6, 140.4);
    over 54 shapes swept with every tile and factor the plan is the fastest measured or within 6 % of it (11 % in one case),
    and over 118 shapes with a plan (m = 33..1024, 14 (n, k)) it takes 0.35 to 0.92 of the unsplit time, median 0.65. Same rule as
    `pick_dense_split_k` in yan_amd/csrc/yan_gemm_capi.hip (a CPU test keeps the two in step).
    The weight-streaming kernel goes before a plan where `get_weight_stream_dense_config` says so; below 8 rows, and up to 16
    on a K beyond 8192, there is no plan where that kernel fits."""
    if m <= 0 or n <= 0 or k <= 0 or ((m < 8 or (m <= 16 and k > 8192)) and get_skinny_dense_config(m, n, k, num_cus)):
        return None         # a handful of rows, or up to 16 on a long K: the one-atom weight-streaming kernel is as fast or faster
    k_tiles = ceil_div(k, 64)
    unsplit = get_best_dense_config(m, n, k, num_cus)
    if unsplit not in _DENSE_SPLIT_K_TILE_US or ceil_div(m, unsplit[0]) * ceil_div(n, unsplit[1]) > num_cus:
        return None
    floor = n * k * 2 / 6.0e6
    base = max(k_tiles * _DENSE_SPLIT_K_TILE_US[unsplit], floor)
    best, best_plan = None, None
    for (bm, bn), extra in _DENSE_SPLIT_K_EXTRA_US.items():
        if bm > 64 and bm >= 2 * m:
            continue                # a tile more than twice as tall as the problem
        tiles = ceil_div(m, bm) * ceil_div(n, bn)
        for split in DENSE_SPLIT_K_FACTORS:
            if split > 4 and (bm, bn) != (64, 64):
                continue            # the last part of a larger tile would hold more partial sums than it has registers for
            if ceil_div(tiles, 8) * 8 * split > min(num_cus, 256) or ceil_div(k_tiles, split) < 16:
                continue
            t = max(ceil_div(k_tiles, split) * _DENSE_SPLIT_K_TILE_US[(bm, bn)] + 0.5 + (split * bm * bn * 4) / 1024 * 0.0125 + extra, floor)
            if best is None or t < best:
                best, best_plan = t, (bm, bn, split)
    if best is not None and base - best >= 0.11 * (base + 3.5):
        return best_plan
    return None


# (BLOCK_M, BLOCK_N) -> cost per unit of tile area; tiles below 128 rows split K over their four waves.
_FLOAT_TILES = {(256, 256): 1.00, (128, 256): 1.015, (128, 128): 1.03, (128, 64): 1.04, (64, 64): 1.13, (32, 64): 1.13, (32, 32): 1.25}


def get_best_float_config(m: int, n: int, num_cus: int) -> Tuple[int, int]:
    """(BLOCK_M, BLOCK_N) of the fp32 GEMM: rounds of workgroups over the CUs times the tile's area times its cost
    per area; ties go to the earlier, larger tile. Same table and rule as `yan::pick_float_tile` in
    gemm/simple_gemm.hpp (a CPU test keeps the two in step)."""
    best, best_cost = None, None
    for (bm, bn), per_area in _FLOAT_TILES.items():
        tiles = ceil_div(m, bm) * ceil_div(n, bn)
        cost = ceil_div(tiles, num_cus) * bm * bn * per_area
        if best_cost is None or cost < best_cost:
            best, best_cost = (bm, bn), cost
    return best


# Split-K of the fp32 GEMM: microseconds a compute unit spends on 1024 k-rows of a tile under sustained load (measured with one
# and with two workgroups per unit, operands cycling: 82-92 % of the matrix rate). Plans use the first four.
_FLOAT_US_PER_1024_K = {(32, 32): 4.7, (32, 64): 8.7, (64, 64): 16.7, (128, 64): 33.1, (128, 128): 64.0, (128, 256): 122.0, (256, 256): 235.0}
_FLOAT_BLOCK_K = {(32, 32): 64, (32, 64): 64, (64, 64): 64, (128, 64): 32}
FLOAT_SPLIT_K_FACTORS = (2, 3, 4, 5, 6, 7, 8)


def get_split_k_float_config(m: int, n: int, k: int, num_cus: int) -> Optional[Tuple[int, int, int]]:
    """(BLOCK_M, BLOCK_N, SPLIT_K) when the fp32 GEMM should split K over SPLIT_K workgroups per tile, else None. The matrix cores
    bound this GEMM, so what splitting buys is an even share of the work: 128 x 2112 has 132 tiles of 32 x 64 for 256 compute
    units, and 462 parts of 64 x 64 tiles in seven are two almost full rounds. The parts of a tile run on one XCD, so a round is a
    part on each of the 32 units of the XCD that has most tiles: 50 tiles of 64 x 64 are 7 on seven XCDs and 1 on the last,
    35 parts in five, two rounds (640 x 320 x 7168: 49 us that way, 38 unsplit). Modelled time of a plan: rounds x (the tile's
    time for its k-rows + 1 us) + 5 us (launch, first copies, the meeting) + 12.5 ns per KB of partial sums the last part reads;
    taken when it is below 0.92 of the unsplit pick's and 1.2 us, the longer way through the entry, below it. Measured (unsplit ->
    plan, operands cycling): 128 x 2112 x 7168 58 -> 45 us, 256 x 2112 x 7168 93 -> 75, 128 x 256 x 8192 36 -> 12; 264 shapes that
    split 0.32 to 0.99 times the unsplit time, 0.78 on average."""
    if m <= 0 or n <= 0 or k <= 0:
        return None
    tile = get_best_float_config(m, n, num_cus)
    base = ceil_div(ceil_div(m, tile[0]) * ceil_div(n, tile[1]), num_cus) * _FLOAT_US_PER_1024_K[tile] * k / 1024 + 3.5
    best, best_plan = min(0.92 * base, base - 1.2), None
    for (bm, bn), block_k in _FLOAT_BLOCK_K.items():
        tiles, k_tiles = ceil_div(m, bm) * ceil_div(n, bn), ceil_div(k, block_k)
        slots = ceil_div(tiles, 8) * 8
        for split in FLOAT_SPLIT_K_FACTORS:
            # 16 MB of partial sums, four counters per tile slot in 16 KB, at least 256 k-rows per part
            part = ceil_div(k_tiles, split) * block_k
            if slots * split * bm * bn * 4 > 1 << 24 or slots > 1024 or part < 256:
                continue
            rounds = ceil_div(slots // 8 * split, max(num_cus // 8, 1))
            t = rounds * (_FLOAT_US_PER_1024_K[(bm, bn)] * part / 1024 + 1) + 5 + split * bm * bn * 4 / 1024 * 0.0125
            if t < best:
                best, best_plan = t, (bm, bn, split)
    return best_plan


# The fp32 GEMM on the bf16 matrix cores (gemm/simple_gemm_bf16x3.hpp): depth of a k-tile (16 for each of the waves that share K), microseconds
# per k-tile while few compute units work, microseconds a tile costs besides (first copies, sums of its waves, epilogue). Fitted, with the rest of the model below, to
# 190 shapes with every tile and split forced in turn, operands cycling: its pick takes 1.015 of the fastest's time on average, 1.13 at
# worst above the limit.
_FLOAT_BF16X3_TILES = {(256, 256): (16, 1.16, 9.8), (256, 128): (32, 1.15, 7.0), (128, 256): (32, 1.17, 6.8), (128, 128): (64, 1.18, 6.9),
                       (128, 64): (64, 0.69, 4.9)}
FLOAT_BF16X3_SPLIT_FACTORS = (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 15)
# m * n * k from which it is the faster one: above it 78 shapes took 0.50 to 1.00 of the fp32 matrix cores' time (0.72 on average), below
# 5e8 it loses nearly everywhere (640 x 320 x 1153 9.3 against 13.9 us), in between it goes either way.
FLOAT_BF16X3_MIN_MNK = 1 << 30


def get_float_bf16x3_config(m: int, n: int, k: int, num_cus: int, may_split: bool = True) -> Optional[Tuple[int, int, int]]:
    """(BLOCK_M, BLOCK_N, SPLIT_K) when the fp32 GEMM should run on the bf16 matrix cores, else None. Modelled time: rounds x (k-tiles of a
    part x the tile's time per k-tile, twice that where every compute unit works (the power limit) + the tile's other costs) + 1.5 us, and
    for a split 1.8 us + 13 ns per KB of partial sums the last part reads.

    The rounding of a sum grows with the products added up in a row. Sixteen of them are six roundings here and eight on the fp32 cores, so K is
    cut at least as often as the plan there cuts it, by waves that share it (tiles below 128 rows: four) and by parts: against 64 bits the
    error is then 0.80 to 0.90 of that plan's (all positive operands 0.66 to 0.99), over 158 shapes where the fastest plan cuts it less often and
    is 1.07 to 1.73 (1.02 to 2.90) times as far off. What that costs (fp32 cores, fastest plan, this one): 3200 x 4096 x 995 204.5, 132.3, 155.8 us,
    2048 x 3200 x 866 93.5, 60.9, 66.4, 1920 x 2368 x 318 31.7, 24.3, 31.3; 0.60 to 1.03 of the fp32 cores' time, 0.77 on average."""
    if m * n * k < FLOAT_BF16X3_MIN_MNK:
        return None
    on_fp32 = (may_split and get_split_k_float_config(m, n, k, num_cus)) or (*get_best_float_config(m, n, num_cus), 1)
    fp32_ways = on_fp32[2] * (4 if on_fp32[0] < 128 else 1)
    best, plan = None, None
    for (bm, bn), (block_k, per_k_tile, per_tile) in _FLOAT_BF16X3_TILES.items():
        tiles, k_tiles = ceil_div(m, bm) * ceil_div(n, bn), ceil_div(k, block_k)
        for split in FLOAT_BF16X3_SPLIT_FACTORS if may_split else (1,):
            if split * (block_k // 16) < fp32_ways:
                continue
            # 16 MB of partial sums, eight counters per tile in 16 KB, two k-tiles per part
            if split > 1 and (tiles * split * bm * bn * 4 > 1 << 24 or tiles > 512 or ceil_div(k_tiles, split) < 2):
                continue
            rounds = ceil_div(tiles * split, num_cus)
            busy = tiles * split / (num_cus * rounds)
            t = 1.5 + rounds * (ceil_div(k_tiles, split) * per_k_tile * (1 + busy) + per_tile)
            if split > 1:
                t += 1.8 + split * bm * bn * 4 / 1024 * 0.0133
            if best is None or t < best:
                best, plan = t, (bm, bn, split)
    return plan
