"""
Analytical ranking of kernel configurations (larger score = expected faster).

Same entry points as the reference's src/cost_model/CostModel.py
(`rank_rowwise_configs` :280, `rank_gemm_configs` :274, `rank_fa_configs` :96
and the `*_score` / `*_occupancy` helpers); the terms are re-derived for a
CDNA4 compute unit.  Only the ordering of the top-N matters: measurement picks
the winner.
"""

from __future__ import annotations

import math
from dataclasses import replace

from deca_amd.driver.driver import cu_occupancy


class CostModel:
    """Kept for interface compatibility (reference: CostModel.py:7-12 is an empty stub)."""

    def cost(self, kernel, arch, compute_pattern):
        raise NotImplementedError("use the rank_* functions of this module")


def _wave_efficiency(grid: int, slots: int) -> float:
    """Useful share of the launch's workgroup waves: the tail of the last wave idles."""
    waves = math.ceil(grid / slots)
    return grid / (waves * slots)


# ---------------------------------------------------------------------------
# row-wise
# ---------------------------------------------------------------------------
def rowwise_occupancy(cfg, arch, op: str, N: int) -> int:
    """Resident workgroups per CU of a row-wise (Softmax / RMSNorm) config."""
    from deca_amd.kernels.rowwise_hip import regs_per_thread

    lds = 0 if cfg.threads_per_row <= arch.warp_size else 8 * cfg.threads // arch.warp_size
    wgs, _ = cu_occupancy(arch, regs_per_thread(cfg, N, op), lds, cfg.threads)
    return max(int(wgs), 1)


def rowwise_score(cfg, arch, op: str, M: int, N: int, type_size: int = 2) -> float:
    """
    Heuristic score of a memory-bound row-wise config.

    - memory parallelism: bytes of loads in flight per CU (every chunk of the
      row is requested up front in `reg` mode, `unroll` chunks in `twopass`)
      against Little's law, HBM bandwidth per CU x latency under load
      (`arch.dram_latency_s`)
    - granularity: a wave can only start reducing once all of its chunks have
      arrived and stores nothing until the row is reduced, so long per-lane chunk
      lists (few lanes per row) serialise load, math and store inside each wave;
      measured on MI355X the sweet spot is two 16-byte chunks per lane
    - wave efficiency of the grid of M / rows_per_block workgroups, and the
      drain bubble of large workgroups (all waves of a workgroup retire
      together, so 1024-lane workgroups leave wave slots idle at their tails)
    - twopass re-reads the row; the re-read hits L2 / Infinity Cache when the
      rows in flight fit
    - rows spanning several waves pay an LDS exchange and a barrier per reduction
    - idle vector lanes of the last chunk (tail) and 8-byte accesses
    - non-temporal accesses: streamed data does not displace lines in L2 /
      Infinity Cache and the writes drain earlier (measured: ~8% on MI355X)
    """
    from deca_amd.kernels.rowwise_hip import ONLINE_MIN_N, num_chunks, use_lines, use_online

    wgs = rowwise_occupancy(cfg, arch, op, N)
    chunks = num_chunks(cfg, N)
    depth = chunks if cfg.mode == "reg" else cfg.unroll
    grid = M // cfg.rows_per_block
    # Every row resident at once: all loads are under way from the start and no round waits for
    # another.  What counts then is the CU with the most rows and the number of waves on a CU: nine to
    # twelve, with 64 lanes a row or more as that takes (1341 x 10744: 10.5 us with 5 waves a CU, 10.6
    # with 10, 11.5 with 21, 11.9 with 42; 780 x 14432: 9.8, 9.0, 8.8 and 10.1 with 3, 6, 12 and 24; more
    # waves meet in a reduction, fewer leave a SIMD idle).  59 shapes of 45 to 300 KiB per CU: mean
    # distance to the best 2.3 % (2.9 % in the caches) against 5.2 and 7.4 % by the terms below; longer
    # softmax rows, whose waves have twice the arithmetic of RMSNorm, gain nothing beyond 140 KiB.
    # Both ends of a half-vector row are the one wave's to patch where a wave has it to itself: 4 %,
    # which decides where two waves are that near (17 of 60 shapes on which a price of 10 % would: they are
    # level there, 2 % ahead in the caches, 1787 x 7260 9.0 against 10.1 us; with 10 % the 60 are 4 %
    # slower on the average).
    rows_per_cu = M / arch.sm_nums
    kib_per_cu = rows_per_cu * N * type_size / 1024
    one_round = (cfg.mode == "reg" and cfg.threads_per_row >= arch.warp_size
                 and cfg.vec * type_size >= 16 and depth <= 20 and grid <= arch.sm_nums * wgs
                 and 45 <= kib_per_cu <= (140 if op == "softmax" else 210))
    if one_round:
        wgs = max(1, math.ceil(grid / arch.sm_nums))
    in_flight = wgs * cfg.threads * depth * cfg.vec * type_size
    need = arch.dram_bw * 1e9 / arch.sm_nums * getattr(arch, "dram_latency_s", 2e-6)
    mem = min(1.0, in_flight / need)

    # (the loss levels off: 16 and 32 chunks per lane measure the same, 0.88 of the best)
    granularity = 1.0 / (1.0 + 0.012 * min(max(0, depth - 2), 11)) * (0.985 if depth == 1 else 1.0)

    wave_eff = _wave_efficiency(grid, arch.sm_nums * wgs)
    drain = 1.0 / (1.0 + 0.10 * max(0.0, cfg.threads / 256 - 2.0))
    rows = 1.0 / (1.0 + 0.015 * abs(math.log2(cfg.rows_per_block) - 1.0))

    passes = 1.0
    if cfg.mode == "twopass":
        footprint = arch.sm_nums * wgs * cfg.rows_per_block * N * type_size
        cache = arch.l2_bytes + getattr(arch, "mall_bytes", 0)
        hit = min(1.0, (0.8 if cfg.hint else 0.5) * cache / footprint)
        reread_bw = getattr(arch, "mall_bw", arch.l2_bw)
        passes = 1.0 + 0.5 * (hit * arch.dram_bw / reread_bw + (1.0 - hit))

    waves_per_row = max(1, cfg.threads_per_row // arch.warp_size)
    reduce = 1.0 / (1.0 + 0.005 * math.log2(waves_per_row))
    if cfg.threads_per_row < arch.warp_size:
        reduce *= 0.97
    if one_round:
        granularity = drain = 1.0
        wave_eff = math.sqrt(rows_per_cu / (math.ceil(grid / arch.sm_nums) * cfg.rows_per_block))
        rows = 1.0 / (1.0 + 0.015 * math.log2(cfg.rows_per_block))
        waves_per_cu = rows_per_cu * waves_per_row
        # (one wave a row is no more than its due where there are more rows: priced against 10.5 waves,
        # 8-byte accesses and two waves a row came first on 65 of 4983 shapes, nearly all of 29 to 32
        # rows per CU, and took 3.8 % longer on the average, 7.6 % in the caches)
        reduce = 1.0 / (1.0 + 0.07 * abs(math.log2(waves_per_cu / max(10.5, rows_per_cu))))
        if cfg.half and waves_per_row == 1 and use_lines(cfg, M, N, op):
            reduce *= 0.96
    online = use_online(cfg, N, op)
    if online:
        # The first pass is done when the last chunk arrives: what lengthens the others' series of
        # load, math and store, and what their large workgroups idle at the end, is not there.
        granularity = drain = 1.0
        # 1024 lanes have half as much of a row to work on behind its last chunk as 512: 1-11 % ahead
        # on 33 of 47 shapes, up to 6 % behind on the others (mean distance to the better 0.8 and
        # 2.8 %); how many workgroups a CU has room for does not tell which.
        reduce = 1.0 if cfg.threads_per_row == 1024 else 0.98

    tail = N / (chunks * cfg.threads_per_row * cfg.vec) if cfg.mode == "reg" else 1.0
    lanes = 1.0 if cfg.vec * type_size >= 16 else 0.985
    # Rows of an odd multiple of 8 bytes have forms with 16-byte accesses (`half`).  Level with 8-byte
    # ones in small grids.  With 42 (softmax: 52) to 75 KiB per CU 1.00-1.32x on 37 of 39 shapes of 770
    # to 18K elements (RMSNorm bf16 1822 x 4628: 9.4 and 7.1 us), 1 % behind on two.  Beyond that
    # 1.02-1.26x on 49 of 49 from these lengths on, but 1-3 % behind on shorter RMSNorm rows, and 2-11 %
    # on 7 of 7 of the length where they come to a few chunks of few lanes.
    if N % 8 == 4 and lanes < 1.0:
        softmax = op == "softmax"
        if kib_per_cu <= 75:
            ahead = kib_per_cu >= (52 if softmax else 42) and N >= 700
        else:
            ahead = N >= (4100 if softmax else 3400) and not (5200 if softmax else 6900) < N < 7900
        if ahead:
            lanes = 0.93
    # Softmax rows of the online form's lengths: its 16-byte accesses are 1.04-1.57x ahead of 8-byte
    # ones on 76 of 76 shapes of 1 to 6 rows per CU (of which those may fit a CU one more).
    if op == "softmax" and N >= ONLINE_MIN_N and cfg.mode == "reg" and cfg.vec * type_size < 16:
        lanes = 0.75
    # A workgroup that has a long row to itself leaves a CU room for two or three others, one with
    # two such rows for none (36K ... 55K elements: 10-37 % behind one row of 256 lanes on 13 of 13
    # shapes), nor do 1024 lanes (33K ... 50K: 2-42 % behind on 20 of 20; with up to 4.5 rows per CU
    # 4-42 % on 24 of 26 from 8.6K to 21K).
    if cfg.rows_per_block > 1 and N > 32768:
        rows *= 0.85
    if not online:
        if cfg.threads_per_row == 1024 and (33000 < N < 50000 or (rows_per_cu <= 4.5 and 8600 < N < 21000)):
            drain *= 0.88
    stream = 1.0 if cfg.hint else getattr(arch, "rowwise_no_hint_factor", 0.92)

    return (mem * granularity * wave_eff * drain * rows * reduce * (0.7 + 0.3 * tail) * lanes *
            stream / passes)


def rank_rowwise_configs(configs, arch, op: str, M: int, N: int, top_n: int | None = None):
    """Sort row-wise configs by `rowwise_score` (best first)."""
    ranked = sorted(configs, key=lambda c: rowwise_score(c, arch, op, M, N), reverse=True)
    return ranked[:top_n] if top_n else ranked


# ---------------------------------------------------------------------------
# FP16 MFMA GEMM
# ---------------------------------------------------------------------------
def gemm_tc_occupancy(cfg, arch) -> int:
    """Resident workgroups per CU of an FP16 MFMA GEMM config."""
    from deca_amd.kernels.gemm_hip import est_regs_per_thread, smem_bytes

    wgs, _ = cu_occupancy(arch, est_regs_per_thread(cfg), smem_bytes(cfg), cfg.threads)
    return max(int(wgs), 1)


def gemm_wave_dram_bytes_per_flop(cfg, arch, M: int, N: int, K: int, slots: int) -> float:
    """HBM bytes per FLOP of A / B (fp16) for one wave of `slots` concurrent
    workgroups.  With grouped rasterisation a wave covers `rows` workgroup rows
    x `cols` columns; every A row block and B column block of the wave is
    fetched once.  Operands that fit comfortably in the Infinity Cache are
    fetched once overall (reference: CostModel.py:182-196, with L2 -> MALL)."""
    cache = getattr(arch, "mall_bytes", arch.l2_bytes)
    if (M * K + K * N) * 2 <= 0.5 * cache:
        return (M * K + K * N) * 2 / (2.0 * M * N * K)
    from deca_amd.kernels.gemm_hip import tile_grid

    GM, GN = tile_grid(cfg, M, N)
    if cfg.raster == 0:  # the tiles in flight form 16 x 16 blocks
        blocks = max(1, math.ceil(min(slots, GM * GN) / 256))
        return blocks * 16 * (cfg.BM + cfg.BN) / (min(slots, GM * GN) * cfg.BM * cfg.BN)
    g = cfg.raster
    cols = min(GN, math.ceil(slots / g))
    rows = min(GM, g * math.ceil(slots / (g * GN)))
    tiles = min(slots, GM * GN)
    return (rows * cfg.BM + cols * cfg.BN) / (tiles * cfg.BM * cfg.BN)


def gemm_mma_peak(cfg, arch) -> float:
    """MFMA peak (GFLOPS) with fp32 accumulation, the only mode of the matrix cores."""
    return arch.peak_mma_sync_flops


# Step times of the tile bodies (16x16x32 tiles, accumulators in AGPRs where they fit, load
# window): (BM, BN, BK, warp_m, warp_n, stages, kgroups) -> microseconds of (a workgroup's
# prologue and epilogue, one K-tile of a workgroup alone on its CU, one K-tile of each of two on
# a CU; None where the LDS ring leaves room for one only).  Fitted to the times of seven shapes
# that are multiples of 64 and of little else (M 704 ... 4800, N 640 ... 7360, K 512 ... 5440),
# within 10 % there; those of the wave groups (kgroups = 2) to 1024^3 and 256 x 4096 x 4096 (the
# 64 x 64 tile) and to what the other two gain over the plain tile of their size on 22 shapes of
# up to one tile per CU (K 512 ... 1024: -3 ... +5 %, 1280 ... 7936: 2-11 %).
# What they show is the CU's load path and the fabric behind its L2 rather than the matrix pipe:
# 32 KiB per 128 x 128 K-tile at 70 KB/us and CU.
GEMM_STEP_TIMES = {
    (256, 256, 64, 128, 64, 2, 1): (6.0, 1.154, None),
    (256, 128, 64, 64, 64, 3, 1): (2.6, 0.776, None),
    (128, 256, 64, 64, 64, 3, 1): (2.7, 0.757, None),
    (128, 128, 64, 64, 32, 3, 1): (1.3, 0.476, None),
    (128, 64, 64, 64, 32, 3, 1): (1.0, 0.304, 0.594),
    (64, 128, 64, 64, 32, 3, 1): (1.0, 0.301, 0.597),
    (64, 64, 64, 32, 32, 5, 1): (1.0, 0.225, 0.390),
    (128, 64, 128, 64, 32, 3, 2): (1.4, 0.558, None),
    (64, 128, 128, 64, 32, 3, 2): (1.4, 0.556, None),
    (64, 64, 128, 64, 32, 3, 2): (1.0, 0.410, None),
}


def gemm_edge_score(cfg, arch, M: int, N: int, K: int) -> float | None:
    """Score of a config by the step times of its tile body: useful share of the matrix peak in
    the time that `GEMM_STEP_TIMES` gives it.  None for a body without an entry."""
    from deca_amd.kernels.gemm_hip import tile_grid

    times = GEMM_STEP_TIMES.get((cfg.BM, cfg.BN, cfg.BK, cfg.warp_m, cfg.warp_n, cfg.stages,
                                 cfg.kgroups))
    if times is None or cfg.mfma != 16:
        return None
    fixed, one, two = times
    rows, cols = tile_grid(cfg, M, N)
    wgs = min(2, gemm_tc_occupancy(cfg, arch))
    full, rest = divmod(rows * cols, arch.sm_nums * wgs)
    t = 1.5 + full * (fixed + K // cfg.BK * (one if wgs == 1 else two))
    if rest:
        t += fixed + K // cfg.BK * (one if rest <= arch.sm_nums else two)
    # between the orders of one tile: operand panels that an XCD's tiles fetch
    per_xcd = min(rows * cols, arch.sm_nums * wgs) / getattr(arch, "num_xcd", 8)
    band = min(cfg.raster or 8, per_xcd)
    panels = band * cfg.BM + math.ceil(per_xcd / band) * cfg.BN
    t *= 1.0 + 1e-5 * panels
    return 2.0 * M * N * K / (arch.peak_mma_sync_flops * 1e3 * t)


def gemm_measured_form(cfg):
    """The config of `cfg`'s tile body and order that `GEMM_STEP_TIMES` was measured with, None
    for a body without an entry."""
    from deca_amd.kernels.gemm_hip import agpr_split_fits, default_spread

    if getattr(cfg, "mfma", 32) != 16 or not cfg.direct:
        return None
    for bm, bn, bk, wm, wn, stages, kgroups in GEMM_STEP_TIMES:
        if (bm, bn, bk, wm, wn, kgroups) == (cfg.BM, cfg.BN, cfg.BK, cfg.warp_m, cfg.warp_n,
                                             cfg.kgroups):
            twin = replace(cfg, stages=stages, tail=False, epi_smem=True, xcd=True, edge=True,
                           early=wm // 32 if wm >= 64 else 0, agpr=False, spread=0)
            return replace(twin, agpr=agpr_split_fits(twin), spread=default_spread(twin))
    return None


def gemm_form_factor(cfg) -> float:
    """What the form of a tile's loop is worth beside the terms of `gemm_general_score`."""
    # 16x16x32 tiles: measured ahead of the 32x32x16 twin where the grid is a single wave of
    # workgroups or leaves a partial one (2048^3 +7 %, 4096^3 +4.5 %, 6144^3 / 10240^3 +2 %),
    # level with it on the large grids; the barrier inside the last k-step adds a little
    form = 1.0
    if getattr(cfg, "mfma", 32) == 16:
        form = 1.02 + (0.004 if getattr(cfg, "early", 0) else 0.0)
        # accumulators in accumulation registers: about 3 % over the builtin form (measured
        # at 4096^3 and 8192^3)
        if getattr(cfg, "agpr", False):
            form += 0.03
        # tile loads dealt over the MFMA groups: the more loads a wave issues per K-tile, the
        # longer the queue at the load path that the burst form makes every wave stand in
        # (measured with 8 loads per lane and K-tile: +2 % at 4096^3, +6 % at 8192^3, +7.5 %
        # at 16384^3; with 4: +1 %)
        if getattr(cfg, "spread", 0):
            loads = (cfg.BM * cfg.BK + cfg.BK * cfg.BN) // 8 // cfg.threads
            form += 0.005 * loads
    return form


def gemm_general_score(cfg, arch, M: int, N: int, K: int) -> float:
    """
    Heuristic score of an FP16 MFMA GEMM config, by its terms (`gemm_tc_score` puts measured
    step times in their place where it has them).

    Per-CU time per FLOP of the main loop, as a roofline whose non-bottleneck
    terms only partially overlap:
    - matrix cores (MFMA 32x32x16, fp32 accumulation)
    - LDS: every wave reads (WM + WN) * 16 * 2 bytes per k16 step for
      2 * WM * WN * 16 FLOPs, and the workgroup fills (BM + BN) * BK * 2 bytes
      per stage (through the LDS write port unless the loads are direct)
    - L2: every workgroup streams its A rows and B columns,
      (BM + BN) / (BM * BN) B/FLOP, from the L2 of its XCD; without the XCD remap
      neighbouring tiles land on different XCDs and share nothing there
    - HBM / Infinity Cache: the unique A / B blocks of one wave of workgroups
    - fabric: the A / B blocks that the tiles in flight on one XCD miss in its L2
    Then:
    - wave efficiency of the workgroup grid
    - issue: with one wave per SIMD nothing covers that wave's own waits (LDS
      latency before the first MFMA of a k-step, the barrier); a second wave does
    - pipelining: bytes in flight ((stages - 1) tiles per workgroup, or one tile
      for the VGPR-staged ring) vs. Little's law on the L2 stream; excess
      stages are penalised by `arch.gemm_excess_stage_penalty` (fitted on MI355X:
      a window of one 64-deep tile already saturates; deeper rings cost ~2% each)
    - one barrier per BK stage
    - epilogue: C is written once; direct stores are 8-byte row segments, the
      staged epilogue writes 16-byte coalesced chunks
    """
    from deca_amd.kernels.gemm_hip import tile_grid

    wgs = gemm_tc_occupancy(cfg, arch)
    slots = arch.sm_nums * wgs
    rows, cols = tile_grid(cfg, M, N)
    grid = rows * cols
    wave_eff = _wave_efficiency(grid, slots)
    if getattr(cfg, "tail", False):
        # the partial last wave runs as quarter tiles: a quarter of the work each, at the
        # lower efficiency of the small tile (measured ~0.3 of a full tile's time)
        from deca_amd.kernels.gemm_hip import tail_tiles

        r = tail_tiles(cfg, M, N)
        wave_eff = (grid / slots) / ((grid - r) / slots + math.ceil(4 * r / slots) * 0.32)
    waves_per_simd = wgs * cfg.num_warps / arch.simds_per_cu
    hiding = min(1.0, 0.82 + 0.09 * min(waves_per_simd, 2.0)) if waves_per_simd >= 1 else \
        0.82 * waves_per_simd

    cus = arch.sm_nums
    wm, wn = cfg.warp_m, cfg.warp_n
    peak = gemm_mma_peak(cfg, arch)
    t_mma = cus / (peak * 1e9)
    fill_bpf = (cfg.BM + cfg.BN) / (cfg.BM * cfg.BN)
    lds_bpf = (wm + wn) / (wm * wn) + (0.0 if cfg.direct else fill_bpf)
    t_lds = lds_bpf / arch.smem_bw_per_sm
    l2_bpf = fill_bpf * (1.0 if cfg.xcd else 1.5)
    t_l2 = l2_bpf * cus / (arch.l2_bw * 1e9)
    dram_bpf = gemm_wave_dram_bytes_per_flop(cfg, arch, M, N, K, slots)
    t_dram = dram_bpf * cus / (arch.dram_bw * 1e9)
    # L2 misses: what the tiles in flight on ONE XCD need from the fabric.  A banded order
    # gives an XCD `raster` rows of tiles, the block order 8 rows by 4 columns per resident
    # workgroup; an order that is not XCD-aware leaves neighbours on different L2s.
    per_xcd = max(1, slots // getattr(arch, "num_xcd", 8))
    if not cfg.xcd:
        rows_x, cols_x = per_xcd, per_xcd
    elif cfg.raster == 0:
        rows_x, cols_x = 8, max(1, per_xcd // 8)
    else:
        rows_x = min(cfg.raster, per_xcd)
        cols_x = min(cols, math.ceil(per_xcd / rows_x))
    fabric_bpf = (rows_x * cfg.BM + cols_x * cfg.BN) / (per_xcd * cfg.BM * cfg.BN)
    t_fabric = fabric_bpf * cus / (getattr(arch, "mall_bw", arch.l2_bw) * 1e9)
    terms = sorted([t_mma, t_lds, t_l2, t_dram, t_fabric])
    t_flop = terms[-1] + 0.25 * sum(terms[:-1])

    # Bytes per CU that must be in flight to cover the L2 / fabric latency at the
    # sustained (power-limited, about half of peak) MFMA rate: ~0.75 us at peak rate.
    need = fill_bpf / t_mma * getattr(arch, "gemm_fill_latency_s", 0.75e-6)
    stage_bytes = wgs * (cfg.BM + cfg.BN) * cfg.BK * 2
    depth = (cfg.stages - 1) if cfg.direct else 1
    in_flight = max(depth, 0.5) * stage_bytes
    pipe = min(1.0, in_flight / need) ** 0.5
    excess = max(0, depth - math.ceil(need / stage_bytes))
    pipe *= 1.0 - getattr(arch, "gemm_excess_stage_penalty", 0.0) * excess

    # CU cycles per stage at the MFMA rate vs. ~100 cycles of barrier + refill issue
    flops_per_cycle = peak * 1e9 / cus / arch.sm_clock_hz
    stage_cycles = 2 * cfg.BM * cfg.BN * cfg.BK / flops_per_cycle
    sync_eff = 1.0 / (1.0 + 100.0 / wgs / stage_cycles)

    epi_eff = 1.0 if cfg.epi_smem else 0.5
    t_epi = (1.0 / K) / epi_eff * cus / (arch.dram_bw * 1e9)
    t_epi *= 1.0 if wgs == 1 else 0.4

    # VGPR-staged fills add global-load, LDS-write and wait instructions to the
    # MFMA issue stream (measured ~15% on MI355X)
    staged = 1.0 if cfg.direct else getattr(arch, "gemm_staged_fill_factor", 0.85)

    form = gemm_form_factor(cfg)
    # (tiles that reach over the edge of C compute more than the shape needs)
    useful = M * N / (grid * cfg.BM * cfg.BN)
    return useful * form * wave_eff * hiding * pipe * sync_eff * staged / ((t_flop + t_epi) / t_mma)


def gemm_step_times_apply(arch, M: int, N: int) -> bool:
    """Shapes whose tile bodies are ranked by `GEMM_STEP_TIMES`: no multiple of 256 both ways,
    or fewer tiles of 256 x 256 than there are CUs."""
    return bool(M % 256 or N % 256 or M * N < 256 * 256 * arch.sm_nums)


def gemm_tc_score(cfg, arch, M: int, N: int, K: int) -> float:
    """Score of an FP16 MFMA GEMM config, larger is faster.

    Where the step times apply, a tile body that has them scores by them whether or not it is
    an `edge` form (the two are the same code where the tile divides C).  Its forms that were
    not measured over the range stand to the measured one as in `gemm_general_score`, another
    ring depth at most level with it (128 x 128 x 64 on 14 shapes: 4 stages 0-8 % behind 3, 5
    stages 0-10 %, where the general score has them up to 22 and 33 % ahead).  All other bodies
    stay on the general score, which reads about a quarter lower: of 175 shapes on which one of
    them came first by it, the measured bodies were level or ahead on 168."""
    edge = getattr(cfg, "edge", False)
    if not (edge or gemm_step_times_apply(arch, M, N)):
        return gemm_general_score(cfg, arch, M, N, K)
    by_steps = gemm_edge_score(cfg, arch, M, N, K) if edge else None
    if by_steps is not None:
        return by_steps
    twin = gemm_measured_form(cfg)
    if twin is None:
        return gemm_general_score(cfg, arch, M, N, K)

    def rest(c):
        return gemm_general_score(c, arch, M, N, K) / gemm_form_factor(c)

    whole = replace(cfg, tail=False)
    ring = replace(whole, stages=twin.stages)
    ratio = (gemm_form_factor(cfg) / gemm_form_factor(twin) * (rest(ring) / rest(twin))
             * min(1.0, rest(whole) / rest(ring)) * (rest(cfg) / rest(whole)))
    return gemm_edge_score(twin, arch, M, N, K) * ratio


def rank_gemm_configs(configs, arch, M: int, N: int, K: int, top_n: int | None = None,
                      per_tile: int | None = None):
    """Sort FP16 MFMA GEMM configs by `gemm_tc_score` (best first).

    `per_tile` keeps only that many tile orders (`raster`, and barrier positions `early`) of each tile set: the orders of
    one tile set score within a percent or two of each other, so that a plain top-N would
    be spent on the six orders of the one or two best tile sets."""
    ranked = sorted(configs, key=lambda c: gemm_tc_score(c, arch, M, N, K), reverse=True)
    if per_tile:
        seen, kept = {}, []
        for c in ranked:
            key = replace(c, raster=1, early=0, agpr=False, spread=0)
            seen[key] = seen.get(key, 0) + 1
            if seen[key] <= per_tile:
                kept.append(c)
        ranked = kept
    return ranked[:top_n] if top_n else ranked


# ---------------------------------------------------------------------------
# FlashAttention forward
# ---------------------------------------------------------------------------
_FA_HIDDEN = 0.0  # share of a workgroup's start-up latency still exposed beside a second workgroup


def fa_occupancy(cfg, arch, D: int, grid: int):
    """Returns (resident workgroups per CU, share of the wave slots in use)."""
    from deca_amd.kernels.flash_attn_hip import est_regs_per_thread, smem_bytes

    wgs, _ = cu_occupancy(arch, est_regs_per_thread(cfg, D), smem_bytes(cfg, D), cfg.threads)
    wgs = max(int(wgs), 1)
    return wgs, wgs * cfg.num_warps / arch.max_resident_warps_per_sm


def fa_split_score(cfg, arch, shape, causal: bool = False) -> float:
    """Score of a config whose waves share the query rows and split the keys (`kv_split`), on
    the scale of `fa_score` (useful share of the matrix peak).

    Its time is modelled directly: a fixed part per workgroup (Q, the first tiles, the meeting
    of the waves in LDS) and a number of key steps per wave whose length grows with the waves
    that share a SIMD.  Fitted on twelve shapes of 256 ... 2048 rows of 32 queries (S = 512 ...
    16384, D = 64 and 128, full and causal), where it is within 10 % of the measured time of
    these forms.  `fa_score` overestimates the plain forms on such small grids, more so under
    the causal mask (their measured times are 1.05x and 1.35x its own at the median), hence
    the last factor."""
    B, H, S_q, S_kv, D = shape
    grid = (S_q // cfg.Br) * B * H
    wgs, _ = fa_occupancy(cfg, arch, D, grid)
    per_cu = min(wgs, math.ceil(grid / arch.sm_nums))

    def key_step(workgroups):
        waves = max(1.0, workgroups * cfg.num_warps / arch.simds_per_cu)
        # a second slot per wave pays while a tile is small (D = 64: -7 %; D = 128: +7 %)
        slots = 1.0 if cfg.stages == 1 else (0.93 if cfg.Bc * D <= 32 * 64 else 1.07)
        return (0.25e-6 + 0.65e-6 * waves * (cfg.Br // 32)) * (cfg.Bc / 32) * (D / 128) * slots

    step = key_step(per_cu)
    fixed, launch = 3.3e-6, 1.5e-6  # per workgroup; of the first one, what every launch costs
    steps = math.ceil(S_kv / (cfg.Bc * cfg.num_warps))
    longest = fixed + steps * step
    rounds = grid / (arch.sm_nums * wgs)
    if causal:
        # (the longest workgroups start first and are alone on their CU towards the end)
        longest = fixed + steps * 0.5 * (step + key_step(1))
        mean = fixed + (S_kv / 2 + cfg.Br / 2) / (cfg.Bc * cfg.num_warps) * step
        t = max(longest, rounds * mean)
    else:
        # (1.2: of 1.0 to 1.3 the factor that leaves the fewest slower choices over the shapes
        # below; at 1.0 there are two more)
        t = math.ceil(rounds) * longest * (1.2 if rounds > 1 else 1.0)
    # From two rows of 32 queries per CU on the plain forms fill their SIMDs too: under the causal
    # mask, whose rows differ in length, the more of them the better they do; without it the
    # fewer keys there are, the more the meeting of the waves weighs.  Of 419 shapes (1 to 8 rows
    # per CU, S_kv 256 ... 13504) 36 took up to 16 % longer than in the plain form without these
    # two terms, most of them full ones with few keys and D 64 (B3 H16 S 384: 8.2 us instead of
    # 7.1); with them 13, all but one by less than 10 %.  (The rows term on full shapes: 18 %
    # lost on B1 H16 S_q 2624 S_kv 3776 D 64, nothing won.)
    rows = B * H * S_q / 32 / arch.sm_nums
    gain = 1.0
    if causal:
        gain = max(1.0, rows / 2) ** -0.15
    elif rows >= 2:
        gain = min(1.0, S_kv * D / (1024 * 64)) ** 0.3
    flops = 4.0 * B * H * S_q * S_kv * D * (0.5 if causal else 1.0)
    return gain * flops / (arch.peak_mma_sync_flops * 1e9) / ((t - launch) * (0.8 if causal else 0.95))


def fa_score(cfg, arch, shape, causal: bool = False) -> float:
    """
    Heuristic score of a FlashAttention config.

    - roofline of one CU per FLOP: matrix-core time vs. LDS time (every wave
      reads the whole K and V tile for its WQ query rows: 1 / WQ bytes per
      FLOP) vs. L2 time (every workgroup streams K/V once: 1 / Br bytes per
      FLOP); the non-bottleneck terms only partially overlap
    - softmax: per score element one exponential plus ~4 full rate operations
      on the vector ALU, which runs beside the matrix cores only when another
      wave on the SIMD has MFMAs to issue (or the loop interleaves them itself)
    - wave efficiency: the tail of the last wave of workgroups is wasted
    - barriers: one per KV step, hidden better by several smaller resident
      workgroups (`arch.fa_cta_sync_penalty`)
    - a 2-deep K/V ring hides the global->LDS latency; a single slot exposes it
    - causal: tiles crossing the diagonal are computed in full, so only the
      useful fraction of the computed score tiles counts
    """
    if getattr(cfg, "kv_split", False):
        return fa_split_score(cfg, arch, shape, causal)
    B, H, S_q, S_kv, D = shape
    from deca_amd.kernels.flash_attn_hip import query_tiles

    nq = query_tiles(cfg, S_q)
    grid = nq * B * H
    wgs, _ = fa_occupancy(cfg, arch, D, grid)
    slots = arch.sm_nums * wgs
    wave_eff = _wave_efficiency(grid, slots)

    waves_per_simd = wgs * cfg.num_warps / arch.simds_per_cu
    wq = cfg.Br // cfg.num_warps
    cus = arch.sm_nums
    t_mma = cus / (arch.peak_mma_sync_flops * 1e9)
    t_lds = (1.0 / wq) / arch.smem_bw_per_sm
    if getattr(cfg, "q_in_smem", False):
        # the wave's WQ x D Q rows are read again beside the 2 x Bc x D of K and V
        t_lds *= 1.0 + wq / (2.0 * cfg.Bc)
    t_l2 = (1.0 / cfg.Br) * cus / (arch.l2_bw * 1e9)
    # vector-ALU time per FLOP: (4 + 4) lane-cycles per score element, 4 * D FLOPs each
    valu_rate = cus * arch.simds_per_cu * 16 * arch.sm_clock_hz  # lane-ops per second
    t_valu = (8.0 / (4.0 * D)) * cus / valu_rate
    # share of the VALU work hidden under matrix work: by other waves on the SIMD,
    # or by the wave itself when its loop is software pipelined
    # (measured on MI355X: only the slot-interleaved loop adds to what a second wave
    # already hides, and even full overlap leaves ~40 % of the vector time exposed)
    overlap = min(1.0, max(0.0, waves_per_simd - 1.0) + (0.25 if int(cfg.pipe) == 2 else 0.0))
    terms = sorted([t_mma, t_lds, t_l2])
    t_flop = terms[-1] + 0.3 * (terms[0] + terms[1]) + (1.0 - 0.6 * overlap) * t_valu
    t_flop = max(t_flop, t_valu)

    pipe = 1.0 if cfg.stages >= 2 else 0.96
    # S^T one tile ahead without the slots: two S^T accumulators and a longer dependent
    # chain for nothing in return (measured 2-8 % behind the plain loop of the same tile)
    if int(cfg.pipe) == 1:
        pipe *= 0.90
    # 16x16x32 tiles, measured against the 32x32x16 twin (S = 4096): slot loop 1-2 % behind
    # on full shapes and level under the causal mask; plain loop 5-8 % ahead at D = 128 and
    # 1-2 % behind at D = 64.
    if getattr(cfg, "mfma", 32) == 16:
        if int(cfg.pipe) == 2:
            pipe *= 0.98 if not causal else 1.0
        else:
            pipe *= 1.04 if D >= 128 else 0.985
    # one copy of the two-stage plain loop: no overlap between the end of a step and the start
    # of the next (measured 1-10 % behind the unrolled form where that fits its registers; the
    # solver only emits it where the unrolled form is expected to spill)
    if getattr(cfg, "roll", False):
        pipe *= 0.99
    elif int(cfg.pipe) == 0 and cfg.stages == 2:
        from deca_amd.kernels.flash_attn_hip import register_fill

        # the unrolled form of a tile this tight is expected to spill (3-67 registers measured)
        if register_fill(cfg, D) >= 0.95:
            pipe *= 0.965
    # Measured on exhaustive runs of the S = 4096 shapes (config pairs that differ in nothing
    # else): Q fragments re-read from LDS cost 1-5 % wherever the Q-in-registers twin fits its
    # registers (they only win for tiles that would spill otherwise, which the solver's
    # register limits already drop).  Requesting tiles two steps ahead instead of one pays for
    # small K/V tiles, whose step is too short to cover a tile's latency (8 KiB: 0 ... +8 %,
    # the D = 64 winner), is level to -3 % at 16 KiB and loses beyond.
    if getattr(cfg, "q_in_smem", False):
        pipe *= 0.975
    if cfg.stages == 3:
        tile_kib = cfg.Bc * D * 2 / 1024
        pipe *= 1.015 if tile_kib <= 8 else (0.98 if tile_kib <= 16 else 0.95)
    # K/V loads dealt over the first groups of a step: +1 % in the slot loop, up to +3 % in the
    # plain loop with short (64-key, D = 64) steps, nothing or a little less elsewhere
    if getattr(cfg, "spread", 0):
        pipe *= 1.01 if int(cfg.pipe) == 2 else (1.02 if cfg.Bc * D <= 64 * 64 else 0.995)
    # no max of the tile ahead of its exponentials (plain ring loops): +3.6 % on the full
    # S = 4096 shapes at both head dims; under the causal mask nothing is gained and the
    # second pass the step keeps in reserve costs 4-7 %
    # (16x16x32 tiles then also take the row sums on the matrix pipe: another +3.9 % at D = 64,
    # +1.2 % at D = 128)
    if getattr(cfg, "trust", False):
        pipe *= 1.035 if not causal else 0.95
        if getattr(cfg, "mfma", 32) == 16 and not causal:
            pipe *= 1.035 if D < 128 else 1.01
    if not getattr(cfg, "swizzle", True):
        pipe *= 0.5  # linear LDS rows: every fragment read is a multi-way bank conflict
    sync = 1.0 / (1.0 + getattr(arch, "fa_cta_sync_penalty", 0.0) * cfg.num_warps / 4 / wgs)
    # longer KV steps amortise the per-step max / barrier; the slot loop has the row
    # statistics inside the matrix work and pays a little less of it
    step = 1.0 / (1.0 + (0.06 if int(cfg.pipe) == 2 else 0.08) * 64 / cfg.Bc)

    useful = S_q / (nq * cfg.Br)  # (`edge`: rows beyond the sequence are computed for nothing)
    if causal:
        # a wave computes every tile that reaches one of its rows in full and skips the
        # tiles beyond its last row
        # (`edge`: a wave whose rows all lie beyond the sequence computes nothing)
        computed = sum(-(-min(r + wq, S_kv) // cfg.Bc) * cfg.Bc * wq for r in range(0, S_q, wq))
        useful = S_q * (S_q + 1) / 2 / computed
        # The workgroups of a causal launch differ in length, and towards the end many CUs
        # hold a single one.  A workgroup that fills its SIMDs with two waves by itself keeps
        # its overlap partner until the end; a smaller one does not (measured: the causal /
        # full ratio of 4-wave configs is 0.84-0.86, of 8-wave configs 0.90).
        if cfg.num_warps < 2 * arch.simds_per_cu:
            useful *= 0.90
        # and a wave with more than one 32-query tile skips fewer masked tiles
        useful /= 1.0 + 0.15 * (wq // 32 - 1)

    # every further 32-query tile of a wave lengthens the dependent chain between barriers
    # and the prologue (twice the Q fragments): 17 % at S = 512, 2 % on long sequences
    chain = 1.0 / (1.0 + (0.02 + 0.18 * min(1.0, 512.0 / S_kv)) * (wq // 32 - 1))

    # A workgroup starts with nothing in flight (Q, then the first K/V tile) and ends with
    # the O store: a few microseconds that only another resident workgroup can cover.
    # It matters when the KV loop is short (measured at S = 512: two 4-wave workgroups per
    # CU beat one 8-wave workgroup by 20 %).  This and the other constants of this function
    # were fitted on exhaustive measurements of twelve shapes (S = 512, 1024, 4096; D = 64,
    # 128; full and causal): the measured best is then among the first 8 for all of them
    # and among the first 3 for ten.
    kv_len = S_kv * (0.5 if causal else 1.0)
    t_loop = 4.0 * cfg.Br * kv_len * D / (0.42 * arch.peak_mma_sync_flops * 1e9 / cus)
    exposed = getattr(arch, "fa_workgroup_latency_s", 4e-6) * (1.0 if wgs == 1 else _FA_HIDDEN)
    ramp = t_loop / (t_loop + exposed)

    return wave_eff * pipe * sync * step * useful * chain * ramp / (t_flop / t_mma)


# Coefficients of `fa_time`, in microseconds where they are times, for head dim 128 where they are
# multiplied by D / 128.  Fitted to 10936 measured times (launches back to back over buffers larger
# than the caches) of 1024 shapes: 1 to 124 rows of 32 queries per CU, S_q 128 ... 16384, S_kv 256 ...
# 16384, D 64 and 128, full and causal: least squares on the logarithm of the times, the
# configurations near a shape's best counting most, and what the first choice loses on the best.
FA_TIME = {
    # one 32 x 32 block of scores in a wave's own chain of instructions (matrix and vector part),
    # and its share of a SIMD that has other waves to fill the gaps; of that, what a key step of a
    # wave takes whatever its tile
    "chain_mfma": 0.238, "chain_valu": 0.112, "busy_mfma": 0.162, "busy_valu": 0.0377, "issue": 0.0806,
    # of one key step: the wait for a tile in a one-slot ring, and of that where waves split the keys
    "one_slot": 0.243, "one_slot_split": 0.162,
    # a 32-key tile on the CU's load path, per wave, where waves split the keys
    "load_split": 0.0709,
    "overlap": 1.2,  # exponent that joins chain, busy pipes and load path into a step's time
    # per workgroup: per 32 query rows of a wave, per 32 keys of a tile (the first one is waited for),
    # more where more workgroups share the CU, and without a second one beside it (per wave); the
    # meeting of the waves that split keys (per wave), more where more workgroups share the CU
    "wg_rows": 1.27, "wg_tile": 0.237, "wg_shared": 0.145, "wg_alone": 0.49,
    "meet": 0.335, "meet_shared": 0.379,
    # under the mask: exponent that joins the sum of the work and the longest row of it, and the
    # share of its steps that the longest row is alone on its CU (all where waves split the keys);
    # of both, where all workgroups fit the CUs at once; where they don't, the wait between one
    # workgroup of a CU and the next
    "causal": 7.17, "causal_split": 4.83, "causal_once": 4.05, "causal_split_once": 4.68,
    "alone": 0.59, "alone_once": 0.798, "alone_split_once": 0.896, "refill": 1.16, "refill_split": 0.884,
    # equal workgroups drift apart: a part-filled last round counts as a whole one behind the first,
    # more and more with its share behind many
    "drift": 0.23,
    # PFLOP/s that the card sustains (power, and the vector work beside the matrix work), joined by
    # this exponent
    "rate_64": 1.09, "rate_128": 1.26, "rate_join": 4.0,
    # memory: bytes at 6.4 TB/s times this, joined by this exponent; the launch
    "memory": 1.24, "memory_join": 1.62, "launch": 1.72,
}
# Logarithms of what the form of a key step does to its time ...
FA_FORM = {
    "mfma16_64": 0.109, "mfma16_128": 0.122, "mfma16_slots": 0.0957, "mfma16_causal": -0.0263,
    "mfma16_roll": -0.0994, "slots": -0.16, "slots_64": 0.0968, "slots_64_causal": 0.000893,
    "ahead": 0.086, "trust": -0.0277, "trust_causal": 0.121, "trust_mfma16_64": -0.119,
    "three_slots": 0.288, "three_slots_64": -0.176, "q_lds": 0.147, "q_lds_64": -0.0915,
    "q_lds_64_rows": 0.037, "spread": 0.0378, "spread_slots": -0.0395, "spread_slots_64": 0.0165,
    "spread_short": -0.0161, "slots_128_keys": -0.068, "plain_128_keys": 0.0566, "roll": -0.00181,
    "roll_64": 0.108, "edge": 0.00279, "two_waves": 0.171, "one_wave": 0.241, "split_128": 0.113,
    "split_two_slots": 0.0767, "split_two_slots_causal": 0.0483,
}
# ... and to the time that the work takes at the sustained rate ("rows": times 128 rows over those of
# all waves, less a half).
FA_RATE = {
    "slots_64": 0.0236, "mfma16": -0.0839, "trust": -0.0364, "rows": 0.0729, "q_lds": 0.0694,
}


def fa_form_factor(cfg, D: int, causal: bool, short: bool) -> float:
    """What the form of a key step (`FA_FORM`) does to its time; `short`: at most eight of them."""
    f, small, full, split = FA_FORM, D < 128, not causal, cfg.kv_split
    mfma16, slots = cfg.mfma == 16, int(cfg.pipe) == 2
    log = f["edge"] * cfg.edge
    if mfma16:
        log += f["mfma16_64"] if small else f["mfma16_128"]
        log += f["mfma16_slots"] * slots + f["mfma16_causal"] * causal + f["mfma16_roll"] * cfg.roll
    if slots:
        log += f["slots"] + (f["slots_64"] + f["slots_64_causal"] * causal) * small
    log += f["ahead"] * (int(cfg.pipe) == 1)
    if cfg.Bc >= 128 and not split:
        if slots:  # (level in four waves, and under the mask)
            log += f["slots_128_keys"] * (full and cfg.num_warps != 4)
        else:
            log += f["plain_128_keys"]
    if cfg.trust:
        log += (f["trust_causal"] if causal else f["trust"]) * (not split)
        log += f["trust_mfma16_64"] * (full and mfma16 and small)
    if cfg.stages == 3:
        log += f["three_slots"] + f["three_slots_64"] * small
    if cfg.q_in_smem:
        log += f["q_lds"] + f["q_lds_64"] * small + f["q_lds_64_rows"] * (cfg.wave_rows > 32)
    if cfg.spread:
        log += f["spread"] + (f["spread_slots"] + f["spread_slots_64"] * small) * slots
        log += f["spread_short"] * short
    if cfg.roll:
        log += f["roll"] + f["roll_64"] * small
    if split:
        log += f["split_128"] * (not small)
        log += (f["split_two_slots"] + f["split_two_slots_causal"] * causal) * (cfg.stages > 1)
    else:
        log += f["two_waves"] * (cfg.num_warps == 2) + f["one_wave"] * (cfg.num_warps == 1)
    return math.exp(log)


def fa_sustained_us(cfg, shape, causal: bool = False) -> float:
    """Microseconds that the matrix and vector work of a launch takes at the rate that the card sustains
    (`FA_TIME` "rate_*", PFLOP/s, and `FA_RATE`), rows and keys that are computed for nothing included."""
    from deca_amd.kernels.flash_attn_hip import query_tiles

    B, H, S_q, S_kv, D = shape
    scores = query_tiles(cfg, S_q) * cfg.Br * S_kv
    if causal:  # a wave computes every tile that reaches one of its rows in full
        wq = cfg.wave_rows
        scores = sum(-(-min(r + wq, S_kv) // cfg.Bc) * cfg.Bc * wq for r in range(0, S_q, wq))
    f = FA_RATE
    log = (f["slots_64"] * (int(cfg.pipe) == 2 and D < 128) + f["mfma16"] * (cfg.mfma == 16)
           + f["trust"] * cfg.trust + f["rows"] * (128 / (cfg.num_warps * cfg.wave_rows) - 0.5)
           + f["q_lds"] * cfg.q_in_smem)
    return B * H * 4.0 * D * scores / (FA_TIME["rate_64" if D < 128 else "rate_128"] * 1e9) * math.exp(log)


def fa_time(cfg, arch, shape, causal: bool = False) -> float:
    """Expected microseconds of a launch, head dims 64 and 128.

    A workgroup is a number of key steps and a fixed part.  A step takes as long as its wave's own
    chain of instructions, or as the busy pipes of a SIMD that its waves share, or as the CU's load
    path, and somewhat longer where two of them are close.  All workgroups at once if they fit the
    CUs; else whole rounds of those that do (equal workgroups end together: 1.2 rounds take two) and
    a last one of those that are left, fewer a CU and so faster; under the causal mask the sum of the
    work or the longest row, which starts first.  Long sequences come to the rate that the card
    sustains.
    Over 1350 sets of configurations of a shape measured in turn (1024 shapes) the first choice of
    `rank_fa_configs` is 1.5 % behind the best on the average, more than 10 % on 53 and 39 % at most;
    fitted to three quarters of them, 1.6 % on the others.  By `fa_score` (without the query edge) it
    is 11 % behind, more than 10 % on 565."""
    from deca_amd.kernels.flash_attn_hip import query_tiles

    c = FA_TIME
    B, H, S_q, S_kv, D = shape
    d, split = D / 128, cfg.kv_split
    grid = query_tiles(cfg, S_q) * B * H
    fit, _ = fa_occupancy(cfg, arch, D, grid)
    per_cu = grid / arch.sm_nums
    together = min(math.ceil(per_cu), fit)
    mq, bc = cfg.wave_rows / 32, cfg.Bc / 32
    steps = math.ceil(S_kv / (cfg.Bc * cfg.num_warps)) if split else S_kv / cfg.Bc
    share = 0.5 * (1.0 + cfg.Br / S_q) if causal else 1.0  # of the keys that the mean row sees
    form = fa_form_factor(cfg, D, causal, steps * share <= 8)
    one_slot = c["one_slot_split" if split else "one_slot"] * (cfg.stages == 1)

    def step(workgroups):
        waves = workgroups * cfg.num_warps / arch.simds_per_cu
        # (a single round is as long as its fullest SIMD)
        waves = max(1.0, math.ceil(waves) if per_cu <= fit and workgroups > 1 else waves)
        chain = mq * bc * (c["chain_mfma"] * d + c["chain_valu"]) + one_slot
        busy = waves * (mq * bc * (c["busy_mfma"] * d + c["busy_valu"]) + c["issue"])
        load = c["load_split"] * cfg.num_warps * workgroups * bc * d if split else 0.0
        p = c["overlap"]
        return (chain**p + busy**p + load**p) ** (1 / p) * form

    def fixed(workgroups):
        t = c["wg_rows"] * mq * d + (c["meet"] * cfg.num_warps * d * mq if split else c["wg_tile"] * bc * d)
        t *= 1.0 + c["meet_shared" if split else "wg_shared"] * (workgroups - 1)
        return t + c["wg_alone"] * cfg.num_warps * d * (fit == 1 and per_cu > 1 and not split)

    if causal:
        mean = steps * share * step(together) + fixed(together)
        kind = ("_split" if split else "") + ("_once" if per_cu <= fit else "")
        alone = c.get("alone" + kind, 1.0)
        longest = steps * (alone * step(1) + (1.0 - alone) * step(together)) + fixed(together)
        q = c["causal" + kind]
        t = ((per_cu / together * mean) ** q + longest**q) ** (1 / q)
        if per_cu > fit:
            t += c["refill" + kind]
    else:
        rounds = math.floor(per_cu / together + 1e-9) if per_cu > fit else 1
        whole = steps * step(together) + fixed(together)
        t = rounds * whole
        left = math.ceil(per_cu - rounds * together - 1e-9)
        if left > 0:
            apart = 1.0 - 1.0 / (1.0 + c["drift"] * (rounds - 1))
            t += steps * step(left) + fixed(left)
            t = (1.0 - apart) * t + apart * per_cu / together * whole
    j, m = c["rate_join"], c["memory_join"]
    t = (t**j + fa_sustained_us(cfg, shape, causal) ** j) ** (1 / j)
    memory = c["memory"] * 2 * B * H * D * 2 * (S_q + S_kv) / 6.4e6
    return (t**m + memory**m) ** (1 / m) + c["launch"]


def rank_fa_configs(configs, arch, shape, causal: bool = False, top_n: int | None = None):
    """Sort FlashAttention configs, best first: by `fa_time` at the head dims it was fitted for
    (64 and 128), by `fa_score` at others."""
    if shape[4] in (64, 128):
        ranked = sorted(configs, key=lambda c: fa_time(c, arch, shape, causal))
    else:
        # Query edges by the score are ahead of the first dividing tile on 45 of 46 shapes of D 192 and
        # 384 and of full ones of D 256 and 320 (0.96 ... 6x).  Under the mask at D 256 and 320 the score
        # does not know what their registers cost: 0.39 ... 1.02x on eight shapes of up to 576 rows,
        # 0.86 ... 1.8x on eight from 960 on.
        late = causal and 192 < shape[4] < 384 and shape[2] < 960
        ranked = sorted(configs, key=lambda c: (not (late and c.edge), fa_score(c, arch, shape, causal)),
                        reverse=True)
    return ranked[:top_n] if top_n else ranked
