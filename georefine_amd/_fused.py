"""Host-side preparation of a mode-0 BCTX frame for the fused kernels.

Everything here is derived data: the frame's byte streams are used as they are.
The fused index is the checkpoint index at a segment length that divides the row
length; rows are grouped by row class into tiles; per class the frequency rows
become a coarse u8 lookup plus a sparse table of the symbols that occur.
"""
from __future__ import annotations

import copy
import ctypes
import heapq
import math
import os

import numpy as np

from . import _native

MAX_LDS = 160 * 1024
LDS_UNIT = 1280  # what a compute unit's LDS is given out in


def lds_share(lds):
    """Workgroups of ``lds`` bytes (a number or an array) that a compute unit's LDS holds: it is given out in
    units of 1280 bytes, and all 128 of them are there to be had.  Measured with workgroups of one wave
    that stay: two of 81920 bytes share a unit, three of 53760 and not of 53776, four of 40960, five of 32000 and
    not of 32016, six of 26880 and not of 26896."""
    return MAX_LDS // (-(-lds // LDS_UNIT) * LDS_UNIT)
LUT_BUDGET = int(os.environ.get("GEOREFINE_FUSED_LUT_BYTES", 32 * 1024))


class FusedUnsupported(ValueError):
    """The frame cannot use the fused kernels (the caller falls back to decode + dense)."""


SMALL_MATRIX = 8 << 20  # elements below which the walk, not the machine, bounds a launch


def choose_segment(cols, preferred=None, rows=None):
    """Segment length that divides the row length: the one asked for (``preferred``), or 64 by
    default (index 1 bit per weight).  A launch takes at least one segment's worth of dependent steps (0.1 us each), so matrices too
    small to fill the GPU several times over get 32 (2 bits per weight of index), the smallest
    16 (4 bits).  That is paid in device memory: bits per weight in all, by default and at 64, 2048 x
    5120 13.5 and 12.5, 2048 x 1024 19.1 and 16.1 (5.5 of them tables, which do not shrink with the
    matrix).  A caller that asks for a length asks for its index: where it does not divide, matrices
    under 8 M weights get 32, others 64, before anything shorter.  GPU time of a product of 1, 8 and 32 rows and of decode(), us:
      3500 x 1024   32: 12.0 15.3 16.1 12.3   16: 11.0 11.3 11.5 11.3
      300 x 4096    32: 11.3 15.0 15.4 10.8   16: 10.2 12.9 13.1  8.9
      2000 x 2048   32: 11.7 13.8 13.9 11.9   16: 11.8 13.7 14.1 11.8
      2048 x 5120   64: 17.9 24.3 26.8 20.6   32: 16.3 20.3 22.8 17.7
      2700 x 5120   64: 23.2 25.6 28.2 28.3   32: 21.9 27.6 29.7 24.3
    Long rows pay for the short segments in sums per row, and keep the longer ones earlier:
      256 x 15360   32: 13.0 16.8 17.4 11.6   16: 14.4 18.6 19.1 10.9
      640 x 16384   64: 21.9 23.4 26.3 22.1   32: 19.5 25.2 27.6 18.2"""
    weights = rows * cols if rows is not None else 1 << 32
    order = [preferred] if preferred else []
    if not preferred and cols <= 4096 and weights < 15 << 18:
        order += [16]
    elif weights < (11 << 20 if not preferred and cols <= 8192 else SMALL_MATRIX):
        order += [32, 64, 16, 128, 256]
    else:
        order += [64, 128, 32, 256, 16]
    for s in order:
        if s and s % 16 == 0 and cols % s == 0:
            return s
    raise FusedUnsupported("row length is not a multiple of 16")


def choose_shift(nc, budget=LUT_BUDGET):
    """Bucket shift so that nc << (16 - shift) bytes stay within the LUT budget."""
    shift = 0
    while (nc << (16 - shift)) > budget and shift < 12:
        shift += 1
    return shift


def sparse_tables(freq, nr, nc, shift, image=None):
    """Per row class: u8 lookup [nc << lognb] and u64 entries [nc][tabn+1].

    Entry(column class c, sparse i): low32 = start | (freq & 0xFFFF) << 16 with 0 standing for
    65536, high32 = image(symbols), the symbol's bits in the BF16 word (default: symbol << 5,
    the context codec's 10-bit main symbol).  Unused entries are (start 0, freq 65536): a forward scan
    always stops on them.  The lookup byte of a bucket is the sparse index of the symbol
    that owns most of the bucket's slots (the first of them on a tie), which minimises the
    slots whose lookup has to scan to a neighbouring entry."""
    nz = freq > 0
    tabn = int(nz.sum(axis=1).max())
    if tabn == 0:
        raise FusedUnsupported("no live context")
    if tabn > 255:
        raise FusedUnsupported("more than 255 distinct symbols in one context")
    nb = 1 << (16 - shift)
    freq = np.ascontiguousarray(freq, dtype=np.uint32)
    symbols = np.arange(freq.shape[1])
    images = np.ascontiguousarray(symbols << 5 if image is None else image(symbols), dtype=np.uint32)
    lut = np.empty((nr, nc * nb), dtype=np.uint8)
    tab = np.empty((nr, nc * (tabn + 1)), dtype=np.uint64)
    if _native.codec().grf_sparse_tables(_native.ptr(freq, ctypes.c_uint32), nr * nc, freq.shape[1], shift,
                                         _native.ptr(images, ctypes.c_uint32), tabn, _native.ptr(lut, ctypes.c_uint8),
                                         _native.ptr(tab, ctypes.c_uint64)):
        raise FusedUnsupported("frequencies of a context do not add up to 65536")
    return lut, tab, tabn


X_PAD = 8


def lds_bytes(nc, lognb, tabn, m, p, s, r, piece_cap):
    a16 = lambda v: (v + 15) // 16 * 16
    total = a16(nc * (a16((tabn + 1) * 8) + (1 << lognb)))
    total = a16(total + r * piece_cap)
    total = a16(total + m * p * (s + X_PAD) * 2)
    total = a16(total + r * p * m * 4)
    total = a16(total + r * m * 4)
    return total


def lds_bytes_waves(nc, lognb, tabn, m, threads, p, r, n_slabs, piece_cap):
    """LDS of the wave-unit GEMV: tables, one row piece per row of every wave's unit, the unit
    sums of every (row, slab), the tile's rows."""
    a16 = lambda v: (v + 15) // 16 * 16
    total = a16(nc * (a16((tabn + 1) * 8) + (1 << lognb)))
    total = a16(total + threads // 64 * (64 // p) * piece_cap)
    total = a16(total + r * n_slabs * m * 4)
    total = a16(total + r * 8)
    return total


GEMM_MAX_TILES = 4  # 16-row activation tiles whose partial sums pass through LDS at a time


def gemm_shape(p, r):
    """(row blocks, quads, threads) of the GEMM workgroup for p lanes per row and r rows: a
    wave walks four lane-segments of sixteen rows."""
    row_blocks, quads = -(-r // 16), -(-p // 4)
    return row_blocks, quads, row_blocks * quads * 64


def lds_bytes_gemm(nc, lognb, tabn, p, r, piece_cap, wave_bytes=0):
    """Tables, then sixteen row pieces of four segments per wave (``wave_bytes`` for the sixteen, where
    given); later every wave's partial sums."""
    a16 = lambda v: (v + 15) // 16 * 16
    waves = gemm_shape(p, r)[2] // 64
    total = a16(nc * (a16((tabn + 1) * 8) + (1 << lognb)))
    total = a16(total + waves * (wave_bytes or 16 * piece_cap))
    return max(total, waves * GEMM_MAX_TILES * 1024)


WINDOW = 8  # bytes the refill reads from the 4-byte aligned cursor on


def piece_capacity(offsets, rows, spr, p):
    """LDS bytes one row piece may need: the longest (16-byte aligned start .. end) span
    over every (row, slab), plus the eight bytes the refill's window may read from the
    cursor on, rounded to 16."""
    off = offsets[:-1].reshape(rows, spr).astype(np.int64)
    end_of_row = np.concatenate((off[1:, 0], [int(offsets[-1])]))
    longest = 0
    for b in range(0, spr, p):
        g0 = off[:, b]
        g1 = off[:, b + p] if b + p < spr else end_of_row
        longest = max(longest, int((g1 - (g0 & ~15)).max()))
    return (longest + WINDOW + 15) // 16 * 16


def quad_piece_capacity(offsets, rows, spr):
    """LDS bytes of a GEMM wave's row piece: four consecutive segments of a row from any first
    segment (fewer at the row's end), from the 16-byte aligned start, plus the refill's window."""
    off = offsets[:-1].reshape(rows, spr)
    end_of_row = np.concatenate((off[1:, :1], offsets[-1:, None]))
    aligned = off & off.dtype.type(0xFFFFFFF0)
    whole = max(0, spr - 4)  # first segments that have four and a further one behind them
    longest = int((off[:, 4:] - aligned[:, :whole]).max()) if whole else 0
    longest = max(longest, int((end_of_row - aligned[:, whole:]).max()))
    return (longest + WINDOW + 15) // 16 * 16


def _tiles(class_rows, r):
    return sum(-(-int(cnt) // r) for cnt in class_rows if cnt)


def _tile_counts(class_rows, most):
    """[.., tiles of r rows, ..] for r = 0 (unused) .. most: the planners look these up thousands
    of times a matrix."""
    r = np.arange(1, most + 1, dtype=np.int64)
    return [0] + (-(-np.asarray(class_rows, dtype=np.int64)[:, None] // r)).sum(axis=0).tolist()


def _spread_rows(tile_counts, r, capacity, floor=1):
    """Fewer rows per tile while the tiles still fit the workgroup slots of the rounds
    already paid for: idle lanes do not slow a workgroup down, idle CUs do (measured +4 % on
    17408 x 5120 going from 464 tiles of 38 rows to 512 of 34)."""
    while r > floor and tile_counts[r - 1] <= capacity:
        r -= 1
    return r


def _walk_share(n_slabs, seg_len, table_bytes):
    """Share of a workgroup's life spent walking, in units of decode steps: before the first
    step a workgroup copies its row class's tables (about a step per 12 KiB, measured on
    53 KiB tables with one 64-step slab: 10 %) and every slab costs a barrier and a staging
    round (about two steps)."""
    steps = n_slabs * seg_len
    return steps / (steps + 3 + table_bytes / 12288 + 2 * n_slabs)


def choose_tiling(spr, class_rows, piece_cap_fn, lds_fn, cus=256, seg_len=64, table_bytes=0):
    """(threads T, lanes_per_row P, rows_per_tile R, ...): best modelled throughput.

    The walk is a chain of dependent steps per lane, so time ~ steps per lane x rounds
    of workgroups, at the speed the resident wave count allows.  The model multiplies
    lane efficiency (idle lanes in the last slab and in a partly filled workgroup), tile
    fill, how evenly the tiles fill the machine, and a penalty below 24 waves per CU
    (measured: the dependent LDS round trips of a step need that many waves to overlap)."""
    candidates = []
    total_rows = sum(int(c) for c in class_rows)
    forced = os.environ.get("GEOREFINE_FUSED_TILING")  # "threads,lanes_per_row[,rows]": experiments only
    thread_choices = range(1024, 0, -64)
    lane_choices = None
    forced_rows = None
    tile_counts = _tile_counts(class_rows, 1024)
    if forced:
        t_, p_, *rest = (int(v) for v in forced.split(","))
        thread_choices, lane_choices = [t_], [min(p_, spr)]
        forced_rows = rest[0] if rest else None
    for threads in thread_choices:
        for p in (lane_choices or range(1, min(spr, threads) + 1)):
            r = threads // p
            if forced_rows:
                r = min(r, forced_rows)
            if r == 0:
                continue
            n_slabs = -(-spr // p)
            if not forced and p > 1 and -(-spr // (p - 1)) == n_slabs:
                continue  # a narrower slab of the same count wastes fewer lanes; it was scored already
            lanes = p * r
            lane_eff = spr / (n_slabs * p) * (lanes / threads)
            tiles = tile_counts[r]
            fill = total_rows / (tiles * r)
            cap = piece_cap_fn(p)
            lds = lds_fn(p, r, cap)
            if lds > MAX_LDS:
                continue
            # A workgroup's waves are dealt round-robin to the CU's four SIMDs; the kernels use
            # up to 72 vector registers, which allows 7 waves per SIMD.
            per_simd = -(-(threads // 64) // 4)
            per_cu = max(1, min(7 // per_simd, lds_share(lds)))
            waves = per_cu * (threads // 64)
            slots = cus * per_cu
            rounds = -(-tiles // slots)
            quant = tiles / (rounds * slots)
            score = lane_eff * fill * quant * min(1.0, waves / 24) * _walk_share(n_slabs, seg_len, table_bytes)
            candidates.append((score, threads, p, r, n_slabs, tiles, cap, lds, rounds * slots))
    if not candidates:
        raise FusedUnsupported("no tiling fits in LDS")
    # Among tilings the model cannot tell apart (1.5 %), the one with the fewest slabs: fewer
    # lanes per row make a row's residual bytes of one slab span fewer 128-byte lines, so more
    # of them straddle two slabs and are fetched twice (measured on gate+up: 10 lanes per row
    # read 1.68x the algorithmic bytes, 20 lanes 1.1x, in the same time).
    top = max(c[0] for c in candidates)
    best = max((c for c in candidates if c[0] >= 0.985 * top), key=lambda c: (-c[4], c[0], c[1]))
    _, threads, p, r, n_slabs, tiles, cap, lds, capacity = best
    if not forced_rows:
        r = _spread_rows(tile_counts, r, capacity)
        tiles, lds = tile_counts[r], lds_fn(p, r, cap)
    return threads, p, r, n_slabs, tiles, cap, lds


SCHEME_SLABS, SCHEME_WAVES = 0, 1
WAVE_ROWS_PER_PASS = 2  # activation rows one launch of the wave-unit kernel carries
WAVES_PER_CU = 24       # of the wave-unit kernels, by their registers
LINES_WAVES_PER_CU = 16  # of the one that stores whole lines
WAVE_UNIT_OVERHEAD = 8  # decode steps' worth of staging, reduction and bookkeeping per unit


WAVE_PIECE_OVERHEAD = 1.7   # decode steps' worth of staging per row piece of a unit (fitted, see below)
WAVE_LATENCY_RATIO = 4.5    # a lone wave's time for a step / its share of a saturated SIMD's issue time


def choose_wave_tiling(spr, class_rows, piece_cap_fn, lds_fn, cus=256, seg_len=64, table_bytes=0, waves=WAVES_PER_CU):
    """Tiling of the wave-unit GEMV: a wave walks units of 64 / P rows x P consecutive
    segments (P a power of two) and the waves of a workgroup share out the units of its tile
    without meeting at a barrier; a tile is a whole number of units (a unit's rows are then a
    block of the resident residual order).

    Modelled time, in decode steps of one SIMD: a launch is bounded by the chain of units its
    busiest wave walks one after the other (each step a round trip of dependent instructions
    and LDS reads: WAVE_LATENCY_RATIO issue slots) and by the instructions all waves of a
    compute unit issue on its four SIMDs; the two are joined as a cubic mean, and the busiest
    wave counts half by its own units and half by the average (waves that finish leave the
    rest the machine).  A unit costs its steps, WAVE_UNIT_OVERHEAD, and WAVE_PIECE_OVERHEAD
    per row piece it stages.  Fitted on a sweep of 120 forced tilings each of 6144 x 5120,
    5120 x 6144, 1024 x 5120, 17408 x 5120 and 5120 x 17408 on the GPU: the model's choice is
    the fastest measured tiling for four of them and 9 % off for the smallest (rank
    correlation 0.89 to 0.99); counting paid lane-steps alone, as before, chose tilings 16 %
    and 29 % slower than the best for the two middle shapes."""
    forced = os.environ.get("GEOREFINE_FUSED_WAVE_TILING")  # "threads,lanes_per_row,rows": experiments only
    if forced:
        t_, p_, r_ = (int(v) for v in forced.split(","))
        cap = piece_cap_fn(p_)
        n_slabs = -(-spr // p_)
        return t_, p_, r_, n_slabs, _tiles(class_rows, r_), cap, lds_fn(t_, p_, r_, n_slabs, cap)
    threads, p, (r,), tiles, cap, lds = search_wave_tilings(
        [(spr, seg_len, class_rows)], piece_cap_fn, lambda t_, p_, heights, cap_: lds_fn(t_, p_, heights[0], -(-spr // p_), cap_),
        cus, table_bytes, waves)
    return threads, p, r, -(-spr // p), tiles, cap, lds


def search_wave_tilings(lengths, piece_cap_fn, lds_fn, cus, table_bytes, waves=WAVES_PER_CU):
    """The fastest wave tiling by ``choose_wave_tiling``'s model, as (threads, lanes per row, rows per
    tile of every length, tiles, piece capacity, LDS bytes), of a launch over matrices of one width
    indexed at several ``lengths``: (segments per row, segment length, rows per class) each, the one
    that sets the pace first.  The tiles of another length are as tall as they can be without
    taking their waves longer (at one height for all, the units of the shorter segments are twice as
    many a tile and go a second round: 2048 x 2560 at 32 with 1024 x 2560 at 16, one row: 17.7 us,
    so 16.2)."""
    best = None
    counts, others = [_tile_counts(class_rows, 128) for _, _, class_rows in lengths], range(1, len(lengths))
    table_steps = 3 + table_bytes / 12288
    for p in (4, 8, 16, 32, 64):
        if p > 4 and all(p // 2 >= spr for spr, _, _ in lengths):
            continue  # half the lanes of every unit would idle
        rpw = 64 // p
        cap = piece_cap_fn(p)
        slabs = [-(-spr // p) for spr, _, _ in lengths]
        unit_steps = [seg_len + WAVE_UNIT_OVERHEAD + WAVE_PIECE_OVERHEAD * rpw for _, seg_len, _ in lengths]
        # (768 threads, two workgroups a compute unit, where the LDS allows: a matrix with a few long
        # rows needs larger pieces, and one wave less per workgroup then keeps two of them resident --
        # 17408 x 5120 with pieces of 912 bytes: 68.7 us with 11 waves against 95.0 with 12 and
        # tiles cut down to 8 rows)
        for threads in (1024, 768, 704, 640, 576, 512) if waves > LINES_WAVES_PER_CU else (1024, 512):
            nwaves = threads // 64
            busiest = lambda units: 0.5 * -(-units // nwaves) + 0.5 * units / nwaves  # units of the wave that has most
            heights = [rpw] * len(lengths)
            for r in range(rpw, 129, rpw):
                heights[0] = r
                units = r // rpw * slabs[0]
                longest = busiest(units) * unit_steps[0]
                tiles = counts[0][r]
                steps = tiles * (units * unit_steps[0] + nwaves * table_steps)
                for k in others:
                    while heights[k] + rpw <= 128 and busiest((heights[k] // rpw + 1) * slabs[k]) * unit_steps[k] <= longest:
                        heights[k] += rpw
                    units = heights[k] // rpw * slabs[k]
                    longest = max(longest, busiest(units) * unit_steps[k])
                    tiles += counts[k][heights[k]]
                    steps += counts[k][heights[k]] * (units * unit_steps[k] + nwaves * table_steps)
                chain, issue = (longest + table_steps) * WAVE_LATENCY_RATIO, steps / cus / 4  # (of one round)
                if best is not None and max(chain, issue) >= best[0]:  # taller tiles only make longer chains
                    if chain >= best[0]:
                        break
                    continue
                lds = lds_fn(threads, p, heights, cap)
                if lds > MAX_LDS:
                    break
                # (the waves that the kernel's registers allow)
                per_cu = max(1, min(waves // nwaves, lds_share(lds)))
                rounds = -(-tiles // (cus * per_cu))
                chain *= rounds
                time = (chain ** 3 + issue ** 3) ** (1 / 3)
                if best is None or time < best[0] * 0.9999:
                    best = (time, threads, p, tuple(heights), tiles, cap, lds, rounds * cus * per_cu)
    if best is None:
        raise FusedUnsupported("no wave-unit tiling fits in LDS")
    _, threads, p, heights, tiles, cap, lds, capacity = best
    if others:  # (idle workgroup slots of the rounds already paid for: 2560 x 5120 at 64 with 2048 at 32 31.1 -> 29.6)
        heights, rpw = list(heights), 64 // p
        for k in others:
            while heights[k] > rpw and tiles + counts[k][heights[k] - rpw] - counts[k][heights[k]] <= capacity:
                tiles += counts[k][heights[k] - rpw] - counts[k][heights[k]]
                heights[k] -= rpw
    return threads, p, tuple(heights), tiles, cap, lds


def wave_time(tiling, seg_len, table_bytes, cus=256, waves=WAVES_PER_CU):
    """What ``choose_wave_tiling``'s model says of one tiling (as ``FramePlan.tiling`` returns it), in
    decode steps of a SIMD."""
    g = tiling["scalars"]
    nwaves, rpw = g["threads"] // 64, 64 // g["lanes_per_row"]
    unit_steps, table_steps = seg_len + WAVE_UNIT_OVERHEAD + WAVE_PIECE_OVERHEAD * rpw, 3 + table_bytes / 12288
    units = -(-g["rows_per_tile"] // rpw) * g["n_slabs"]
    rounds = -(-g["n_tiles"] // (cus * max(1, min(waves // nwaves, lds_share(tiling["lds"])))))
    chain = rounds * ((0.5 * -(-units // nwaves) + 0.5 * units / nwaves) * unit_steps + table_steps) * WAVE_LATENCY_RATIO
    issue = g["n_tiles"] / cus * (units * unit_steps + nwaves * table_steps) / 4
    return (chain ** 3 + issue ** 3) ** (1 / 3)


GEMM_WAVES_PER_SIMD = int(os.environ.get("GEOREFINE_GEMM_WAVES", "6"))
# a single matrix's GEMM may be cut along K ("0": never; experiments and tests of the uncut kernel)
GEMM_SPLIT = os.environ.get("GEOREFINE_FUSED_GEMM_SPLIT", "1") != "0"


GEMM_K_PARTS = (1, 2, 3, 4, 6, 8)  # cuts along K the planner tries for a single matrix


def choose_gemm_tiling(spr, class_rows, piece_cap_fn, lds_fn, cus=256, seg_len=64, table_bytes=0, split=False):
    """``plan_gemm_tiling`` where every row's piece is given the LDS of the longest."""
    return plan_gemm_tiling(spr, class_rows, piece_cap_fn, lambda p, r, cap, _: lds_fn(p, r, cap), cus, seg_len, table_bytes,
                            split)[:8]


# gemm_times: rows, then steps' worth of work a slab, of work a table copy per 12 KiB, the latency of a step in
# issue slots, the exponent that joins chain and issue, and us: of a launch, of a cut along K, of each part, of
# an issue slot; and the weight of the fullest compute unit against the mean one.
GEMM_TIMES = ((6, 0.827, 5.44, 3.759, 3.167, 4.93, 2.66, 0.0, 0.036, 0.842), (32, 0.165, 7.23, 3.57, 3.264, 5.64, 2.94, 0.0, 0.041, 0.812),
              (64, 1.861, 11.06, 3.283, 3.076, 5.54, 3.27, 0.0, 0.043, 0.762), (100, 0.0, 10.05, 2.271, 3.486, 4.85, 3.8, 0.405, 0.07, 0.615))


def gemm_times(threads, tallest, blocks, n_slabs, tiles, k, lds, spr, seg_len, table_bytes, cus=256):
    """Modelled us of matrix-core launches of 6, 32, 64 and 100 rows with each of several tilings (arrays;
    ``tallest``, ``blocks``: blocks of sixteen rows the tallest tile has, and a tile on average), for frames of the context codec.  A launch is bounded by the chain of slabs a wave walks one after
    the other and by what the fullest SIMD issues, joined as a power mean.  The waves of a workgroup
    are dealt to the four SIMDs in turn, so a count that is no multiple of four fills one SIMD before the
    others (two workgroups of ten: 6 waves where 5 are the mean); waves whose quad a row's last slab
    does not reach leave, and cost nothing there.  Above 64 rows fewer workgroups share a compute unit
    (``shares_units`` in fused_kernels.h).  Fitted to forced tilings of fourteen matrices with kernels before the
    present ones.  Against those (profiles/gemm_tilings.csv: 1655 tilings of 44 matrices, made by the program
    beside it) the times are 5, 7, 6 and 3 % long on average, and 9, 12, 13 and 14 % rms around that; what that is
    worth between two tilings of one matrix is what ``gain_to_ask`` goes by."""
    waves, quads = threads // 64, -(-spr // 4)
    each = -(-n_slabs // k)
    most, fullest = np.maximum(1, np.minimum(GEMM_WAVES_PER_SIMD // -(-waves // 4), lds_share(lds))), -(-tiles // cus)
    shared = (tiles > 256) & (threads <= 640) & (lds <= 79 * 1024)
    fewer = np.where(shared, most, np.maximum(1, np.minimum(4 // -(-waves // 4), lds_share(lds))))
    times = []
    for rows, unit, table, latency, power, launch, cut, part, slot, weight in GEMM_TIMES:
        per_cu = most if rows <= 64 else fewer
        at_once, rest = np.minimum(fullest, per_cu), waves % 4
        extra = np.where(rest == 0, 0, np.where(at_once == 1, 1, np.where(at_once == 2, 1 + (rest >= 2), -(-at_once * rest // 4) + (rest == 2))))
        uneven = 4 * (at_once * (waves // 4) + np.minimum(extra, at_once)) / (at_once * waves)
        copy = table * table_bytes / 12288
        chain = -(-fullest // per_cu) * (each * (seg_len + unit) + copy) * latency
        walks = (fullest * weight * tallest + tiles / cus * (1 - weight) * blocks) * quads / k
        copies = (fullest * weight + tiles / cus * (1 - weight)) * waves
        issue = (walks * (seg_len + unit) * uneven + copies * copy) / 4
        times.append(slot * (chain ** power + issue ** power) ** (1 / power) + launch + np.where(k > 1, cut + part * k, 0.0))
    return np.stack(times)


def spread_apart(tiles, slots, unit):
    """Whether a launch whose workgroups share compute units by the tight reservation (``unit`` bytes a wave) is spread
    over the ``slots`` it had without: where its tiles all have one of those, shorter tiles only mean more
    copies of the tables (three of 4612 x 768 at one, 32, 100 rows in 480 tiles or spread to 768: 19.5 22.7 31.8 us, 21.0
    24.4 33.6; 7162 x 1408 in 512 or 720: 16.9 19.5 26.9, 19.8 22.9 30.4)."""
    return unit > 0 and tiles <= slots


def closer_workgroups_pay(p, n_slabs):
    """Whether the tight reservation, which lets more and smaller workgroups share a compute unit, is worth taking for
    tiles of ``p`` lanes a row: not where a wave walks one slab of two quads, 512 columns of 64-symbol segments,
    which is little beside its copy of the tables (two of 14853 x 512 at one, 32, 100 rows in 512 tiles of eight
    waves or 768 of six: 20.1 25.0 37.1 us, 21.8 26.6 38.1; 7609 and 5555 x 512 16.1 19.5 30.2, 17.1 20.9 31.6)."""
    return p > 8 or n_slabs > 1


def gain_to_ask(threads, tiles, k, lds, rows, cus=256):
    """What ``gemm_times`` has to promise (as a logarithm, over all row counts) before each of several
    tilings is taken in place of the last one, the slot model's choice, of a matrix of ``rows`` rows: 0.05, and
    0.08 where the workgroups are dealt less evenly to the compute units or have more waves.  Where the slot
    model's workgroups share units, the model makes their launch too slow, and it does not know that the
    sums of the parts of K are written and read once more.  There the lines are what measuring says of
    tilings below and above them (profiles/gemm_tilings.csv, 281 pairs; mean over 2 to 128 rows by the promise):
      fewer parts: 0.05, as above: 38 pairs from 0.084 on gain 4 to 44 %
      cut where the slot model does not cut: 0.147 +5 % (4506 x 2752), 0.132 -1 %, below -2 to -12 %; 0.168 +7 % (6144
        x 5120).  Never with three workgroups a unit (0.172 -2 %, 8232 x 3072), nor in more than two parts where ten
        waves or fewer share units above 64 rows too (0.136 -4 %, -20 % at 128 rows, 4837 x 2496)
      cut finer: 0.05 with up to 8192 sums a row of activations (0.117 +11 %, 1500 x 2064), else 0.165 (0.141 -7 %, 2932 x
        12160; 0.159 +3 %; 0.184 +5 %, 1483 x 9856)
      as many parts: 0.15 (0.088 -6 %, 15289 x 768; 0.198 +15 %, 7576 x 512), 0.05 for one workgroup a unit in place of
        two, 0.19 for one in place of three of eight waves, which fill the unit (0.188 -1 %, 16003 x 512)
    Of the 227 pairs that pass none loses in the mean; 13 % is gained, and 8 % lost at most at one row count.
    With 0.05 and 0.08 for all, 35 of 281 lost up to 12 % in the mean and up to 20 % at a row count."""
    at_once = np.maximum(1, np.minimum(np.minimum(GEMM_WAVES_PER_SIMD // -(-(threads // 64) // 4), lds_share(lds)), -(-tiles // cus)))
    even = tiles / (-(-tiles // cus) * cus)  # (the fit is least sure of workgroups dealt less evenly to the units)
    ask = np.where(even < even[-1], 0.08, 0.05)
    if at_once[-1] == 1:
        return np.where(threads > threads[-1], 0.08, ask)
    if k[-1] == 1:
        refused = (at_once[-1] >= 3) | ((threads[-1] <= 640) & (k > 2))
        finer = np.where(refused, np.inf, 0.165)
    else:
        finer = np.where(rows * k <= 8192, ask, 0.165)
    if at_once[-1] == 2:
        alike = np.where(at_once == 1, ask, 0.15)
    else:
        alike = np.where((threads[-1] >= 512) & (at_once == 1), 0.19, 0.15)
    return np.where(k > k[-1], finer, np.where(k < k[-1], ask, alike))


def plan_gemm_tiling(spr, class_rows, piece_cap_fn, lds_fn, cus=256, seg_len=64, table_bytes=0, split=False, unit_fn=None,
                     fitted=False):
    """Tiling of the GEMM kernel: workgroups of (row blocks of 16) x (quads of 4
    lane-segments) waves.  Same model as choose_tiling, counted in waves: a wave is busy
    for as long as its busiest lane, so idle lanes inside a wave are free, idle waves and
    idle CUs are not.  With ``split`` the launch may also be cut into k parts along K (every
    row tile k times, each copy walking a k-th of the slabs, the parts' sums added by a small
    second kernel): a matrix with few rows then fills the machine with full blocks of sixteen
    rows.  ``unit_fn()``: the LDS that the pieces of any sixteen rows take together, a fifth to a
    third less than sixteen of the longest; a tiling reserves that where it lets more workgroups
    share a compute unit.  ``fitted``: that choice against the one that ``gemm_times`` finds the fastest, taken
    where it is modelled 4 % faster at every row count and as much faster over them all as ``gain_to_ask`` says (us
    at 6, 20, 50, 100 rows, the slot model's choice and the fitted one: 5120 x 6144 36.1 38.5 41.1 61.4 / 32.7 36.2 40.2
    53.5, 2560 x 5120 23.2 26.0 28.0 33.4 / 19.4 22.3 24.9 32.3, 1024 x 5120 15.0 15.5 18.6 22.1 / 13.5 14.0 17.3 20.6,
    450 x 6144 15.1 15.7 18.8 22.5 / 12.3 12.7 16.3 19.4).  Returns (threads, lanes per row,
    rows per tile, slabs, tiles of the launch, piece capacity, LDS bytes, k, LDS bytes of a wave's pieces or 0)."""
    best, timed, whole_blocks = None, [], sum(-(-int(c) // 16) for c in class_rows)
    total_rows = sum(int(c) for c in class_rows)
    tile_counts = _tile_counts(class_rows, 1024)
    forced = os.environ.get("GEOREFINE_FUSED_GEMM_TILING")  # "lanes_per_row,rows[,k_parts]": experiments only
    if forced:
        values = [int(v) for v in forced.split(",")]
        choices = [(min(values[0], spr), values[1], values[2] if len(values) > 2 and split else 1)]
    else:
        choices = [(min(4 * quads, spr), 16 * blocks, k) for quads in range(1, -(-spr // 4) + 1)
                   for blocks in range(1, 17) if quads * blocks <= 16
                   for k in (GEMM_K_PARTS if split else (1,))]
    for p, r, k in dict.fromkeys(choices):
        row_blocks, quads, threads = gemm_shape(p, r)
        if threads > 1024:
            continue
        n_slabs = -(-spr // p)
        if k > n_slabs:
            continue
        cap = piece_cap_fn(p)
        by_waves = GEMM_WAVES_PER_SIMD // -(-(threads // 64) // 4)
        lds, unit = lds_fn(p, r, cap, 0), 0
        share = lds_share(lds)
        # (a quad's first segment is then a multiple of four, as in unit_fn's count)
        apart = share  # workgroups a unit where every piece has the LDS of the longest
        if share < by_waves and unit_fn is not None and (p % 4 == 0 or n_slabs == 1) and closer_workgroups_pay(p, n_slabs):
            tight = lds_fn(p, r, cap, unit_fn())
            if min(by_waves, lds_share(tight)) > share:
                lds, unit, share = tight, unit_fn(), lds_share(tight)
        if lds > MAX_LDS:
            continue
        per_cu = max(1, min(by_waves, share))
        slots = cus * per_cu
        rounds = -(-(tile_counts[r] * k) // slots)
        # Spread over idle workgroup slots, except a single block of rows where one workgroup has a
        # compute unit to itself, or where whole blocks take half of the slots at most: the block's
        # wave issues the same for fewer rows, and every further workgroup copies the tables (256
        # tiles of 13 or 15 rows against 192 and 256 of 16, 20 activation rows: 1024 x 5120 17.2
        # -> 16.2 us, 901 x 8192 20.1 -> 19.2; 257 tiles of one row against 17: 257 x 560 10.7 ->
        # 8.9).  Where they pay: 3000 x 3072, 512 tiles of 12 rows 21.2, 384 of 16 21.7.
        whole = row_blocks == 1 and (per_cu == 1 or 2 * tile_counts[r] * k <= slots)
        room = rounds * slots
        if spread_apart(tile_counts[r] * k, cus * apart, unit):
            room = cus * apart
        r_used = r if forced or whole else _spread_rows(tile_counts, r, room // k, floor=16 * (row_blocks - 1) + 1)
        tiles_used = tile_counts[r_used] * k
        slabs_each = -(-n_slabs // k)
        # work = lane-steps; capacity = every wave slot of every round for the whole walk
        work = total_rows * spr
        paid = rounds * slots * (threads // 64) * 16 * 4 * slabs_each
        waves = per_cu * (threads // 64)
        score = work / paid * min(1.0, waves / 24) * _walk_share(slabs_each, seg_len, table_bytes)
        if k > 1:  # the second kernel, and every part's sums written and read once more
            score *= 0.97 - 0.015 * k
        if best is None or score > best[0] + 1e-9:
            best = (score, threads, p, r_used, n_slabs, tiles_used, cap, lds_fn(p, r_used, cap, unit), k, unit)
        # (workgroups below eight waves copy the tables too often for the other model to be held to them)
        if fitted and threads >= 512 and p >= 8:
            r_used = r if row_blocks == 1 else r_used
            # (a taller tile's blocks are cut whole where a class allows, build_gemm_tiles)
            average = whole_blocks / tile_counts[r_used]
            if row_blocks == 1 or average > row_blocks - 1:  # (else spread so far that a block fewer holds them)
                timed.append((threads, p, r_used, n_slabs, tile_counts[r_used] * k, cap, lds_fn(p, r_used, cap, unit), k, unit,
                              1.0 if row_blocks == 1 else average))
    if best is None:
        raise FusedUnsupported("no GEMM tiling fits in LDS")
    if timed:
        taller = -(-best[3] // 16) > 1
        timed.append((*best[1:], whole_blocks * best[8] / best[5] if taller else 1.0))
        columns = [np.array(v) for v in zip(*timed)]
        threads, _, r, n_slabs, tiles, _, lds, k, _, blocks = columns
        times = np.log(gemm_times(threads, -(-r // 16), blocks, n_slabs, tiles, k, lds, spr, seg_len, table_bytes, cus))
        # (one tile of rows serves 2 to 16 of them, the others 17 to 32, 33 to 64, 65 to 128: three octaves and
        # one each)
        gain = times[:, -1:] - times
        total = np.array([3, 1, 1, 1]) / 6 @ gain
        total[(gain < 0.04).any(axis=0) | (total < gain_to_ask(threads, tiles, k, lds, total_rows, cus))] = 0.0
        # (of those that the model cannot tell apart the one with the fewest parts; and the slot model's choice
        # unless the gain is past what the fit is mostly wrong by between two tilings of one matrix)
        if total.max() > 0:
            return timed[min(np.flatnonzero(total >= total.max() - 0.02), key=lambda i: (k[i], -total[i]))][:9]
    return best[1:]


def order_residuals(raw, rows, cols, seg_len, block, position, held):
    """The packed 6-bit residuals of a frame (12-byte groups of 16 fields, frame order) in the
    order the tile walker reads them: rows at their positions, in blocks of ``block`` rows;
    inside a block by position in the segment, then by segment, then by row -- group t of
    segment s of position q at (((q // block * G + t) * spr + s) * block + q % block) * 12 with
    G = seg_len // 16.  A permutation of groups (no field is touched); positions that no row
    has hold zeros."""
    return order_records(raw, rows, cols, seg_len, block, position, held, 16, 12)


def order_index(values, rows, spr, block, position, held):
    """An index array of a frame (segment states or offsets, ``rows * spr + 1`` entries in the
    frame's order: the end of a segment is the entry after it) in the blocked order of the
    residuals: every row gets ``spr + 1`` entries of its own -- the last one is the end of its
    stream, i.e. the next row's first entry -- and entry s of position q goes to
    ``((q // block) * (spr + 1) + s) * block + q % block``.  The entries that a wave unit, or the
    sixteen rows of a matrix-core wave, read at one visit are then one run of bytes instead of a
    few bytes out of every row's own line.  Positions that no row has hold zeros."""
    values = np.asarray(values)
    per_row = np.empty((rows, spr + 1), dtype=values.dtype)
    per_row[:, :spr] = values[:rows * spr].reshape(rows, spr)
    per_row[:, spr] = values[spr::spr][:rows]
    ordered = np.zeros((held, spr + 1), dtype=values.dtype)
    ordered[position] = per_row
    return np.ascontiguousarray(ordered.reshape(held // block, block, spr + 1).transpose(0, 2, 1)).reshape(-1)


def order_records(raw, rows, cols, seg_len, block, position, held, record_symbols, record_bytes):
    """``order_residuals`` for records of another size: ``record_symbols`` consecutive symbols of a
    row in ``record_bytes`` bytes (the predictive codec's 32 five-bit residuals in 20 bytes, or
    the 32 four-bit reference bins in 16).  Record t of segment s of position q goes to
    (((q // block * U + t) * spr + s) * block + q % block) * record_bytes, U = seg_len //
    record_symbols; positions that no row has hold zeros."""
    spr, per_seg = cols // seg_len, seg_len // record_symbols
    raw = np.ascontiguousarray(raw, dtype=np.uint8)[:rows * spr * per_seg * record_bytes]
    position = np.ascontiguousarray(position, dtype=np.uint32)
    ordered = np.zeros(held * spr * per_seg * record_bytes, dtype=np.uint8)
    if raw.size != rows * spr * per_seg * record_bytes or _native.codec().grf_order_records(
            _native.ptr(raw, ctypes.c_uint8), rows, spr, per_seg, record_bytes, block, _native.ptr(position, ctypes.c_uint32),
            held, _native.ptr(ordered, ctypes.c_uint8)):
        raise ValueError("records do not fit the order")
    return ordered


def build_tiles(row_class, nr, r):
    """Rows grouped by class (index order inside a class), cut into tiles of r rows."""
    order = np.argsort(row_class, kind="stable").astype(np.uint32)
    counts = np.bincount(row_class, minlength=nr)
    tiles = -(-counts // r)
    out = np.full(int(tiles.sum()) * r, 0xFFFFFFFF, dtype=np.uint32)
    at = slot = 0
    for rho in np.flatnonzero(counts):
        cnt = int(counts[rho])
        out[slot:slot + cnt] = order[at:at + cnt]
        at += cnt
        slot += int(tiles[rho]) * r
    return out, np.repeat(np.arange(len(counts), dtype=np.uint8), tiles)


def build_balanced_tiles(row_class, nr, unit_rows, slots, max_rows):
    """Rows grouped by class (index order inside a class) into at most ``slots`` tiles whose
    heights are as equal as the classes allow: every class gets tiles in proportion to its
    rows -- one at least -- and cuts its rows into them evenly, in whole units of ``unit_rows``
    rows.  A launch is as long as its tallest tile; cut at one height for all classes, a frame
    whose classes differ widely in size (the row labels of a predictive frame) leaves workgroup
    slots empty or pays a second round for a few tiles.  Returns (tile_rows with stride R,
    tile_class, R) or None when no cut within ``slots`` tiles and ``max_rows`` rows exists."""
    order = np.argsort(row_class, kind="stable").astype(np.uint32)
    counts = np.bincount(row_class, minlength=nr)
    live = [rho for rho in range(nr) if counts[rho]]
    if not live or len(live) > slots:
        return None
    units = {rho: -(-int(counts[rho]) // unit_rows) for rho in live}
    tiles = {rho: 1 for rho in live}
    height = lambda rho: -(-units[rho] // tiles[rho])
    # the next tile to the class whose tiles are tallest (among equals: the fullest tiles, then the first class)
    order_of = lambda rho: (-height(rho), -units[rho] / tiles[rho], rho)
    queue = [order_of(rho) for rho in live]
    heapq.heapify(queue)
    for _ in range(slots - len(live)):
        rho = queue[0][2]
        if height(rho) <= 1:
            break
        tiles[rho] += 1
        heapq.heapreplace(queue, order_of(rho))
    tallest = max(height(rho) for rho in live) * unit_rows
    if tallest > max_rows:
        return None
    used = [min(tiles[rho], units[rho]) for rho in live]  # (tiles without a row are left out)
    out = np.full((sum(used), tallest), 0xFFFFFFFF, dtype=np.uint32)
    at = tile = 0
    for rho, n in zip(live, used):
        rows, u = int(counts[rho]), units[rho]
        # units per tile differ by at most one: u % n tiles of one more, then the rest
        tall, low = u % n, u // n * unit_rows
        split = min(tall * (low + unit_rows), rows)
        for first, height, count, t in ((0, low + unit_rows, split, tile), (split, low, rows - split, tile + tall)):
            if not count:
                continue
            whole = count // height
            out[t:t + whole, :height] = order[at + first:at + first + whole * height].reshape(whole, height)
            rest = count - whole * height
            if rest:
                out[t + whole, :rest] = order[at + first + whole * height:at + first + count]
        at += rows
        tile += n
    return out.reshape(-1), np.repeat(np.asarray(live, dtype=np.uint8), used), tallest


GEMM_BALANCE = os.environ.get("GEOREFINE_GEMM_BALANCE", "1") != "0"  # "0": tiles of one height (experiments)


def _blocks_paid(tile_rows, height):
    """Blocks of sixteen rows that the waves of a launch walk: every tile's rows rounded up."""
    held = (tile_rows.reshape(-1, height) != 0xFFFFFFFF).sum(axis=1)
    return int(((held + 15) // 16).sum())


def build_gemm_tiles(row_class, nr, r, first_tile=0, lead=0, cus=256):
    """Row tiles of the matrix-core kernel: (tile_rows, tile_class, R, tall tiles).

    A wave of that kernel holds a block of sixteen rows and issues the same instructions
    whether the block is full or holds four rows, so tiles cut at one height r that is not a
    multiple of 16 (68 rows: four blocks and a quarter) pay for a block they barely use.  The
    same number of tiles is cut in whole blocks instead, heights differing by one block (of
    1088 rows in 16 tiles: four tiles of 80 rows and twelve of 64), wherever that pays for
    fewer blocks; waves whose block is empty leave at once.  The tall tiles then decide the
    launch's length, so they should not share a compute unit: with every tile resident at
    once, workgroup i and workgroup i + cus land on the same unit, and the tall tiles are
    placed so that their launch positions (``first_tile`` + index) differ modulo ``cus``,
    starting at position ``lead`` (the tall tiles other members of a grouped launch have
    placed already)."""
    tile_rows, tile_class = build_tiles(row_class, nr, r)
    if not GEMM_BALANCE or r % 16 == 0:
        return tile_rows, tile_class, r, 0
    even = build_balanced_tiles(row_class, nr, 16, len(tile_class), 16 * -(-r // 16))
    # (as many tiles as planned: tiles shorter than a block that spread a small matrix over the
    # workgroup slots stay as they are)
    if even is None or len(even[1]) != len(tile_class) or _blocks_paid(even[0], even[2]) >= _blocks_paid(tile_rows, r):
        return tile_rows, tile_class, r, 0
    tile_rows, tile_class, r = even
    table = tile_rows.reshape(-1, r)
    height = ((table != 0xFFFFFFFF).sum(axis=1) + 15) // 16
    tall = height == height.max()
    n_tall = int(tall.sum()) if height.max() > height.min() else 0
    if n_tall:
        tall_at, short_at = np.flatnonzero(tall), np.flatnonzero(~tall)
        start = (lead - first_tile) % cus
        if start + n_tall > len(tile_class) or start > len(short_at):
            start = 0
        order = np.concatenate((short_at[:start], tall_at, short_at[start:]))
        table, tile_class = table[order], tile_class[order]
    return np.ascontiguousarray(table).reshape(-1), tile_class, r, n_tall


# Segments a wave of the row gather walks.  Fewer than a wave has lanes: more waves issue the table
# copy and hide each other's steps (8192 x 5120: 64 rows 13.3 -> 12.7 us, 2048 rows 34.4 -> 33.8, 777
# rows 17.2 -> 17.9); at 12 the waves' issue slots are the limit (777 rows: 30 us).
GATHER_LANES = 32


def lines_limit(rows, cols):
    """Up to how many times the GEMV's modelled time the whole-line tiling of a decode is taken (``FramePlan.lines_tiling``)."""
    return 1.25 if 2 * rows * cols >= 48 << 20 else 1.14


def fewer_lookups_pay(seg_len, spr, tiling, lds, gain):
    """Whether a predictive weight's matrix-core products take their small lookups, whose ``tiling`` uses
    ``gain`` times the share of the wave slots by ``plan_gemm_tiling``'s model: where that is half as much again,
    three workgroups of eight waves, all that a unit holds, share it, and their waves' quads leave at
    most a sixteenth of the lanes without a segment of 64 symbols.  Two, six and 96 rows, us, 64 / 16 KiB
    (profiles/predictive_lookups.csv, 229 matrices): 4096 x 4096 34.3 34.1 44.1 / 30.3 30.2 41.2, 16384 x 1024
    29.6 29.4 39.7 / 28.1 27.9 37.8, 8489 x 1984 30.8 30.4 39.0 / 29.1 28.7 38.5; not with shorter segments (4926 x 1952
    22.0 21.6 29.2 / 24.4 23.9 31.4), emptier slabs (8650 x 1856 29.7 29.3 37.6 / 32.9 32.2 41.8), seven waves (9821 x
    1728 29.9 29.4 38.0 / 32.4 31.9 42.4) or two workgroups (2048 x 8192 34.7 34.3 44.7 / 30.7 30.4 52.7)."""
    lanes = -(-tiling["lanes_per_row"] // 4) * 4 * tiling["n_slabs"]
    return (gain >= 1.5 and seg_len >= 64 and tiling["threads"] == 512 and tiling["n_tiles"] > 512 and lds_share(lds) >= 3
            and 16 * spr >= 15 * lanes)


class FramePlan:
    """Frame-level derived arrays (shared by every tiling) and a tiling factory."""

    def __init__(self, shape, nr, nc, row_class, main_freq, seg_states, seg_offsets, main_bytes, seg_len,
                 image=None, lut_budget=None):
        rows, cols = shape
        if rows * cols > 0xFFFFFFFF:
            raise FusedUnsupported("matrix too large")
        self.rows, self.cols, self.nr, self.nc, self.seg_len = rows, cols, nr, nc, seg_len
        self.spr = cols // seg_len
        self.shift = choose_shift(nc, lut_budget or LUT_BUDGET)
        self.lognb = 16 - self.shift
        self.lut, self.tab, self.tabn = sparse_tables(main_freq, nr, nc, self.shift, image)
        # a context that is one symbol of frequency 65536 (entry field 0): the kernels then keep the
        # scan that knows such entries
        self.whole_range = int((np.asarray(main_freq) >= 65536).any())
        self.seg_state = np.concatenate((seg_states, [1 << 23])).astype(np.uint32)
        self.seg_offset = np.concatenate((seg_offsets, [main_bytes])).astype(np.uint32)
        self.row_class = np.asarray(row_class)
        self.class_rows = np.bincount(self.row_class, minlength=nr)
        self._caps, self._tilings = {}, {}

    def for_vector_alus(self, main_freq, budget, image=None):
        """This plan, or one like it with lookups of at most ``budget`` bytes where the launches of
        the wave units (one row, the store sink) are the faster for them: where this plan's waves
        have more than a unit each and the smaller tables' tiling is modelled 14 % faster.  Fewer bytes
        mean more scans (of the predictive codec's wave steps 21 % at 32 KiB, 12 % at 64), and leave
        the LDS two workgroups a compute unit, which cut the rows finer.  One row and the store
        sink, us, predictive frames at 64 / 32 KiB, by units a wave and the modelled advantage:
          4096 x 4096   1.1 units, 1.35   31.8 34.3 / 27.5 29.0
          8192 x 4096   2.1 units, 1.23   43.0 51.3 / 39.2 49.3
          5120 x 8192   2.6 units, 1.17   48.4 57.2 / 48.6 56.9
          4096 x 11008  3.2 units, 1.15   53.8 62.2 / 49.1 60.0
          5120 x 17408  6.2 units, 1.10   92.2 112.5 / 92.9 117.7
          5120 x 5120   1.9 units, 1.10   34.7 41.7 / 35.6 45.6
          1024 x 1024   0.2 units, 1.16   11.7 11.3 / 13.8 13.2
          3000 x 4096   0.8 units, 1.11   21.2 22.9 / 25.2 26.9"""
        other = self.with_lookups(main_freq, budget, image)
        if other.lognb >= self.lognb:
            return self
        try:
            tall, fine = self.tiling(1, waves=True), other.tiling(1, waves=True)
        except FusedUnsupported:
            return self
        g = tall["scalars"]
        units = -(-g["rows_per_tile"] // (64 // g["lanes_per_row"])) * g["n_slabs"]
        gain = wave_time(tall, self.seg_len, self.table_bytes()) / wave_time(fine, self.seg_len, other.table_bytes())
        return other if units > g["threads"] // 64 and gain >= 1.14 else self

    def for_matrix_cores(self, main_freq, budget, image=None):
        """This plan, or one like it with lookups of at most ``budget`` bytes where the matrix-core
        launches of the matrix are the faster for them (``fewer_lookups_pay``).  Fewer bytes mean more scans,
        13 % of the same tiling's time, and let three workgroups share a unit that had one.  A grouped launch keeps
        this plan's (three of 4096 x 4096 at six, 32 and 96 rows: 67.2 69.2 96 us / 72.6 74.8 125)."""
        other = self.with_lookups(main_freq, budget, image)
        if other.lognb >= self.lognb:
            return self
        try:
            tall, fine = self.gemm_tiling(), other.gemm_tiling()
        except FusedUnsupported:
            return self
        gain = other.gemm_share(fine) / self.gemm_share(tall)
        return other if fewer_lookups_pay(self.seg_len, self.spr, fine["scalars"], fine["lds"], gain) else self

    def gemm_share(self, tiling):
        """What ``plan_gemm_tiling``'s model says of one tiling: the share of the machine's wave slots that do
        useful steps."""
        g = tiling["scalars"]
        waves, k = g["threads"] // 64, max(1, g["k_parts"])
        per_cu = max(1, min(GEMM_WAVES_PER_SIMD // -(-waves // 4), lds_share(tiling["lds"])))
        slabs, slots = -(-g["n_slabs"] // k), 256 * per_cu
        paid = -(-g["n_tiles"] // slots) * slots * waves * 64 * slabs
        share = self.rows * self.spr / paid * min(1.0, per_cu * waves / 24) * _walk_share(slabs, self.seg_len, self.table_bytes())
        return share * (0.97 - 0.015 * k) if k > 1 else share

    def with_lookups(self, main_freq, budget, image=None):
        """This plan with lookups of at most ``budget`` bytes."""
        other = copy.copy(self)
        other.shift = choose_shift(self.nc, budget)
        other.lognb = 16 - other.shift
        other.lut = sparse_tables(main_freq, self.nr, self.nc, other.shift, image)[0]
        other._tilings = {}
        return other

    def residual_order(self, block=None):
        """(block rows B, row positions u32[rows], rows of the array) of the resident residual
        order: the rows by class, index order inside a class, as every tiling takes them, each
        class starting on a multiple of 16; B = the rows of a wave unit of the GEMV (1 where
        the GEMV has no wave tiling), so that a unit's rows are the rows of one block -- or the
        ``block`` asked for (1, 2, 4, 8, 16): 16 makes a wave of the matrix-core kernel, which
        holds sixteen rows, read whole lines, for matrices that are served in batches."""
        if block is not None:
            if block not in (1, 2, 4, 8, 16):
                raise FusedUnsupported("residual blocks have 1, 2, 4, 8 or 16 rows")
        else:
            try:
                block = 64 // self.tiling(1, waves=True)["scalars"]["lanes_per_row"]
            except FusedUnsupported:
                block = 1
        order = np.argsort(self.row_class, kind="stable")
        starts = np.zeros(self.nr + 1, dtype=np.int64)
        for rho in range(self.nr):
            starts[rho + 1] = (starts[rho] + int(self.class_rows[rho]) + 15) // 16 * 16
        first = np.concatenate(([0], np.cumsum(self.class_rows)[:-1]))  # of each class, in `order`
        sorted_class = self.row_class[order]
        position = np.empty(self.rows, dtype=np.uint32)
        position[order] = (starts[sorted_class] + np.arange(self.rows) - first[sorted_class]).astype(np.uint32)
        return block, position, int(starts[-1])

    def table_bytes(self):
        """LDS bytes of one row class's lookup tables (what every workgroup copies first)."""
        return self.nc * (((self.tabn + 1) * 8 + 15) // 16 * 16 + (1 << self.lognb))

    def scalars(self):
        return dict(rows=self.rows, cols=self.cols, nr=self.nr, nc=self.nc, seg_len=self.seg_len,
                    segs_per_row=self.spr, shift=self.shift, lognb=self.lognb, tabn=self.tabn,
                    whole_range=self.whole_range)

    def quad_cap(self):
        """Capacity of the row pieces of the GEMM's waves (four segments)."""
        if "quad" not in self._caps:
            self._caps["quad"] = quad_piece_capacity(self.seg_offset, self.rows, self.spr)
        return self._caps["quad"]

    def quad_bytes(self):
        """LDS bytes that the pieces of four segments of any sixteen rows that follow one another in a
        class take, one behind the other in 16-byte units (``grf_unit_pieces``)."""
        if "quads" not in self._caps:
            order = np.argsort(self.row_class, kind="stable").astype(np.uint32)
            most = ctypes.c_uint32()
            if _native.codec().grf_unit_pieces(_native.ptr(self.seg_offset, ctypes.c_uint32), self.rows, self.spr,
                                               _native.ptr(order, ctypes.c_uint32), 4, 16, ctypes.byref(most)):
                raise FusedUnsupported("index offsets")
            self._caps["quads"] = 16 * most.value
        return self._caps["quads"]

    def _cap(self, p):
        if p not in self._caps:
            self._caps[p] = piece_capacity(self.seg_offset, self.rows, self.spr, p)
        return self._caps[p]

    def tiling(self, m, waves=False):
        """Host arrays and scalars of a ``grf_fused_tiling`` sized for m activation rows
        (m = 0: the store sink).  ``waves``: the wave-unit scheme of the GEMV, one tiling for
        every row count (launches carry at most two rows each)."""
        if waves and m:
            key = "waves", os.environ.get("GEOREFINE_FUSED_WAVE_TILING")
            if key not in self._tilings:  # (one for every row count; the residual order asks for it too)
                self._tilings[key] = self._wave_tiling()
            return self._tilings[key]
        threads, p, r, n_slabs, n_tiles, cap, lds = choose_tiling(
            self.spr, self.class_rows, self._cap,
            lambda p_, r_, cap_: lds_bytes(self.nc, self.lognb, self.tabn, m, p_, self.seg_len, r_, cap_),
            seg_len=self.seg_len, table_bytes=self.table_bytes())
        tile_rows, tile_class = build_tiles(self.row_class, self.nr, r)
        assert len(tile_class) == n_tiles
        return dict(tile_rows=tile_rows, tile_class=tile_class,
                    scalars=dict(threads=threads, lanes_per_row=p, rows_per_tile=r, n_slabs=n_slabs,
                                 n_tiles=n_tiles, piece_cap=cap, scheme=SCHEME_SLABS), lds=lds)

    def lines_tiling(self):
        """The wave units of the kernel that stores whole lines (HOLD 2 of fused_wave_store_kernel), which
        holds 64 columns back and has registers for sixteen waves a compute unit: workgroups of
        sixteen or eight.  None where the walk's segments are no multiple of 64, and where the
        model's time with sixteen waves is too far above the GEMV's with twenty-four: 1.25 times it where the
        result is 48 MiB or more, which the caches do not take up beside what is read, else 1.14 times.  us,
        four results written in turn, the GEMV's tiling and this one (profiles/whole_lines.csv, 125 matrices): from
        48 MiB 1.20 5120 x 17408 109.0 93.1, 1.085 5120 x 6144 44.7 41.3, 1.24 8658 x 3904 47.2 42.0 (one result over and
        over, which stays in the last-level cache, 33.1 35.4 for 5120 x 6144); below 1.13 621 x 13696 20.9 18.3, 1.07
        4096 x 4096 20.8 21.5, 1.16 1062 x 16384 25.0 25.8, 1.19 3177 x 5760 25.6 27.6, 1.25 11580 x 2048 28.5 33.0."""
        if self.seg_len % 64:
            return None
        key = "lines", os.environ.get("GEOREFINE_FUSED_WAVE_TILING")
        if key not in self._tilings:
            lines, walk = self._wave_tiling(0, LINES_WAVES_PER_CU), self.tiling(WAVE_ROWS_PER_PASS, waves=True)
            slower = (wave_time(lines, self.seg_len, self.table_bytes(), waves=LINES_WAVES_PER_CU)
                      > lines_limit(self.rows, self.cols) * wave_time(walk, self.seg_len, self.table_bytes()))
            self._tilings[key] = None if slower and not key[1] else lines
        return self._tilings[key]

    def _wave_tiling(self, m=WAVE_ROWS_PER_PASS, waves=WAVES_PER_CU):
        self._wave_limits()
        threads, p, r, n_slabs, n_tiles, cap, lds = choose_wave_tiling(
            self.spr, self.class_rows, self._cap,
            lambda t_, p_, r_, s_, cap_: lds_bytes_waves(self.nc, self.lognb, self.tabn, m, t_, p_, r_, s_, cap_),
            seg_len=self.seg_len, table_bytes=self.table_bytes(), waves=waves)
        tile_rows, tile_class = build_tiles(self.row_class, self.nr, r)
        assert len(tile_class) == n_tiles
        if not os.environ.get("GEOREFINE_FUSED_WAVE_TILING"):
            # classes of very different sizes: the same workgroup slots, cut so that no tile is
            # taller than it has to be (the kernel walks a tile's real height)
            nwaves, rpw = threads // 64, 64 // p
            per_cu = max(1, min(waves // nwaves, lds_share(lds)))
            slots = -(-n_tiles // (256 * per_cu)) * 256 * per_cu
            even = build_balanced_tiles(self.row_class, self.nr, rpw, slots, r)
            if even is not None and (even[2] < r or (even[2] == r and len(even[1]) > n_tiles)):
                tile_rows, tile_class, r = even
                n_tiles = len(tile_class)
                lds = lds_bytes_waves(self.nc, self.lognb, self.tabn, m, threads, p, r, n_slabs, cap)
        return dict(tile_rows=tile_rows, tile_class=tile_class,
                    scalars=dict(threads=threads, lanes_per_row=p, rows_per_tile=r, n_slabs=n_slabs,
                                 n_tiles=n_tiles, piece_cap=cap, scheme=SCHEME_WAVES), lds=lds)

    def gather_shape(self):
        """(segments a wave walks, piece capacity) of the row gather: every requested row has a
        workgroup of its own, which walks all of the row's segments at once where it has the lanes."""
        waves = min(16, -(-self.spr // GATHER_LANES))
        lanes = min(64, -(-(-(-self.spr // waves)) // 4) * 4)  # dealt evenly, whole quads
        cap = self._cap(min(self.spr, lanes))
        if (self.table_bytes() + 15) // 16 * 16 + waves * cap > MAX_LDS:
            raise FusedUnsupported("gather tile does not fit in LDS")
        return lanes, cap

    def _wave_limits(self):
        """Kernels over wave tilings address rows and segments with 24-bit multiplies."""
        if self.rows + 16 + 16 * self.nr >= 1 << 24 or self.cols >= 1 << 24:  # (row positions stay below 2^24 too)
            raise FusedUnsupported("wave tilings take fewer than 2^24 rows and columns")

    def gemm_tiling(self, fitted=None):
        """The one tiling every fused GEMM launch uses, whatever its row count: the order in
        which an output element accumulates follows the tiling, so it must not change with M.
        ``fitted`` (default: for the context codec): may be ``gemm_times``' choice.  The fit is the context
        codec's; predictive frames with lookups of 64 KiB, a workgroup a unit, gain by it as well (1024 x
        4096 at six and 96 rows 18.5 24.6 -> 15.9 22.1 us, 512 x 8192 18.5 26.2 -> 16.8 24.1, 1000 x 16384
        40.1 56.4 -> 35.0 48.3; eight others keep their tiling).  Planned once for a matrix and its clones: it
        takes 1.7 ms, a third more than before there was a fit, and a predictive tensor's first product paid for it."""
        fitted = GEMM_SPLIT and (self.nc <= 4 if fitted is None else fitted)
        key = "gemm", fitted, GEMM_SPLIT, GEMM_BALANCE, GEMM_WAVES_PER_SIMD, os.environ.get("GEOREFINE_FUSED_GEMM_TILING")
        if key not in self._tilings:
            self._tilings[key] = self._gemm_tiling(fitted)
        return self._tilings[key]

    def _gemm_tiling(self, fitted):
        self._wave_limits()
        threads, p, r, n_slabs, n_tiles, cap, lds, k, unit = plan_gemm_tiling(
            self.spr, self.class_rows, lambda lanes: self.quad_cap(),
            lambda p_, r_, cap_, unit_: lds_bytes_gemm(self.nc, self.lognb, self.tabn, p_, r_, cap_, unit_),
            seg_len=self.seg_len, table_bytes=self.table_bytes(), split=GEMM_SPLIT, unit_fn=self.quad_bytes, fitted=fitted)
        # the row tiles; the launch has k of each
        tile_rows, tile_class, r, _ = build_gemm_tiles(self.row_class, self.nr, r)
        threads = gemm_shape(p, r)[2]  # (classes that fit fewer blocks of sixteen rows than were planned)
        n_tiles = len(tile_class) * k
        lds = lds_bytes_gemm(self.nc, self.lognb, self.tabn, p, r, cap, unit)
        return dict(tile_rows=tile_rows, tile_class=tile_class,
                    scalars=dict(threads=threads, lanes_per_row=p, rows_per_tile=r, n_slabs=n_slabs,
                                 n_tiles=n_tiles, piece_cap=cap, scheme=SCHEME_WAVES, k_parts=k, wave_bytes=unit), lds=lds)


def plan_group(plans, m=None, gemm=False, waves=False, mixed=False):
    """Tilings of several frames of one width for one grouped launch: planned as if the
    members' row classes belonged to one matrix (so a small member's tiles fill the
    workgroup slots a large one leaves), with one thread count, lanes per row and rows per
    tile for all; returns one tiling (as ``FramePlan.tiling``) per member.

    ``mixed``: the members may be indexed at different segment lengths (what ``choose_segment``
    gives siblings of different sizes); the length of the member with the most rows sets the
    pace, the others walk theirs in more slabs or fewer.  One and eight rows, us: 2048 + 512 + 512 x
    2048 at 32, 16, 16 15.0 17.0, all at 32 14.8 19.8, a launch each 30.5 39.6; 2560 + 2048 x 5120 at
    64, 32 30.7 41.4, both at 64 33.1 43.0; 1536 + 512 x 4096 at 32, 16 16.3 24.2, both at 32 15.1
    26.6 (the one case of seven where one row is slower for the mixture)."""
    first = max(plans, key=lambda pl: pl.rows)
    if any(pl.cols != first.cols or (pl.seg_len != first.seg_len and not mixed) for pl in plans):
        raise FusedUnsupported("group members need one width and one segment length")
    class_rows = np.concatenate([pl.class_rows for pl in plans])
    cap_fn = lambda lanes: max(pl._cap(lanes) for pl in plans)
    table = max(pl.table_bytes() for pl in plans)
    slabs = lambda pl, lanes: -(-pl.spr // lanes)
    scheme = SCHEME_SLABS
    if gemm or waves:
        for pl in plans:
            pl._wave_limits()
    if gemm:
        scheme = SCHEME_WAVES
        lds_fn = lambda p_, r_, cap_, unit_: max(lds_bytes_gemm(pl.nc, pl.lognb, pl.tabn, p_, r_, cap_, unit_) for pl in plans)
        quad_cap = max(pl.quad_cap() for pl in plans)
        plan = dict(seg_len=first.seg_len, table_bytes=table)
        if all(pl.spr == first.spr for pl in plans):
            threads, p, r, _, _, cap, lds, _, unit = plan_gemm_tiling(first.spr, class_rows, lambda lanes: quad_cap, lds_fn, **plan,
                                                                      unit_fn=lambda: max(pl.quad_bytes() for pl in plans))
        else:  # (lanes per row follow the first member's length: a slab of another's may begin between two quads)
            threads, p, r, _, _, cap, lds, _ = choose_gemm_tiling(first.spr, class_rows, lambda lanes: quad_cap,
                                                                  lambda p_, r_, cap_: lds_fn(p_, r_, cap_, 0), **plan)
            unit = 0
    elif waves:
        scheme = SCHEME_WAVES
        seg_lens = list(dict.fromkeys(pl.seg_len for pl in [first, *plans]))
        lengths = [(first.cols // n, n, np.concatenate([pl.class_rows for pl in plans if pl.seg_len == n])) for n in seg_lens]
        lds_fn = lambda t_, p_, heights, cap_: max(
            lds_bytes_waves(pl.nc, pl.lognb, pl.tabn, WAVE_ROWS_PER_PASS, t_, p_, heights[seg_lens.index(pl.seg_len)],
                            slabs(pl, p_), cap_) for pl in plans)
        forced = os.environ.get("GEOREFINE_FUSED_WAVE_TILING")  # "threads,lanes_per_row,rows": experiments only
        if forced:
            threads, p, r = (int(v) for v in forced.split(","))
            heights, cap = [r] * len(seg_lens), cap_fn(p)
            lds = lds_fn(threads, p, heights, cap)
        else:
            threads, p, heights, _, cap, lds = search_wave_tilings(lengths, cap_fn, lds_fn, 256, table)
        height_of = dict(zip(seg_lens, heights))
    else:
        lds_fn = lambda p_, r_, cap_: max(lds_bytes(pl.nc, pl.lognb, pl.tabn, m, p_, pl.seg_len, r_, cap_) for pl in plans)
        threads, p, r, _, _, cap, lds = choose_tiling(first.spr, class_rows, cap_fn, lds_fn,
                                                      seg_len=first.seg_len, table_bytes=table)
    tilings = []
    if gemm:  # whole blocks of sixteen rows per tile; one slot stride and LDS demand for all members
        cut, at, lead = [], 0, 0
        for pl in plans:
            cut.append(build_gemm_tiles(pl.row_class, pl.nr, r, first_tile=at, lead=lead))
            at, lead = at + len(cut[-1][1]), lead + cut[-1][3]
        height = max(c[2] for c in cut)
        lds = lds_fn(p, height, cap, unit)
        for pl, (tile_rows, tile_class, r_, _) in zip(plans, cut):
            if r_ != height:  # (a member the cut did not pay for: its slots widened to the common stride)
                wide = np.full((len(tile_class), height), 0xFFFFFFFF, dtype=np.uint32)
                wide[:, :r_] = tile_rows.reshape(-1, r_)
                tile_rows = wide.reshape(-1)
            tilings.append(dict(tile_rows=tile_rows, tile_class=tile_class,
                                scalars=dict(threads=threads, lanes_per_row=p, rows_per_tile=height, n_slabs=slabs(pl, p),
                                             n_tiles=len(tile_class), piece_cap=cap, scheme=scheme, wave_bytes=unit), lds=lds))
        return tilings
    for pl in plans:
        height = height_of[pl.seg_len] if waves else r
        tile_rows, tile_class = build_tiles(pl.row_class, pl.nr, height)
        tilings.append(dict(tile_rows=tile_rows, tile_class=tile_class,
                            scalars=dict(threads=threads, lanes_per_row=p, rows_per_tile=height, n_slabs=slabs(pl, p),
                                         n_tiles=len(tile_class), piece_cap=cap, scheme=scheme), lds=lds))
    return tilings


VALIDATE_USES = {"decode": 0, "gemv": 1, "gemm": 2, "gather": 3}


def validate_host(plan, tiling, use, *, row_pos=None, block=0, main_bytes=None):
    """The device library's host-side validator (``grf_bctx_fused_validate_host``) on a plan and
    one of its tilings (as ``FramePlan.tiling`` / ``gemm_tiling`` return them): what the kernels
    take on trust from the index and the tiling arrays -- offsets in order and inside the
    stream, every staged piece within ``piece_cap``, rows and classes of the tiles, the LDS
    demand.  Needs no GPU.  Raises ``FusedUnsupported`` with the library's message."""
    import ctypes
    from . import _hip_abi, _native
    lib = _native.hip()
    f = _hip_abi.GrfBctxFused()
    for key, value in plan.scalars().items():
        setattr(f, key, value)
    f.main_n_bytes = int(plan.seg_offset[-1]) if main_bytes is None else main_bytes
    f.raw_interleaved = block
    g = _hip_abi.GrfFusedTiling()
    for key, value in tiling["scalars"].items():
        setattr(g, key, value)
    offsets = plan.seg_offset
    if block:  # the library reads the index in the order the frame structure declares
        if row_pos is None:
            raise FusedUnsupported("the blocked order needs the rows' positions")
        held = -(-(int(np.max(row_pos)) + 1) // block) * block
        offsets = order_index(offsets, plan.rows, plan.spr, block, row_pos, held)
    arrays = [np.ascontiguousarray(offsets, dtype=np.uint32),
              np.ascontiguousarray(tiling["tile_rows"], dtype=np.uint32),
              np.ascontiguousarray(tiling["tile_class"], dtype=np.uint8),
              np.ascontiguousarray(plan.row_class, dtype=np.uint8),
              None if row_pos is None else np.ascontiguousarray(row_pos, dtype=np.uint32)]
    status = lib.grf_bctx_fused_validate_host(ctypes.byref(f), ctypes.byref(g), VALIDATE_USES[use],
                                              *[a.ctypes.data if a is not None else None for a in arrays])
    if status:
        raise FusedUnsupported(lib.grf_last_error().decode(errors="replace"))
