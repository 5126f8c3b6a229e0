"""``x @ W^T + b`` for a Linear's weight ``[out, in]``, and its fused forms.

float32: the hand-written true-float32 kernels, always (the gated unit in their
epilogue; of up to ``ops.F32_FEW_ROWS`` rows also the norm in front and the add into the stream).  bfloat16 with up to
``FUSED_ROWS`` rows (decode steps, the output head), and up to 64 or 128 rows where
it is the faster one (a small weight, a long K): the hand-written
matrix-core kernels that stream the weight once and take over their neighbours'
work: a SiLU-gate behind (``epilogue="silu"``), the add into the float32
residual stream (``into=residual``), or float32 results for the logits.  They
come in two forms: waves that share K and own all rows (few rows; the q/k/v and
o_proj products, logits of up to 3 rows and narrow float32 results), and waves that
own columns and share the rows through LDS (the SiLU-gate product up to 96 rows, every
product whose K is cut, logits of 4 to 96 rows).
bfloat16 with more rows, and from ``FEW_TILE_ROWS`` or 17 rows on (``cut_tiles``, ``gate_tiles``;
``part_tiles``): tiles of this package's own (``csrc/gemm_direct.hip``, and
``csrc/gemm_tiles.hip`` for a K that is no multiple of 64) where they are the faster ones, else the
vendor library's product (hipBLASLt through a thin cached interface of this
package), as the reference leaves its products to a library
(src/cloud_engine/model.py:89-137), with the small kernels around it.
"""

from __future__ import annotations

import functools
import math
import weakref
from dataclasses import dataclass
from typing import Any, NamedTuple, Optional, Union

import torch

from ..kernels import ops

# Rows up to which the hand-written fused bf16 kernel replaces the library product.  Measured on
# MI355X (3B shapes): up to 16 rows it beats the library by 1.5-2x; with 17 to 64 rows it wins where K
# is long and is cut into parts (the down product: 17-20 us against the library's 27-32 us); its gate/up
# product loses from 32 rows on (34 us against 26 + 5 us at 64 rows: every workgroup re-reads the rows of A).
FUSED_ROWS = 16
# ... and up to 128 rows (the down product alone, weight from memory, own kernel against the library, us: 3B shape at
# 72 / 96 / 128 rows 18.3 / 19.9 / 24.2 against 27.7 / 28.4 / 28.4; 7B 41.6 / 45.8 / 54.4 against 96 / 95 / 84; 14B
# 36.3 / 39.8 / 48.2 against 50.0 / 61.6 / 60.9: the library has no good algorithm for a long K and few rows, and at
# row counts that do not recur it takes its heuristic's first choice)
FUSED_PARTS_ROWS = 128
# With 17 to 128 rows it also wins where the weight is small (q/k/v and o_proj of the 3B shape at 32 / 64 / 96 rows: 7.7 / 9.3 /
# 9.4 us and 7.4 / 7.7 / 9.0 against the library's 12-18 us inside a step at up to 64 rows and 9.1-12.4 beyond;
# and the rotation, the cache write, the residual add and the next
# norm ride along); from about 6M weight values on the library is faster (7B o_proj at 64 rows: 12.6 us against
# 11.1 us).
FUSED_SMALL_ROWS = 128
FUSED_SMALL_WEIGHT = 6 << 20
# float32 logits of more rows than this go to the library (the hand-written kernel streams the weight once per
# 64 rows; up to 64 rows it is one pass either way)
FUSED_LOGIT_ROWS = 64
# An ``into=`` product with fewer than this many 16-column tiles and a K of at least ``PART_MIN_K`` cuts K
# into parts for more workgroups (each part adds its products into the stream with atomic adds; ``plan_shared_parts``).
PART_BELOW_TILES = 512
PART_MIN_K = 4096
PART_K = 1024           # the shortest stretch of K a part takes
# ... and of a product that has at least this many workgroups side by side (narrower ones were not measured).  896 columns,
# K 4,864, us: 4 parts 7.2 at 8 rows, 13.7 at 96; 8 parts 5.4, 10.2; 10 parts 4.7, 8.8; 16 parts 4.8, 9.7.  1,536 columns,
# K 8,960: 8 parts 8.3, 16.0; 10 parts 7.5, 15.4.
PART_K_WIDE, PART_WIDE_BLOCKS = 512, 8


def cuts_k(n: int, k: int) -> bool:
    """Whether a product of few rows that joins the stream has its K cut, so that it is added in no fixed order."""
    return -(-n // 16) < PART_BELOW_TILES and k >= PART_MIN_K


# SiLU-gate products of up to this many rows take the form whose waves own columns and share the rows of A
# through LDS (gate/up of the 3B shape at 32 / 64 rows: 19 / 22.5 us against the library's 26 / 27 us and 5 us
# for the SiLU kernel behind it; 14B: 50 / 56 against 55 / 62 + 6; 7B: level); from 65 to 96 rows, on six row tiles
# (3B / 7B / 14B at 72 rows: 28.3 / 67.7 / 63.7 us against 31.4 / 75.2 / 70.4 for the library and its SiLU kernel,
# at 96 rows 29.6 / 69.6 / 65.0 against 32.2 / 71.1 / 64.6); beyond that the library is level or ahead (3B at 128
# rows: 35 against 30 + 5 us; 7B: 111 against 66).
SHARED_SILU_ROWS = 96
# Float32 results take that form at 17 to 80 rows (the head of the 3B shape at 64 rows 137 us, 169 in the form whose waves share
# K), and with fewer or more rows where the columns give each unit a workgroup (of 128 columns) all the time: what the form
# takes is what its fullest unit takes, and a narrow product leaves the others idle while one workgroup walks all of K.
# us, the form whose waves share K and this one, K 2,048, 4 / 8 / 16 rows:
#   columns      32  4.2, 11.2 / 4.4, 11.2 / 4.8, 11.2       2,048 (K 4,096)  7.6, 24.0 / 8.1, 24.2 / 9.4, 24.4
#            32,768  27.5, 25.3 / 28.2, 25.2 / 29.6, 24.6 (one turn of 256 units)       40,000 (two turns, 61 % of them)
#                    31.4, 36.0 / 32.4, 36.1 / 35.1, 35.6       65,536 (two turns)  49.4, 48.3 / 50.5, 47.2 / 55.8, 47.1
#            73,728 (three turns, 75 %)  56.4, 57.5 / 58.1, 58.0 / 66.8, 59.0       152,064 (93 %)  111, 110 / 114, 111 / 132, 115
# Hence the share of the turns' units that must have work, up to so many rows:
SHARED_LOGIT_FILL = ((3, None), (8, 0.9), (16, 0.75), (80, 0.0))
# The library and this one, 81 / 96 rows: 32 columns 6.0, 25.2 / 5.9, 25.3; 32,768 (K 1,024) 18.5, 19.5 / 17.8, 19.9; 50,304
# (K 4,096) 103, 96 / 105, 98, (K 5,120) 106, 123 / 106, 125; 65,536 (K 1,024, 4,096, 5,120) 37, 34, 131, 109, 126, 139 at 81;
# 152,064 166, 144 / 168, 147, (K 5,120) 342, 320 / 331, 327: from so many turns on, up to and beyond this K.
SHARED_LOGIT_ROWS, SHARED_LOGIT_TURNS, SHARED_LOGIT_K = 96, (2, 4), 4096


@functools.lru_cache(maxsize=4096)
def _shares_rows_f32(rows: int, n: int, k: int, units: int) -> bool:
    groups = -(-n // 128)
    for upto, fill in SHARED_LOGIT_FILL:
        if rows <= upto:
            return fill is not None and groups >= fill * units * -(-groups // units)
    return rows <= SHARED_LOGIT_ROWS and groups >= SHARED_LOGIT_TURNS[k > SHARED_LOGIT_K] * units


def shares_rows_f32(rows: int, n: int, k: int) -> bool:
    """Whether a float32 result of ``rows`` rows and ``n`` columns takes the shared-rows form."""
    return _shares_rows_f32(rows, n, k, ops.compute_units())


def plan_shared_silu(pairs: int) -> tuple[int, bool]:
    """Waves per workgroup (each wave takes one gate tile and its up tile) for the shared-rows SiLU product,
    and whether every workgroup then has a compute unit of its own.  A compute unit streams at most some
    30 GB/s however many loads it has under way, so what counts is the most pairs that meet on one unit:
    workgroups of four waves, or of three where that needs fewer turns (688 pairs of the 3B shape: 172
    workgroups of four or 230 of three, one turn each; 1,184 of the 7B shape: two turns of four waves or
    two of three, 70 against 61 us at 64 rows; 864 of the 14B shape: one turn of four, 56 against 81 us)."""
    best = None
    units = ops.compute_units()
    for waves in (4, 3, 2):
        turns = -(-(-(-pairs // waves)) // units)
        if best is None or turns * waves < best[0]:
            best = (turns * waves, waves, turns == 1)
    return best[1], best[2]


def plan_shared_parts(tiles: int, k: int) -> tuple[int, int, int]:
    """(column tiles per wave, waves, parts of K) of a cut product in the shared-rows form: workgroups of four
    waves, one tile of 16 columns per wave (two for a wide result), and as many parts as give about one
    workgroup per compute unit.  Measured at 8 / 64 rows (us; the form of waves that share K, at its best
    cut, beside it): 128 tiles, K 11,008: 8 parts 11.0 / 14.8 (13.2 / 17.7); 224 tiles, K 18,944: 4 parts
    26.1 / 35.3 (29.7 / 43.8); 320 tiles, K 13,824, two tiles per wave: 4 parts 28.6 / 38.7 (30.0 / 44.0)."""
    units = ops.compute_units()
    column_tiles = 1 if tiles <= units else 2
    waves = 4
    blocks = -(-tiles // (column_tiles * waves))
    most = -(-k // PART_K_WIDE) if blocks >= PART_WIDE_BLOCKS else k // PART_K
    parts = max(1, min(units // blocks, 16, most))
    stretch = -(-(-(-k // parts)) // 128) * 128  # (what the kernel gives a part: whole slices, and none a part without k)
    return column_tiles, waves, -(-k // stretch)


# Products of more rows than the kernels above take (beyond ``FUSED_PARTS_ROWS``) go to tiles of this package or to the
# vendor library, whichever the models below say is faster: the tiles that load straight into LDS (``DIRECT_US``) where K is a
# multiple of 64, else those of csrc/gemm_tiles.hip (``TILE_US``), each against the one model of the library.
# ``TILE_US`` and the library's are fitted to 608 products timed inside captured chains on MI355X with the kernels between them
# (q/k/v, o_proj, gate/up and down of six shapes from 896 to 8,192 wide, at 16 to 30 row counts from 130 to 2,048).  Their K are
# multiples of 64, which these tiles no longer see; any other K takes them as many slices as the next multiple.
# Those tiles (within 6 % of the measured, root mean square), us: a start, and per slice of 64 k of a workgroup alone on its unit
# and of every further one that meets it there (what bounds them is the rate at which a unit is fed from its L2, some 20 bytes
# a cycle, hence the advantage of large tiles where they are many).  The tiles are dealt to the 8 XCDs in equal runs and each
# XCD has an eighth of the units: 33 workgroups on one of them take two turns, though there are fewer than 256 in all.
TILE_US = {(64, 64): (4.9, 0.251, 0.233), (128, 64): (6.1, 0.405, 0.346), (128, 128): (7.8, 0.628, 0.525),
           (128, 256): (9.5, 0.880, 1.04)}
TILE_PARTS = (1, 2, 3, 4, 6, 8)
TILE_PARTS_US = 0.356  # parts of K: float32 sums written by the product and read by the norm, us per MB
XCDS = 8
# The library (within 12 %; it takes its first choice of algorithm for a row count that does not recur, now and then a bad
# one: 7B down at 400 rows 200 us where this says 114 and the tiles take 81; 1,999 rows x 6,144 and 4,736, K 2,048, inside a
# prompt 57 and 55 where it says 41 and 33): the way through one tile's K and its weight rows
# (us, per 1,000 k, per million weights), and the products at a rate (PFLOP/s) that goes by the tiles of 128 x 128 a unit.
LIBRARY_US = (8.6, 1.0, 0.40)
LIBRARY_RATE, LIBRARY_MOST = 0.85, 1.32
LIBRARY_TUNED = (1.0, 0.90, 0.85)  # ... and its share of that where its candidates, or all its algorithms, were timed


@dataclass(frozen=True, eq=False)
class Behind:
    """What the library's product costs beyond what the tiles and their epilogue do.  ``us`` and ``us_per_million`` numbers of
    the product: the kernel behind it, or the branch that is rounded, written and read again.  ``host_us``: a step of more
    than 128 rows runs launch by launch, and where a layer's kernels together take less than some 120 us the host is the
    slower side: the library's call costs it 3 us more than the tiles', a kernel behind it 8.  ``host_upto`` (us of the
    tiles) is where the layer around such a product has that length; beyond it the GPU is the slower side.

    Whole prompts, 12 layers, without regard for the host and with it, us: 0.5B shape, 400 rows 1,622, 1,330; 800 1,698,
    1,317; 1,500 1,698, 1,646; 3B shape, 150 rows 1,714, 1,411; 800 2,932, 2,819."""

    us: float
    us_per_million: float
    host_us: float
    host_upto: float
    margin_timed: float = 1.15  # (``DIRECT_MARGIN`` where the library's algorithms are timed)


BEHIND_NOTHING = Behind(0.0, 0.0, 3.0, 15.0)
BEHIND_GATE = Behind(2.15, 1.2, 11.0, 40.0, 1.03)  # the gate's kernel
BEHIND_BRANCH = Behind(-1.3, 1.9, 3.0, 15.0)     # the norm that adds the branch
BEHIND_ROTATION = Behind(1.1, 1.8, 11.0, 21.0)   # the rotation and cache write
# Where the host does not matter the tiles of csrc/gemm_tiles.hip are taken if they are modelled to be faster by the first of
# these, beyond 25 us by the second (a good algorithm that the library happens to have costs more there): of the 608 products 27
# were then more than 2 % slower than the library's inside a captured chain, and all together 6.3 % faster.
TILES_MARGIN, TILES_MARGIN_LONG, TILES_LONG_US = 1.05, 1.15, 25.0


def _tile_us(columns: int, tile_rows: int, parts: int, rows: int, n: int, k: int, units: int, times: dict = TILE_US) -> float:
    start, first, further = times[columns, tile_rows]
    tiles = -(-rows // tile_rows) * -(-n // columns)
    turns = -(-(-(-tiles // XCDS) * parts) // max(1, units // XCDS))
    slices = -(-(-(-k // parts)) // 64)
    return start + slices * (first + (turns - 1) * further) + (parts * rows * n * 4e-6 * TILE_PARTS_US if parts > 1 else 0.0)


def _library_us(rows: int, n: int, k: int, units: int, tuned: int) -> float:
    share = -(-rows // 128) * -(-n // 128) / units
    rate = min(LIBRARY_MOST, LIBRARY_RATE * share ** (0.46 if share < 1.0 else 0.51))
    start, per_k, per_weight = LIBRARY_US
    return LIBRARY_TUNED[tuned] * math.hypot(start + per_k * 1e-3 * k + per_weight * 1e-6 * n * k, 2e-9 * rows * n * k / rate)


# The tiles whose operands go straight into LDS (csrc/gemm_direct.hip; K a multiple of 64), by the same model, fitted to 7,500
# timings (0.5B, 3B, 7B and 14B widths at 16 row counts from 112 to 2,048; 10 % root mean square): the form it picks takes
# 1.7 % more than the best of all in the mean.  (Over 500 further products of any width and K, without and with the gate, 19 %:
# it leaves out the weight's way from memory and the result's to it, some 0.3 us a million weights and 0.6 a million results,
# which hardly choose between the forms.)  Against the tiles above and the library, us, each product alone (the kernel
# behind the library's not counted): 3B gate/up 256 rows 40 -> 33, 777 81 -> 72, 2,048 186 -> 157; down 613 47 -> 36, 2,048
# 100 -> 91; 7B gate/up 777 272 -> 175, 2,048 541 -> 445, down 777 167 -> 98.  What decides is how the turns come out: 777 rows
# x 37,888 are 740 tiles of 256 x 160, three turns of 256 units, and 1,036 of 256 x 128, five.
DIRECT_US = {(64, 64): (3.1, 0.239, 0.246), (96, 64): (3.4, 0.301, 0.299), (96, 128): (5.3, 0.390, 0.494),
             (128, 64): (3.0, 0.405, 0.340), (128, 128): (4.8, 0.467, 0.554), (128, 192): (5.4, 0.577, 0.671),
             (128, 256): (6.8, 0.662, 0.821), (192, 128): (5.7, 0.604, 0.684), (192, 192): (7.3, 0.713, 0.856),
             (192, 256): (6.9, 1.078, 1.208), (256, 128): (6.2, 0.750, 0.854), (256, 160): (7.7, 0.826, 0.977),
             (256, 256): (8.1, 1.299, 1.481)}
# Of the forms within this share of the fastest the one that reads least: level in the timings, less power inside a step (3B
# gate/up of 2,048 rows, tiles of 192 x 192 that the model prefers by 3 %: 161 us alone, 174 inside a prompt).
DIRECT_LEVEL = 1.04
# ... taken where they are modelled to be faster than the library by this, or, at the row counts whose algorithms it times, by
# ``Behind.margin_timed``: of 500 products at 256 to 2,048 such rows 399 were taken by 1.03, 29 of them more than 4 % slower than
# the library where the host is not what takes the time (512 rows x 4,096, K 11,136, 94 us against 82); by 1.15, and 1.03 for the
# gate, 346 and 7, the gain in the mean the same 13.4 %.  At 400 row counts that do not recur, where the library takes its first
# choice, eight of the 336 taken by 1.03.
DIRECT_MARGIN = 1.03
# ... but of up to this K also where they are modelled up to 1.15 times slower, at row counts that do not recur, and with nothing
# behind them of fewer columns than this (products between the two lines, 129 to 2,047 rows, K 512 to 4,096, tiles over the library and
# the kernel behind it in the mean, how many more than 4 % slower: plain, up to 8,191 columns 118, 0.87, 6; 8,192 to 28,000 222, 0.92, 49,
# 1,315 rows x 17,920, K 2,176 106.9 us for 92.5; the gate, 5,000 to 40,000 columns 143, 0.92, 8, all of 522 to 564 rows x some
# 17,000; a branch of 512 to 5,000 210, 0.89, 12, most of 232 to 280 rows; none with the rotation lies there.  1,999 rows x 4,736,
# K 2,048 45.4 -> 38.3 us, x 6,144 49.0 -> 47.4).  Beyond this K 14 of 51 plain ones were slower, 858 x 12,992, K 8,000, by 26 %.
DIRECT_MARGIN_SHORT, DIRECT_SHORT_K, DIRECT_SHORT_COLUMNS = 1 / 1.15, 4096, 8192
# Sums of K in parts are at most this many bytes (2,048 rows: 4 parts of the 3B shape's down product 67 MB, 2 of 7B's 59)
PARTS_BYTES = 128 << 20


@functools.lru_cache(maxsize=4096)
def _plan_tiles(rows: int, n: int, k: int, most_parts: int, behind: Behind, units: int,
                searched: frozenset) -> Optional[tuple[int, int, int]]:
    forms = [(columns, tile_rows, parts) for columns, tile_rows in TILE_US for parts in TILE_PARTS
             if parts <= most_parts and -(-(-(-k // parts)) // 64) * 64 * (parts - 1) < k]  # (every part has some of K)
    cost, form = min((_tile_us(*form, rows, n, k, units), form) for form in forms)
    library = _library_us(rows, n, k, units, ops._tune_level(rows)) + behind.us + behind.us_per_million * rows * n * 1e-6
    if cost <= behind.host_upto:
        return form if cost * TILES_MARGIN < library + behind.host_us else None
    return form if cost * (TILES_MARGIN if cost <= TILES_LONG_US else TILES_MARGIN_LONG) < library else None


def plan_tiles(rows: int, n: int, k: int, most_parts: int = 1, behind: Behind = BEHIND_NOTHING) -> Optional[tuple[int, int, int]]:
    """(columns, rows, parts of K) of the tiles that a bfloat16 product of some hundred rows takes, or ``None`` where the
    library's product, with what it costs ``behind`` it, is the faster one."""
    return _plan_tiles(rows, n, k, most_parts, behind, ops.compute_units(), ops._search_rows)


class Tiles(NamedTuple):
    """How a product of many rows runs: tiles of ``columns`` x ``rows``, K in ``parts`` parts, and whether its operands go
    straight into LDS."""

    columns: int
    rows: int
    parts: int
    direct: bool


@functools.lru_cache(maxsize=4096)
def _choose_direct(rows: int, n: int, k: int, most_parts: int, behind: Behind, units: int, searched: frozenset) -> Optional[Tiles]:
    forms = [(columns, tile_rows, parts) for columns, tile_rows in DIRECT_US for parts in TILE_PARTS
             if parts <= most_parts and -(-(-(-k // parts)) // 64) * 64 * (parts - 1) < k
             and (parts == 1 or parts * rows * n * 4 <= PARTS_BYTES)]
    times = {form: _tile_us(*form, rows, n, k, units, DIRECT_US) for form in forms}
    cost = min(times.values())
    reads = lambda f: (-(-rows // f[1]) * -(-n // f[0]) * (f[0] + f[1]), f[2])  # noqa: E731
    form = min((f for f in forms if times[f] <= cost * DIRECT_LEVEL), key=reads)
    timed = ops._tune_level(rows)
    library = _library_us(rows, n, k, units, timed) + behind.us + behind.us_per_million * rows * n * 1e-6
    library += behind.host_us if cost <= behind.host_upto else 0.0
    short = k <= DIRECT_SHORT_K and (n < DIRECT_SHORT_COLUMNS or behind is not BEHIND_NOTHING)
    margin = behind.margin_timed if timed else DIRECT_MARGIN_SHORT if short else DIRECT_MARGIN
    return Tiles(*form, True) if cost * margin < library else None


def choose_tiles(rows: int, n: int, k: int, row_stride: int, most_parts: int = 1, behind: Behind = BEHIND_NOTHING) -> Optional[Tiles]:
    """The tiles that a product of many rows takes, or ``None``: the library.  Whatever fits the kernel that loads straight
    into LDS is that kernel's or the library's; the other tiles have what is left (a K that is no multiple of 64)."""
    if ops.direct_fits(rows, n, k, row_stride):
        return _choose_direct(rows, n, k, most_parts, behind, ops.compute_units(), ops._search_rows)
    form = plan_tiles(rows, n, k, most_parts=most_parts, behind=behind)
    return None if form is None else Tiles(*form, False)


# Products of up to FUSED_PARTS_ROWS rows (more: the models above).  The forms whose waves read every row for every 16 or 32
# columns take longer with every row; the tiles that load straight into LDS read a row once for their 64 to 128 columns, but
# stream a weight no faster, and add more sums: which is faster goes by shape (MI355X, us, the other way and the tiles: down 3B
# 64 rows 14.9, 14.0, 128 23.3, 18.5; 4,096 x 4,096 in 8 parts of 128 rows at 96 rows 16.4, 20.3; 5,120 x 22,016 64 rows 51.7,
# 59.4; gate/up 0.5B 128 rows 14.5, 8.8, 14B 72.6, 65.7, 28,672 x 6,144 72 rows 71.7, 80.0, 1,024 x 6,144 112 rows 15.3, 18.2).  So
# both sides are modelled, each a sum of what it does, fitted to 28,000 timings inside captured chains, weights from memory
# (260 products of any width and K added into the stream, 260 gates, 97 products in parts with the norm behind them, at 8 or 9
# row counts from 17 to 128; 8 to 10 % root mean square for the tiles, 6 and 5 % for the forms of streaming waves, 10 for the
# library).  Tiles: a start, per slice of 64 k, and per million weights (by the rows of a tile) and sums.
FEW_CUT_US = {(64, 64): (1.83, 0.224), (96, 64): (1.95, 0.278), (128, 64): (1.63, 0.374), (96, 128): (2.38, 0.411),
              (128, 128): (1.67, 0.493)}
FEW_GATE_US = {(64, 64): (2.77, 0.166), (96, 64): (2.73, 0.217), (128, 64): (2.13, 0.305), (96, 128): (3.38, 0.325),
               (128, 128): (2.39, 0.397)}
FEW_CUT_WEIGHTS, FEW_CUT_SUMS = {64: 0.153, 128: 0.101}, 3.15
FEW_GATE_WEIGHTS, FEW_GATE_SUMS = {64: 0.238, 128: 0.206}, 0.473
# The other side: the cut product of streaming waves (a start, per 32 rows, per slice, the slice's 32 rows and those of all its
# column tiles, per million sums and weights), their gate (a start, per slice and 32 rows, per slice and pair that
# meets on a unit, per million weights and results), the library's gate with the kernel behind it (a start, per 1,000 k, per
# million weights and results).
SHARED_CUT_US = (1.90, 0.478, 0.0945, 0.0454, 0.0526, 2.62, 0.117)
SHARED_GATE_US = (4.29, 0.1364, 0.0743, 0.0219, 0.855)
LIBRARY_GATE_US = (8.28, 1.14, 0.385, 1.18)
# Tiles are taken where they are modelled to be faster by this: of the 2,080 cut products 1,491 are then, 34 of them more than 2 %
# slower than the other way (5,120 and 6,144 x 22,016 among them, 13 %: a K whose rows crowd few channels), of 1,560 gates against
# streaming waves 1,165 and 4 (27,648 x 2,048 at 72 rows 26.9, 30.8), of 780 against the library 684 and 9 (narrow ones at 128
# rows, where it times its candidates); in the mean 11, 23 and 19 % faster than without tiles.
FEW_CUT_MARGIN, FEW_GATE_MARGIN = 0.95, 0.93
FEW_TILE_ROWS = 48  # (at 32 rows the two are level)
FEW_TILE_PARTS = (1, 2, 4, 8)
# A product whose parts the next norm sums goes to tiles from FUSED_ROWS + 1 rows on (us, the library and the norm that adds its
# branch, tiles and the norm that sums parts: 3,584 x 3,584 17 rows 16.2, 12.3, 96 24.5, 16.8; 8,192 x 29,568 32 rows 110, 93; up
# to 40 million weights 584 timings, 11 more than 2 % slower, in the mean 20 % faster), but for a large weight whose rows lie a
# multiple of 8 KB apart, which the library streams at up to 4.8 TB/s: that from 65 rows on (8,192 x 8,192 32 rows 34, 40, 64 39,
# 38; 12,288 x 8,192 32 rows 49, 52, 72 63, 55; 8,192 x 16,384 48 rows 65, 72; from K 20,480 on it is the slower one again).  Of
# 800 timings beyond 40 million weights 73 are then more than 2 % slower, by up to 15 % (K 11,008, 3,072 and 5,120 of the
# widest most), in the mean 12 % faster.
FEW_PARTS_WEIGHTS, FEW_PARTS_APART, FEW_PARTS_K, FEW_PARTS_ROWS = 40 << 20, 4096, 16384, 65


def _few_us(form: tuple[int, int, int], rows: int, n: int, k: int, gate: bool) -> float:
    columns, tile_rows, parts = form
    times, weights, sums = ((FEW_GATE_US, FEW_GATE_WEIGHTS, FEW_GATE_SUMS) if gate else (FEW_CUT_US, FEW_CUT_WEIGHTS, FEW_CUT_SUMS))
    start, per_slice = times[columns, tile_rows]
    return (start + -(-(-(-k // parts)) // ops.DIRECT_SLICE) * per_slice + n * k * 1e-6 * weights[tile_rows]
            + parts * rows * n * 1e-6 * sums)


@functools.lru_cache(maxsize=4096)
def plan_few_tiles(rows: int, n: int, k: int, most_parts: int, units: int, gate: bool = False) -> Optional[tuple[int, int, int]]:
    """(columns, rows, parts) of the tiles of up to FUSED_PARTS_ROWS rows, or ``None`` if no form meets the units in one turn (each
    XCD has an eighth of the tiles and of the units): of those that do the fastest by the model."""
    forms = []
    for columns, tile_rows in FEW_CUT_US:
        if tile_rows > 64 >= rows:
            continue
        for parts in FEW_TILE_PARTS:
            groups = -(-(-(-n // columns) * -(-rows // tile_rows)) // XCDS) * parts
            if (parts <= most_parts and groups <= units // XCDS
                    and -(-(-(-k // parts)) // ops.DIRECT_SLICE) * ops.DIRECT_SLICE * (parts - 1) < k):
                forms.append((columns, tile_rows, parts))
    return min(forms, key=lambda form: _few_us(form, rows, n, k, gate), default=None)


@functools.lru_cache(maxsize=4096)
def _cut_tiles(rows: int, n: int, k: int, units: int) -> Optional[tuple[int, int, int]]:
    form = plan_few_tiles(rows, n, k, FEW_TILE_PARTS[-1], units)
    if form is None:
        return None
    column_tiles, _waves, parts = plan_shared_parts(-(-n // 16), k)
    slices, pairs = -(-(-(-k // parts)) // 64), -(-rows // 32)
    start, per_rows, per_slice, per_pair, per_tile, per_sums, per_weights = SHARED_CUT_US
    other = (start + pairs * per_rows + slices * (per_slice + pairs * (per_pair + column_tiles * per_tile))
             + parts * rows * n * 1e-6 * per_sums + n * k * 1e-6 * per_weights)
    return form if _few_us(form, rows, n, k, False) < FEW_CUT_MARGIN * other else None


@functools.lru_cache(maxsize=4096)
def _gate_tiles(rows: int, n: int, k: int, units: int) -> Optional[tuple[int, int, int]]:
    form = plan_few_tiles(rows, n, k, 1, units, True)
    if form is None:
        return None
    if rows <= SHARED_SILU_ROWS:
        pairs = -(-n // 32)
        waves, _own = plan_shared_silu(pairs)
        start, per_rows, per_pair, per_weights, per_results = SHARED_GATE_US
        other = start + k / 64 * (-(-rows // 32) * per_rows + -(-(-(-pairs // waves)) // units) * waves * per_pair)
    else:
        start, per_k, per_weights, per_results = LIBRARY_GATE_US
        other = start + k * 1e-3 * per_k
    other += n * k * 1e-6 * per_weights + rows * n * 1e-6 * per_results
    return form if _few_us(form, rows, n, k, True) < FEW_GATE_MARGIN * other else None


def _few_fits(x: torch.Tensor, weight: torch.Tensor, into: Optional[torch.Tensor], fewest: int) -> bool:
    rows, k = x.shape
    return (fewest <= rows <= FUSED_PARTS_ROWS and takes_tiles(rows, x, weight, into, beyond=FUSED_ROWS)
            and ops.direct_fits(rows, weight.shape[0], k, x.stride(0)))


def cut_tiles(x: torch.Tensor, weight: torch.Tensor, into: Optional[torch.Tensor] = None) -> Optional[tuple[int, int, int]]:
    """(columns, rows, parts of K) of the tiles that a product takes whose other way is the cut form of streaming waves, or
    ``None``: that one."""
    if not _few_fits(x, weight, into, FEW_TILE_ROWS):
        return None
    return _cut_tiles(x.shape[0], weight.shape[0], x.shape[1], ops.compute_units())


def part_tiles(x: torch.Tensor, weight: torch.Tensor, into: torch.Tensor) -> Optional[tuple[int, int, int]]:
    """... whose other way is the library."""
    n, k = weight.shape
    large = n * k > FEW_PARTS_WEIGHTS and k % FEW_PARTS_APART == 0 and k <= FEW_PARTS_K
    if not _few_fits(x, weight, into, FEW_PARTS_ROWS if large else FUSED_ROWS + 1):
        return None
    return plan_few_tiles(x.shape[0], n, k, FEW_TILE_PARTS[-1], ops.compute_units())


def gate_tiles(x: torch.Tensor, weight: torch.Tensor) -> Optional[tuple[int, int, int]]:
    """(columns, rows, 1) of the tiles that a gated unit's product takes, or ``None``: the form of streaming waves, or the library."""
    if not _few_fits(x, weight, None, FEW_TILE_ROWS):
        return None
    return _gate_tiles(x.shape[0], weight.shape[0], x.shape[1], ops.compute_units())


@dataclass
class RowSumsq:
    """Stands where a branch output would: the branch was already added into the
    residual stream, and ``sumsq`` [rows, parts] holds partial sums of squares of
    the residual's rows (what an RMSNorm needs of them).  ``scaled``, if given, is
    the new residual times the weight of ``norm`` in bf16: that norm's output
    short of each row's 1/rms."""

    sumsq: torch.Tensor
    scaled: Optional[torch.Tensor] = None
    norm: Any = None


@dataclass
class ScaledRows:
    """Stands where an RMSNorm's output would: ``rows`` [M, hidden] bf16 lack the
    factor ``rsqrt(sum(sumsq[m]) / hidden + eps)`` of their row, which a product
    that reads them applies to its sums (a product is linear in its rows)."""

    rows: torch.Tensor
    sumsq: torch.Tensor
    eps: float
    residual: torch.Tensor
    norm: Any

    @property
    def shape(self):
        return self.rows.shape

    def complete(self) -> torch.Tensor:
        """The norm's output after all (for a reader that cannot apply the factor)."""
        return ops.rmsnorm_from_sumsq(self.residual, self.sumsq, self.norm.weight, self.eps)


@dataclass
class Added:
    """Stands where a branch output would: the branch was already added into the residual stream, and
    nothing else is known of the stream's rows (a product whose K was cut into parts, each of which added
    its share with atomic adds)."""


@dataclass
class KParts:
    """Stands where a branch output would: the branch is the sum of ``parts`` [P, rows, hidden] (float32), still to be
    added into the stream, in order: a product whose K was cut.  A norm that says ``takes_parts`` sums them itself."""

    parts: torch.Tensor

    def join(self, residual: torch.Tensor) -> None:
        """Add the branch into the stream (for a reader that cannot sum the parts)."""
        for part in self.parts:
            residual.add_(part)


@dataclass
class StreamRows(Added):
    """An ``Added`` that also carries the whole stream rounded to the activation type (``rows``): what a layer
    whose sublayers read the stream itself, not a norm of it, hands to the next one."""

    rows: Optional[torch.Tensor] = None


@dataclass
class SummedBranch:
    """A branch output that is still a sum: ``main`` [T, H] (or ``None``) plus the ``P`` rows of each token in
    ``parts`` (float32 [T, P, H]).  Whoever adds the branch sums them, in that order.  ``weights`` (float32 [T, P]):
    each row of ``parts`` counts that much; ``main_gate`` (float32 [T], logits): ``main`` counts ``sigmoid`` of it.
    Only a norm that applies them (``GroupedRMSNorm``) may be handed a branch that has them."""

    main: Optional[torch.Tensor]
    parts: Optional[torch.Tensor]
    weights: Optional[torch.Tensor] = None
    main_gate: Optional[torch.Tensor] = None


@dataclass
class WeightedPair:
    """A branch output that is still a weighted sum of two: ``scales[0] * first + scales[1] * second`` (two mixers
    that ran side by side).  A block whose adding kernel takes two branches hands them over as they are; any other
    asks for :meth:`combined`."""

    first: torch.Tensor
    second: torch.Tensor
    scales: tuple[float, float] = (1.0, 1.0)

    def combined(self) -> torch.Tensor:
        total = self.first.float() * self.scales[0] + self.second.float() * self.scales[1]
        return total.to(self.first.dtype)


@dataclass
class RawRows:
    """Stands where an RMSNorm's output would, before anything was computed: the rows are the norm ``norm``
    of the float32 stream ``residual``.  Only a part that says ``takes_raw_rows`` is shown it (the attention
    part's q/k/v product then makes its rows itself, with up to ``ops.FOLDED_NORM_ROWS`` rows: every workgroup
    reads the few rows once, where a kernel of its own for the norm costs a decode layer 4.6 us; behind a branch that
    was added in parts the feed-forward's first product too)."""

    residual: torch.Tensor
    norm: Any
    dtype: torch.dtype = torch.bfloat16

    @staticmethod
    def fits(residual: torch.Tensor, dtype: torch.dtype) -> bool:
        rows, width = residual.shape
        if dtype == torch.float32:
            return ops.folds_norm_f32(residual)
        return dtype == torch.bfloat16 and residual.is_cuda and ops.folds_norm(rows, width)

    @property
    def shape(self):
        return self.residual.shape

    def joins_f32(self, weight: torch.Tensor) -> bool:
        """Whether the float32 product with this weight can make the norm itself."""
        return (self.dtype == weight.dtype == torch.float32 and weight.data_ptr() % 16 == 0
                and self.norm.weight_f32.data_ptr() % 16 == 0)

    def joins_silu(self, weight: torch.Tensor) -> bool:
        """... and whether the bfloat16 SiLU-gate product can."""
        return (self.dtype == weight.dtype == torch.bfloat16 and weight.data_ptr() % 16 == 0 and self.residual.is_contiguous()
                and self.residual.data_ptr() % 16 == 0 and self.norm.weight_f32.data_ptr() % 16 == 0)

    def complete(self) -> torch.Tensor:
        """The norm's output after all."""
        return ops.add_rmsnorm(self.residual, None, self.norm.weight, self.norm.eps, self.dtype)


def linear_beside(x: torch.Tensor, weight: torch.Tensor, act_out: torch.Tensor) -> torch.Tensor:
    """One product for two readers of the same rows: ``x @ weight.T``, whose last columns (as many as ``act_out`` has) go
    to ``act_out`` as the square of their relu (in the product's own epilogue where the hand-written form runs, in a
    kernel behind it otherwise).  The columns in front of them come back (their rows may lie apart)."""
    rows, k = x.shape
    n = weight.shape[0]
    split = n - act_out.shape[1]
    if _fusable(rows, k, x.stride(0) if rows > 1 else k, weight) and (
            rows <= FUSED_ROWS or (rows <= FUSED_SMALL_ROWS and n * k <= FUSED_SMALL_WEIGHT)):
        return ops.gemm_fused(weight, ops.EPI_BF16, x, act_out=act_out)
    out = linear(x, weight)
    ops.squared_relu(out[:, split:], act_out)
    return out[:, :split]


def logits_at(x: torch.Tensor, weight: torch.Tensor, out_at: torch.Tensor) -> bool:
    """``x @ weight.T`` in float32 into the contiguous matrix whose address ``out_at`` holds when the kernel runs, if the form that
    :func:`linear` takes for it can write there; else nothing is done."""
    rows, k = x.shape
    n = weight.shape[0]
    if not (x.is_cuda and rows >= 1 and x.stride(1) == 1):
        return False
    if weight.dtype == torch.float32:
        if x.dtype != torch.float32 or rows > ops.F32_FEW_ROWS:
            return False
        ops.gemm_f32_at(x, weight, out_at)
        return True
    if not _fusable(rows, k, x.stride(0) if rows > 1 else k, weight) or x.data_ptr() % 16 or weight.data_ptr() % 16:
        return False
    if shares_rows_f32(rows, n, k):
        ops.gemm_shared_rows(weight, ops.EPI_F32, x, waves=4, out_at=out_at)
        return True
    if rows > FUSED_LOGIT_ROWS:
        return False
    ops.gemm_fused(weight, ops.EPI_F32, x, out_at=out_at)
    return True


# Two products of few rows that wait for the same things run in one launch (a layer whose mixer and feed-forward read the same
# stream; MI355X, us, apart and together, 1 / 8 / 16 rows): gate/up and 6,144 columns of the 3B widths 27.5, 24.0 / 27.3, 23.3 / 28.4, 23.4,
# 4,096 columns 24.0, 21.8 / 24.9, 22.0 / 25.7, 22.0; 0.5B and 2,304 10.7, 7.5 / 11.3, 7.6 / 11.5, 7.7; 7B and 7,168 65.7, 59.5 / 68.3,
# 57.6 / 72.3, 57.8; down and an output product, as parts: 3B 16.9, 13.8 / 17.6, 14.1 / 18.3, 14.3; 0.5B 8.7, 5.1 / 9.1, 5.3 / 9.3, 5.4; 7B 36.0,
# 35.8 / 37.2, 36.6 / 38.7, 37.2; 14B 44.9, 39.6 / 47.0, 39.9 / 50.8, 40.6.
def plan_silu_beside(pairs: int, tiles: int, units: int) -> int:
    """Waves per workgroup of the SiLU product of ``pairs`` gate tiles and a product of ``tiles`` column tiles in one launch: the
    fewest pairs (or two tiles) that meet on a unit, each XCD's turns counted as :func:`plan_shared_silu` counts them."""
    return min((4, 3, 2), key=lambda waves: -(-(-(-pairs // waves) + -(-tiles // (2 * waves))) // units) * waves)


def plan_parts_beside(tiles: int, k: int, k2: int, units: int) -> tuple[int, int]:
    """Parts of the two products' K: as many together as give about one workgroup per unit, the longest stretch the shortest."""
    together = max(2, min(units // -(-tiles // 4), 16))
    stretch = lambda k, parts: -(-(-(-k // parts)) // 128) * 128  # noqa: E731
    parts2 = min(range(1, together), key=lambda p: max(stretch(k, together - p), stretch(k2, p)))
    parts = together - parts2
    return -(-k // stretch(k, parts)), -(-k2 // stretch(k2, parts2))  # (none a part without k)


def _beside(x: torch.Tensor, weight: torch.Tensor) -> bool:
    rows, k = x.shape
    return (x.dtype == torch.bfloat16 and x.is_cuda and x.stride(1) == 1 and 1 <= rows <= FUSED_ROWS
            and _fusable(rows, k, x.stride(0) if rows > 1 else k, weight) and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)


def silu_beside(x: torch.Tensor, weight: torch.Tensor, x2: torch.Tensor, weight2: torch.Tensor,
                bias2: Optional[torch.Tensor]) -> Optional[tuple[torch.Tensor, torch.Tensor]]:
    """(``silu(gate) * up`` of ``x``, ``x2 @ weight2.T + bias2``) in one launch, or ``None`` where that takes another form."""
    if not (_beside(x, weight) and _beside(x2, weight2) and weight.shape[0] % 2 == 0 and weight.shape[1] == weight2.shape[1]
            and x.shape[0] == x2.shape[0]):
        return None
    waves = plan_silu_beside(-(-weight.shape[0] // 32), -(-weight2.shape[0] // 16), ops.compute_units())
    return ops.gemm_silu_beside(weight, x, weight2, x2, bias2, waves)


def parts_beside(x: torch.Tensor, weight: torch.Tensor, x2: torch.Tensor, weight2: torch.Tensor) -> Optional[KParts]:
    """``x @ weight.T + x2 @ weight2.T`` as parts, from one launch, or ``None`` where that takes another form."""
    n, k = weight.shape
    if not (_beside(x, weight) and _beside(x2, weight2) and weight2.shape[0] == n and x.shape[0] == x2.shape[0]
            and -(-n // 16) < PART_BELOW_TILES):
        return None
    parts, parts2 = plan_parts_beside(-(-n // 16), k, weight2.shape[1], ops.compute_units())
    return KParts(ops.gemm_parts_beside(weight, x, parts, weight2, x2, parts2))


_WIDENED: dict[int, tuple["weakref.ref", torch.Tensor]] = {}


def _widened(weight: torch.Tensor) -> torch.Tensor:
    """``weight`` in float32, made at its first use (an output head of 150,000 rows is not copied every step)."""
    key = id(weight)
    kept = _WIDENED.get(key)
    if kept is not None and kept[0]() is weight:
        return kept[1]
    wide = weight.float()
    _WIDENED[key] = (weakref.ref(weight, lambda _gone, key=key: _WIDENED.pop(key, None)), wide)
    return wide


def _fusable(rows: int, k: int, row_stride: int, weight: torch.Tensor) -> bool:
    return weight.dtype == torch.bfloat16 and rows >= 1 and k % 8 == 0 and row_stride % 8 == 0


def takes_tiles(rows: int, x: torch.Tensor, weight: torch.Tensor, into: Optional[torch.Tensor] = None,
                beyond: int = FUSED_PARTS_ROWS) -> bool:
    """Whether the tile kernels take these operands (of a product that is ``_fusable``): beyond the rows of the streaming
    kernels, on the GPU, in rows that lie apart and at addresses that 16-byte loads and stores can use.  Whatever else a
    caller brings (rows read across, rows that share their numbers, as one row expanded to many does, a stream that starts
    off a 16-byte line, host tensors) is the library's or torch's, as it was."""
    if rows <= beyond or not x.is_cuda:
        return False
    apart, inner = x.stride()
    return (inner == 1 and apart >= x.shape[1] and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
            and (into is None or (into.is_cuda and into.dtype == torch.float32 and into.data_ptr() % 16 == 0)))


def linear(x: Union[torch.Tensor, ScaledRows, RawRows], weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
           out_dtype: Optional[torch.dtype] = None, epilogue: Optional[str] = None,
           into: Optional[torch.Tensor] = None, then_norm: Any = None,
           sums_parts: bool = False) -> Union[torch.Tensor, RowSumsq, Added, KParts]:
    """``x @ weight.T + bias``.

    ``epilogue="silu"``: weight stacks gate rows over up rows; returns
    ``silu(gate) * up``.  ``into=residual``: the caller wants the result added to
    the float32 residual stream; if a fused kernel runs it adds it in place, and a
    :class:`RowSumsq` comes back, or (a product whose K was cut into parts that
    each add their share) an :class:`Added`; otherwise the plain
    result comes back and the caller adds it (the next norm kernel does).
    ``sums_parts``: the caller's block takes :class:`KParts` too.
    ``then_norm`` (with ``into``): the norm that follows, if it can be folded into
    this product and the next (``RMSNorm.folds_into_products``): the residual
    epilogue then also leaves that norm's output short of the rows' scale.
    ``x`` may be such rows (:class:`ScaledRows`): the SiLU product of few rows
    applies the scale itself, any other reader gets the completed rows.  :class:`RawRows`:
    the SiLU product of few rows makes their norm itself."""
    if isinstance(x, ScaledRows):
        rows, k = x.rows.shape
        if epilogue == "silu" and weight.shape[0] % 2 == 0 and bias is None and weight.dtype == torch.bfloat16:
            if _fusable(rows, k, x.rows.stride(0) if rows > 1 else k, weight):
                tiles = gate_tiles(x.rows, weight)
                if tiles is not None:
                    return ops.gemm_tiles_silu_scaled(weight, x.rows, tiles[0], tiles[1], x.sumsq, x.eps)
                waves, own_unit = plan_shared_silu(-(-weight.shape[0] // 32))
                if FUSED_ROWS < rows <= SHARED_SILU_ROWS or (rows <= FUSED_ROWS and own_unit):
                    return ops.gemm_shared_rows(weight, ops.EPI_SILU, x.rows, waves=waves, row_sumsq=x.sumsq, eps=x.eps)
                if rows <= FUSED_ROWS:
                    return ops.gemm_fused(weight, ops.EPI_SILU, x.rows, row_sumsq=x.sumsq, eps=x.eps)
            # more rows: the library's product of the rows as they are, the scale in the SiLU kernel behind it
            out = ops.gemm_library(x.rows, weight) if x.rows.stride(1) == 1 else None
            if out is not None:
                return ops.silu_mul(out, row_sumsq=x.sumsq, hidden=k, eps=x.eps)
        x = x.complete()
    if isinstance(x, RawRows):
        if epilogue == "silu" and weight.shape[0] % 2 == 0 and bias is None and into is None and x.joins_f32(weight):
            return ops.gemm_f32_normed(x.residual, x.norm.weight_f32, x.norm.eps, weight)
        if epilogue == "silu" and weight.shape[0] % 2 == 0 and bias is None and into is None and x.joins_silu(weight):
            waves, _own_unit = plan_shared_silu(-(-weight.shape[0] // 32))
            return ops.gemm_shared_rows_normed(x.residual, x.norm.weight_f32, x.norm.eps, weight, waves)
        x = x.complete()
    rows, k = x.shape
    n = weight.shape[0]
    silu = epilogue == "silu"
    wants_f32 = out_dtype == torch.float32
    if rows == 0 and into is None:  # nothing to multiply: no kernel, and no widened copy of the weight
        return torch.empty((0, n // 2 if silu else n), dtype=torch.float32 if wants_f32 else x.dtype, device=x.device)
    fusable = _fusable(rows, k, x.stride(0) if rows > 1 else k, weight)
    cut_k = into is not None and cuts_k(n, k) and into.is_contiguous() and tuple(into.shape) == (rows, n)
    if fusable and cut_k and rows <= FUSED_PARTS_ROWS:
        # (atomic adds cost the product nothing, measured against partial products written for the next norm
        # kernel to sum: 10.3 us either way for the 3B shape's down product at 8 rows; and the kernel that summed
        # them falls away)
        tiles = cut_tiles(x, weight, into)
        if tiles is not None:
            ops.gemm_tiles(weight, ops.TILE_ATOMIC, x, tiles[0], tiles[1], bias, into, tiles[2], direct=True)
            return Added()
        column_tiles, waves, parts = plan_shared_parts(-(-n // 16), k)
        ops.gemm_shared_rows(weight, ops.EPI_ATOMIC, x, bias=bias, column_tiles=column_tiles, waves=waves,
                             k_parts=parts, add_into=into)
        return Added()
    if (fusable and into is None and sums_parts and not silu and not wants_f32 and rows <= FUSED_PARTS_ROWS and cuts_k(n, k)
            and x.data_ptr() % 16 == 0):
        # a branch that whoever adds it sums itself (the down product of the parallel block, 8 rows, K 11,008: 17 us whole,
        # 11 in 8 parts, and 0.4 more in the kernel that adds them)
        tiles = cut_tiles(x, weight)
        if tiles is not None:
            return KParts(ops.gemm_tiles(weight, ops.TILE_PARTS, x, tiles[0], tiles[1], bias, None, tiles[2], direct=True))
        column_tiles, waves, parts = plan_shared_parts(-(-n // 16), k)
        return KParts(ops.gemm_shared_rows(weight, ops.EPI_PARTIAL, x, bias=bias, column_tiles=column_tiles, waves=waves,
                                           k_parts=parts))
    if fusable and silu and n % 2 == 0 and bias is None and into is None and not wants_f32 and rows <= FUSED_PARTS_ROWS:
        tiles = gate_tiles(x, weight)
        if tiles is not None:
            return ops.gemm_tiles(weight, ops.TILE_SILU, x, tiles[0], tiles[1], direct=True)
    if fusable and silu and n % 2 == 0 and bias is None and into is None and not wants_f32 and rows <= SHARED_SILU_ROWS:
        waves, own_unit = plan_shared_silu(-(-n // 32))
        if rows > FUSED_ROWS or own_unit:
            return ops.gemm_shared_rows(weight, ops.EPI_SILU, x, waves=waves)
    if (fusable and wants_f32 and into is None and not silu and shares_rows_f32(rows, n, k)
            # (beyond these rows the library is the other way, which takes operands that start off a 16-byte line too)
            and (rows <= SHARED_LOGIT_FILL[-1][0] or (x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0))):
        return ops.gemm_shared_rows(weight, ops.EPI_F32, x, bias=bias, waves=4)
    if fusable and wants_f32 and rows > FUSED_LOGIT_ROWS and into is None and not silu and bias is None:
        out = ops.gemm_library(x, weight, out_dtype=torch.float32)  # logits of many rows: one pass over the weight
        if out is not None:
            return out
    small = rows <= FUSED_SMALL_ROWS and n * k <= FUSED_SMALL_WEIGHT and not silu
    if fusable and (rows <= FUSED_ROWS or wants_f32 or small):
        if into is not None:
            if then_norm is not None:
                scaled = torch.empty((rows, n), dtype=torch.bfloat16, device=x.device)
                sumsq = ops.gemm_fused(weight, ops.EPI_RESID, x, bias=bias, residual_out=into,
                                       norm_weight=then_norm.weight_f32, scaled_out=scaled)
                return RowSumsq(sumsq, scaled, then_norm)
            return RowSumsq(ops.gemm_fused(weight, ops.EPI_RESID, x, bias=bias, residual_out=into))
        elif silu and n % 2 == 0:
            return ops.gemm_fused(weight, ops.EPI_SILU, x)
        elif not silu:
            return ops.gemm_fused(weight, ops.EPI_F32 if wants_f32 else ops.EPI_BF16, x, bias=bias)
    if (fusable and not wants_f32 and not silu and into is not None and sums_parts and FUSED_ROWS < rows <= FUSED_PARTS_ROWS
            and into.is_contiguous() and tuple(into.shape) == (rows, n)):
        tiles = part_tiles(x, weight, into)
        if tiles is not None:  # (the norm behind it sums the parts)
            return KParts(ops.gemm_tiles(weight, ops.TILE_PARTS, x, tiles[0], tiles[1], bias, None, tiles[2], direct=True))
    if fusable and not wants_f32 and takes_tiles(rows, x, weight, into):
        stride, most = x.stride(0), TILE_PARTS[-1] if sums_parts else 1
        if into is not None and not silu and into.is_contiguous() and tuple(into.shape) == (rows, n):
            tiles = choose_tiles(rows, n, k, stride, most_parts=most, behind=BEHIND_BRANCH)
            if tiles is not None and tiles.parts > 1:
                return KParts(ops.gemm_tiles(weight, ops.TILE_PARTS, x, tiles.columns, tiles.rows, bias, None, tiles.parts, tiles.direct))
            if tiles is not None:
                ops.gemm_tiles(weight, ops.TILE_RESID, x, tiles.columns, tiles.rows, bias, into, 1, tiles.direct)
                return Added()
        elif into is None and silu and n % 2 == 0 and bias is None:
            tiles = choose_tiles(rows, n, k, stride, behind=BEHIND_GATE)
            if tiles is not None:
                return ops.gemm_tiles(weight, ops.TILE_SILU, x, tiles.columns, tiles.rows, None, None, 1, tiles.direct)
        elif into is None and not silu:
            tiles = choose_tiles(rows, n, k, stride, most_parts=most)
            if tiles is not None and tiles.parts > 1:
                return KParts(ops.gemm_tiles(weight, ops.TILE_PARTS, x, tiles.columns, tiles.rows, bias, None, tiles.parts, tiles.direct))
            if tiles is not None:
                return ops.gemm_tiles(weight, ops.TILE_BF16, x, tiles.columns, tiles.rows, bias, None, 1, tiles.direct)
    if weight.dtype == torch.float32:
        if silu and n % 2 == 0 and bias is None:
            return ops.gemm_f32(x, weight, gate=True)
        if (into is not None and not silu and 1 <= rows <= ops.F32_FEW_ROWS and into.is_cuda and into.dtype == torch.float32
                and into.is_contiguous() and tuple(into.shape) == (rows, n)):
            ops.gemm_f32_into(x, weight, bias, into)  # (the next norm need not add it: it may ride in the product behind it)
            return Added()
        out = ops.gemm_f32(x, weight, bias)
    elif wants_f32:
        # a shape the kernel refuses (a width that is no multiple of 8): widened operands, exact products,
        # float32 sums; the widened weight is made once and kept for as long as the weight lives
        out = x.float() @ _widened(weight).t()
        out = out if bias is None else out + bias.float()
    else:
        out = ops.gemm_library(x, weight, bias) if x.is_cuda and x.stride(1) == 1 else None
        if out is None:  # a shape the library's own interface has no algorithm for
            out = torch.nn.functional.linear(x, weight, bias)
    return ops.silu_mul(out) if silu else out
