"""Grouped-query softmax attention over the paged cache.

Reference: ``Qwen2Attention.project`` (src/cloud_engine/model.py:103-137),
``apply_rope`` (src/cloud_engine/attention.py:75-85), the KV write before the
read (src/cloud_engine/cache.py:398-413) and the ragged attention of
``kernel.py:324-405``: query head ``h`` reads KV head ``h // group``, scores are
``q.k / sqrt(D)``, a token sees every cached key up to itself.  Here q, k and v
are one fused product, rotation and cache write are one kernel, and sizes, bias
switches, scale, position encoding and an optional window are parameters.
"""

from __future__ import annotations

import functools
import math
import warnings
from dataclasses import dataclass
from typing import Optional

import torch

from ..cache.manager import PagedKV
from ..config.specs import PartSpec
from ..kernels import ops
from ..weights.tensors import TensorSpec
from .base import Part, build_part, register_part
from .linear import Added, BEHIND_ROTATION, FUSED_ROWS, FUSED_SMALL_ROWS, FUSED_SMALL_WEIGHT, RawRows, choose_tiles, cuts_k, linear, takes_tiles


class Attention(Part):
    graph_safe = True
    adds_to_residual = True
    folds_next_norm = True  # its output product can leave the next norm's rows short of their scale
    takes_raw_rows = True  # its first product can make the norm of a few rows itself
    sums_parts = True  # its last product may come back as parts of K
    adds_unordered = True  # ... or merge a decode step's shares itself, and add their sums to the stream in no fixed order
    def __init__(self, hidden_size: int, num_heads: int, num_kv_heads: int, head_dim: int,
                 qkv_bias: bool, out_bias: bool, position: PartSpec, window: Optional[int] = None,
                 scale: Optional[float] = None) -> None:
        if num_heads % num_kv_heads:
            raise ValueError(f"{num_heads} query heads are no multiple of {num_kv_heads} key heads")
        if head_dim % 8 or head_dim > 256:
            raise ValueError(f"head_dim must be a multiple of 8 up to 256 for the attention kernels, got {head_dim}")
        if window is not None and window < 1:
            raise ValueError("window must be positive")
        self.hidden_size = hidden_size
        self.num_heads = num_heads
        self.num_kv_heads = num_kv_heads
        self.head_dim = head_dim
        self.qkv_bias = qkv_bias
        self.out_bias = out_bias
        self.window = window
        self.scale = float(scale) if scale is not None else 1.0 / math.sqrt(head_dim)
        self.position = build_part("position", position)
        # A head size that the matrix-core attention does not take (80, 112, 40, ...) runs as the next one it does:
        # the projections' rows of a head are padded with zero rows, which changes no score and no output (the keys'
        # and values' extra dimensions are zeros in the cache, o_proj's extra columns are zeros), and costs that much
        # more cache.  The generic kernel, which takes every size, is 20 (decode) to 180 (a 2,048-token prompt) times
        # slower.  A variant that works on the projected heads (``shape_projection``) sees the heads as they are.
        self.kernel_head_dim = head_dim
        if type(self).shape_projection is Attention.shape_projection:
            self.kernel_head_dim = next((size for size in ops.MFMA_HEAD_DIMS if size >= head_dim), head_dim)

    def cache_need(self) -> PagedKV:
        return PagedKV(self.num_kv_heads, self.kernel_head_dim, self.window)

    def expected_tensors(self, prefix: str) -> dict[str, TensorSpec]:
        q_out = self.num_heads * self.head_dim
        kv_out = self.num_kv_heads * self.head_dim
        out = {
            prefix + "q_proj.weight": TensorSpec((q_out, self.hidden_size)),
            prefix + "k_proj.weight": TensorSpec((kv_out, self.hidden_size)),
            prefix + "v_proj.weight": TensorSpec((kv_out, self.hidden_size)),
            prefix + "o_proj.weight": TensorSpec((self.hidden_size, q_out)),
        }
        if self.qkv_bias:
            out[prefix + "q_proj.bias"] = TensorSpec((q_out,))
            out[prefix + "k_proj.bias"] = TensorSpec((kv_out,))
            out[prefix + "v_proj.bias"] = TensorSpec((kv_out,))
        if self.out_bias:
            out[prefix + "o_proj.bias"] = TensorSpec((self.hidden_size,))
        return out

    def bind(self, tensors, prefix, dtype, device) -> None:
        super().bind(tensors, prefix, dtype, device)
        names = ("q_proj", "k_proj", "v_proj")
        extra = self.kernel_head_dim - self.head_dim

        def per_head(t: torch.Tensor) -> torch.Tensor:
            # [heads * head_dim, ...] -> [heads * kernel_head_dim, ...], each head followed by zero rows
            if not extra:
                return t
            heads = t.shape[0] // self.head_dim
            padded = t.new_zeros((heads, self.kernel_head_dim) + tuple(t.shape[1:]))
            padded[:, : self.head_dim] = t.reshape((heads, self.head_dim) + tuple(t.shape[1:]))
            return padded.reshape((heads * self.kernel_head_dim,) + tuple(t.shape[1:]))

        self.w_qkv = torch.cat([per_head(tensors[f"{prefix}{n}.weight"]) for n in names], dim=0).contiguous()
        self.b_qkv = (
            torch.cat([per_head(tensors[f"{prefix}{n}.bias"]) for n in names], dim=0).contiguous()
            if self.qkv_bias else None
        )
        self.w_o = per_head(tensors[prefix + "o_proj.weight"].t()).t().contiguous()
        self.cuts_o = cuts_k(*self.w_o.shape)  # (whose sum has no fixed order then, whoever merges its rows)
        self.b_o = tensors[prefix + "o_proj.bias"].contiguous() if self.out_bias else None
        self.cos, self.sin = self.position.tables(device)

    def warm_up(self, rows: int) -> None:
        blank = lambda width: torch.zeros((rows, width), dtype=self.w_qkv.dtype, device=self.w_qkv.device)
        linear(blank(self.hidden_size), self.w_qkv, self.b_qkv)
        linear(blank(self.num_heads * self.kernel_head_dim), self.w_o, self.b_o)

    def shape_projection(self, qkv: torch.Tensor, batch) -> torch.Tensor:
        """The seam between projection and rotation: what a variant of this mixer does to the projected
        rows ``[tokens, (query heads + 2 key heads) * head_dim]`` (bias added; queries first, then keys,
        then values) before they are rotated and the keys and values go to the cache, such as a norm over
        each query and key head.  The default does nothing, and only a mixer that leaves it so lets the
        projection's own kernel rotate and write the cache."""
        return qkv

    def forward(self, x, batch, view, writes: bool = True, residual: Optional[torch.Tensor] = None,
                next_norm=None, sums_parts: bool = False, unordered: bool = False):
        if batch.max_context > self.position.max_position and self.position.rotates:
            raise ValueError(
                f"position {batch.max_context - 1} is beyond the rotary table of {self.position.max_position}"
            )
        rows = x.shape[0]
        few = rows <= FUSED_ROWS or (rows <= FUSED_SMALL_ROWS and self.w_qkv.numel() <= FUSED_SMALL_WEIGHT)
        head_dim = self.kernel_head_dim  # what the kernels and the cache see
        # the projection's own kernel rotates whole heads only, and only an untouched projection
        rotary_dim = getattr(self.position, "rotary_dim", self.head_dim) if self.position.rotates else None
        untouched = (type(self).shape_projection is Attention.shape_projection
                     and rotary_dim in (None, head_dim) and head_dim == self.head_dim)
        if isinstance(x, RawRows):
            if untouched and head_dim % 32 == 0 and self.w_qkv.dtype == torch.bfloat16:
                # the product makes the norm of its rows itself
                qkv = ops.gemm_qkv_rope(
                    self.w_qkv, None, self.b_qkv, self.cos, self.sin, batch.positions, batch.seq_of_token,
                    batch.seq_slot, view.block_table, view.k_pool, view.v_pool, self.num_heads, self.num_kv_heads,
                    head_dim, rotate=self.position.rotates, write_kv=writes,
                    folded=(x.residual, x.norm.weight_f32, x.norm.eps))
                return self._attended(qkv, batch, view, residual, next_norm, sums_parts, unordered)
            turning = head_dim if rotary_dim is None else rotary_dim
            if (type(self).shape_projection is Attention.shape_projection and head_dim % 16 == 0 and turning % 16 == 0
                    and x.joins_f32(self.w_qkv)):
                qkv = ops.gemm_f32_qkv_rope(
                    x.residual, x.norm.weight_f32, x.norm.eps, self.w_qkv, self.b_qkv, self.cos, self.sin, batch.positions,
                    batch.seq_of_token, batch.seq_slot, view.block_table, view.k_pool, view.v_pool, self.num_heads,
                    self.num_kv_heads, head_dim, rotate=self.position.rotates, write_kv=writes, rotary_dim=turning)
                return self._attended(qkv, batch, view, residual, next_norm, sums_parts, unordered)
            x = x.complete()
        fused = (x.dtype == torch.bfloat16 and untouched and head_dim % 32 == 0
                 and x.shape[1] % 8 == 0 and (rows == 1 or x.stride(0) % 8 == 0))
        # (the tiles' epilogue saves the rotation's kernel)
        tiles = (choose_tiles(rows, self.w_qkv.shape[0], x.shape[1], x.stride(0), behind=BEHIND_ROTATION)
                 if fused and not few and takes_tiles(rows, x, self.w_qkv) else None)
        if tiles is not None:
            qkv = ops.gemm_tiles_rope(self.w_qkv, x, self.b_qkv, self.cos, self.sin, batch.positions, batch.seq_of_token,
                                      batch.seq_slot, view.block_table, view.k_pool, view.v_pool, self.num_heads,
                                      self.num_kv_heads, head_dim, tiles.columns, tiles.rows,
                                      rotate=self.position.rotates, write_kv=writes, direct=tiles.direct)
        elif fused and few:
            # few rows (where the hand-written product is the faster one): its epilogue rotates and writes the cache
            qkv = ops.gemm_qkv_rope(self.w_qkv, x, self.b_qkv, self.cos, self.sin, batch.positions,
                                    batch.seq_of_token, batch.seq_slot, view.block_table, view.k_pool, view.v_pool,
                                    self.num_heads, self.num_kv_heads, head_dim,
                                    rotate=self.position.rotates, write_kv=writes)
        else:
            qkv = self.shape_projection(linear(x, self.w_qkv, self.b_qkv), batch)
            ops.rope_kv_write(qkv, self.cos, self.sin, batch.positions, batch.seq_of_token, batch.seq_slot,
                              view.block_table, view.k_pool, view.v_pool, self.num_heads, self.num_kv_heads,
                              head_dim, rotate=self.position.rotates, write_kv=writes, rotary_dim=rotary_dim)
        return self._attended(qkv, batch, view, residual, next_norm, sums_parts, unordered)

    def _attended(self, qkv: torch.Tensor, batch, view, residual: Optional[torch.Tensor], next_norm, sums_parts: bool,
                  unordered: bool = False):
        """The attention of rotated heads, and the product behind it."""
        context = attend(qkv, batch, view, self.num_heads, self.num_kv_heads, self.kernel_head_dim, self.window, self.scale,
                         unmerged=(unordered or self.cuts_o) and joins_merge(qkv.shape[0], self.w_o, residual))
        if isinstance(context, Shares):
            ops.merge_project(context.part_o, context.part_ml, self.w_o, self.b_o, residual, self.num_heads, self.num_kv_heads,
                              self.kernel_head_dim, context.splits, context.tile_rows)
            return Added()
        return linear(context, self.w_o, self.b_o, into=residual, then_norm=next_norm, sums_parts=sums_parts)


WIDE_DECODE_KEYS = 2048  # contexts from which decode rows go to the four-wave form
# (the four-wave form cuts long contexts for as many workgroups as the GPU has compute units)
FEW_DECODE_UNITS = 8  # (sequence, kv head) pairs below which they do not: parts of one wave fill the GPU better
MANY_DECODE_UNITS = 96  # (sequence, kv head) pairs from which decode rows take the four-wave form at any context
MANY_PART_BYTES = 300 << 10  # keys and values of one pair below which its keys are not cut then
SOME_DECODE_UNITS = 33  # ... and from which they may with a merge of their own: whole while a pair reads no more than so many bytes,
WHOLE_UNIT_BYTES = 176 << 10
SOME_DECODE_KEYS = 48 << 10  # in parts where all pairs together have so many keys (and not as many as they may come to have)
SHARED_DECODE_KEYS = 96  # contexts from which four waves share a decode row's keys without cutting them
SPLIT_MIN_KEYS = 32  # the fewest keys of a one-wave part
SPLIT_DECODE_KEYS = 192  # contexts from which the keys of decode rows are cut into parts at all
JOINED_DECODE_ROWS = 32  # up to this many single-token sequences beside prompt portions ride in the prompt form's launch
PROMPT_SPLIT_KEYS = 512  # the fewest keys of a part when a prompt portion's keys are cut
# (cutting a prompt form's keys aims at as many workgroups as the GPU has compute units)
# Tiles of 64 rows x kv heads (as a share of the compute units) from which prompt portions take the form that shares keys and
# values through LDS, whatever is beside them; up to JOINED_DECODE_ROWS single tokens ride in the other form's launch, and have
# one of their own beside this one (8 over 2,000 keys and 600 tokens of 3B heads, 150 tiles: 25.7 us joined, 26.8).
EIGHT_WAVE_TILES = 0.75  # of the compute units
# With nothing to join from fewer tiles on, or from so many tiles times keys of the longest: few tiles have their keys cut for
# as many workgroups as the GPU has units in either form (MI355X, us, the form without LDS and this one; 3B heads: 600 tokens,
# 150 tiles, 18.1, 15.1, behind 2,000 keys 51.6, 33.2; 400 tokens, 100 tiles, 12.8, 12.1, behind 500 18.3, 19.5, 2,000 43.9, 26.7;
# 200 tokens, 50 tiles, 7.4, 9.5, behind 1,000 18.5, 18.2, 4,000 42.5, 26.2; 64 tokens, 16 tiles, behind 4,000 18.9, 19.2, 8,000 27.4,
# 21.4; five prompts of 613 tokens in all 16.7, 10.8; 16 heads on 16, 600 tokens 18.3, 14.5; 14 heads of 64 dimensions, 132 tiles,
# 10.5, 10.9, behind 1,000 25.4, 18.4).
ALONE_TILES = 0.55  # of the compute units
ALONE_TILE_KEYS = 96_000
# (A window's keys are not cut, and few tiles then have few workgroups: with pages of 16, whose table the form through LDS reads
# for every 16 keys, it is 9 % slower in the mean of 46 such batches, 135 tokens of 12 heads on 2 under a window of 4,096 73.7, 89.8;
# with larger pages 5 to 34 % faster in 46.)
WINDOW_PAGE = 32
LARGE_TILES_ABOVE = 1.0  # tiles of 128 rows x kv heads (as a share of the compute units) above which that form takes them


_SAID_GENERIC: set = set()  # geometries whose bfloat16 attention was sent to the generic kernel, each said once


def plan_splits(units: int, max_keys: int, target_waves: int = 1024, min_keys: int = 128) -> tuple[int, int]:
    """How many parts to cut a decode tile's keys into so that the GPU is filled:
    (number of splits, keys per split as a multiple of 32)."""
    wanted = max(1, target_waves // max(units, 1))
    splits = min(wanted, max(1, max_keys // min_keys))
    if splits <= 1:
        return 1, 0
    per_split = -(-(-(-max_keys // splits)) // 32) * 32
    return -(-max_keys // per_split), per_split


def takes_prompt_form(tiles: int, keys: int, singles: int, captured: bool, cus: int) -> bool:
    """Whether prompt portions of so many tiles of 64 rows x kv heads, over up to ``keys`` keys of their own and beside ``singles``
    single tokens, take the form that shares keys and values through LDS.  (A captured step's keys are known when it is replayed.)"""
    if tiles >= max(1, EIGHT_WAVE_TILES * cus):
        return True
    if tiles == 0 or 0 < singles <= JOINED_DECODE_ROWS:
        return False
    return tiles >= ALONE_TILES * cus or (not captured and tiles * keys >= ALONE_TILE_KEYS)


@dataclass
class Shares:
    """Stands where the attention's output would: the keys of a step of single tokens were cut, row m is tile m, and its parts
    are still to be merged."""

    part_o: torch.Tensor
    part_ml: torch.Tensor
    splits: int
    tile_rows: int


# The output product merges a decode step's shares itself (``ops.merge_project``) where every workgroup, which reads the shares of
# its 128 k, has no more than this many to read (of all rows, rounded up to a power of two; 512 bytes each), and where the weight
# has no more numbers than this: beyond it the sums that meet in the stream cost more than the merge kernel (MI355X, us, attention,
# merge and product apart and with the merge in the product, 1 / 8 rows over 4,000 keys: 3B heads, 4 million 15.9, 10.4 / 21.1, 16.1; 512
# shares of one row 19.7, 14.1; 7B, 13 million 19.8, 17.1 / 30.1, 26.5; 32 heads on 8 and 4,096 columns, 17 million 21.3, 20.1 / 40.9, 39.9,
# 16 rows 64.4, 64.3; 14B, 26 million 25.1, 28.3 / 45.1, 48.7).  The SiLU-gate product behind it, which then makes its norm itself, is 0 to
# 0.6 us slower (7B 1.4).
MERGE_SHARES = 512
MERGE_WEIGHT = 14 << 20


def joins_merge(rows: int, weight: torch.Tensor, residual: Optional[torch.Tensor]) -> bool:
    """Whether the output product can take the keys' shares of a step of single tokens as they are."""
    return (residual is not None and rows <= ops.MERGE_PROJECT_ROWS and weight.dtype == torch.bfloat16 and weight.is_cuda
            and weight.shape[1] % ops.MERGE_PROJECT_SLICE == 0 and weight.numel() <= MERGE_WEIGHT and weight.data_ptr() % 16 == 0
            and residual.dtype == torch.float32 and residual.is_contiguous() and tuple(residual.shape) == (rows, weight.shape[0]))


def attend(qkv: torch.Tensor, batch, view, num_heads: int, num_kv_heads: int, head_dim: int,
           window: Optional[int], scale: float, unmerged: bool = False) -> "torch.Tensor | Shares":
    """Pick the attention kernel for this step's rows.  ``unmerged``: of a step of single tokens whose keys are cut in a few
    shares (``MERGE_SHARES``) these may come back instead.

    bfloat16 with a head size the matrix-core kernel takes: sequences that bring
    one token go to the split-context decode form, prompt portions to the tiled
    form with up to 64 rows per tile (four waves per tile where pages hold at
    least 16 keys, one wave otherwise).  float32 with heads of 32 to 128
    dimensions: :func:`attend_f32`.  Everything else (other head sizes, groups of
    more than 64 heads, pages of fewer than 4 tokens): the generic kernel."""
    group = num_heads // num_kv_heads
    decode_tiles = 1 if group <= 16 else 2 if group <= 32 else 4  # 16-row tiles that hold one token's heads
    page_size = view.page_size
    cus = ops.compute_units()  # compute units of the GPU
    if (qkv.dtype == torch.float32 and head_dim in ops.F32_HEAD_DIMS and group <= ops.F32_TILE_ROWS
            and page_size >= 4 and page_size & (page_size - 1) == 0):
        return attend_f32(qkv, batch, view, num_heads, num_kv_heads, head_dim, window, scale)
    # (a token's heads of one key head share a tile: up to 64 rows, 16 where the head has 256 dimensions)
    if (qkv.dtype != torch.bfloat16 or head_dim not in ops.MFMA_HEAD_DIMS or group > (64 if head_dim <= 128 else 16)
            or page_size < 4 or page_size & (page_size - 1)):
        if qkv.dtype == torch.bfloat16 and (head_dim, group, page_size) not in _SAID_GENERIC:
            # right, and many times slower than the matrix-core forms: said once per geometry, not silently
            _SAID_GENERIC.add((head_dim, group, page_size))
            warnings.warn(f"bfloat16 attention with head size {head_dim}, {group} query heads per key head and pages of "
                          f"{page_size} takes the generic kernel (the matrix-core forms take head sizes "
                          f"{ops.MFMA_HEAD_DIMS}, up to 64 heads per key head, 16 at head size 256, and pages of a power "
                          f"of two >= 4)",
                          RuntimeWarning, stacklevel=2)
        return ops.paged_attention_generic(
            qkv, qkv.stride(0), view.k_pool, view.v_pool, view.block_table, batch.positions,
            batch.seq_of_token, batch.seq_slot, batch.tokens, num_heads, num_kv_heads, head_dim, window, scale)
    out = torch.empty((batch.tokens, num_heads * head_dim), dtype=qkv.dtype, device=qkv.device)
    common = (batch.seq_slot, batch.seq_start, batch.seq_q_len, batch.q_start_loc, out, num_heads, num_kv_heads,
              head_dim, window, scale)
    max_keys = batch.max_context if window is None else min(batch.max_context, window + 64)
    wide = page_size >= 16 and scale > 0
    # Prompt portions with enough rows take tiles of 128 rows and eight waves, whose keys and values pass
    # through LDS once per tile.  (A short portion behind a long context also has its keys cut into parts.)
    prompt_tokens, prompt_keys, singles = batch.portions
    if window is not None:
        prompt_keys = min(prompt_keys, window + 64) if page_size >= WINDOW_PAGE else 0
    bound = batch.static_plan.max_keys if batch.static_plan is not None else max_keys
    cuts = max(1, bound // PROMPT_SPLIT_KEYS) if wide and window is None else 1  # (a window's keys stay whole)
    big_tiles = -(-prompt_tokens * group // 128) * num_kv_heads
    small_tiles = -(-prompt_tokens * group // 64) * num_kv_heads
    # That form has tiles of 128 rows for eight waves, and tiles of 64 rows for four, two such workgroups to a
    # compute unit, where the larger tiles would not give every unit more than one (isolated kernel, us, 128 rows
    # -> 64: 2,048 tokens of one prompt, 3B heads, 256 large tiles: 50.8 -> 46.8, 1,024 tokens 27.5 -> 24.8; 7B
    # heads, 456 large tiles: 55.3 -> 70.5; heads of 64 dimensions, where the softmax arithmetic per key is the same
    # and the products are half: 2,048 tokens 40.2 -> 33.0, against 43.1 in the form of four waves without LDS).
    eight = (wide and head_dim in (64, 128) and group <= 64
             and takes_prompt_form(small_tiles, prompt_keys, singles, batch.static_plan is not None, cus))
    lds_row_tiles = 8 if head_dim == 128 and big_tiles > LARGE_TILES_ABOVE * cus else 4

    def decode_form(bound: int, units: int, room: int) -> tuple[int, dict]:
        joined = room > 0  # (up to so many shares of a unit come back unmerged)
        # Decode rows, `units` (sequence, kv head) pairs over up to `bound` keys.  Long contexts: four waves
        # per (sequence, kv head, part of the keys) take the part's blocks in turn with their loads running
        # ahead (15.8 against 18.1 us for 8 x 4,096 keys).  A few pairs do not fill the GPU that way: they take the
        # one-wave form below, whose parts are smaller (one sequence of the 3B shape over 32,000 keys: 333 -> 363
        # tokens/s; from four sequences on the forms are level).  Where the output product merges the shares (``joined``) it
        # reads every one of them: there the line is the number of keys in all, and a unit has no more shares than are needed for a
        # workgroup each (MI355X, us, attention and output product, with parts of one wave down to 32 keys and so: 8 rows of 16
        # heads on 2 over 1,600 keys 15.7 -> 13.4, 16 rows over 1,000 17.4 -> 14.4, 2,000 20.6 -> 17.7; heads of 64 13.7 -> 10.6,
        # 14.6 -> 10.7, 17.1 -> 12.0; 28 heads on 4, 8 rows over 1,000 21.5 -> 20.0; one wave and four level at 8 rows over 1,000).
        if wide and units >= FEW_DECODE_UNITS and (bound >= WIDE_DECODE_KEYS or (
                joined and units < MANY_DECODE_UNITS and units * bound >= FEW_DECODE_UNITS * WIDE_DECODE_KEYS)):
            return ops.TILE_WAVES, dict(target_waves=cus, min_keys=64 if joined else 32 * ops.TILE_WAVES)
        # ... and with a merge of its own from some dozens of pairs on: whole where a pair has little to read, four waves where
        # all have much (us, merge with it, one wave's parts, four waves whole, four waves' parts: 24 rows of 14 heads of 64 on 2 over 300
        # keys 7.9, 6.3, 9.0, 640 10.4, 9.1, 10.3, 1,600 14.5, 14.6, 12.1; of 16 heads of 128 on 2 over 300 9.0, 9.1, 10.4, 640 11.9, 13.6,
        # 12.6, 1,600 17.9, 25.1, 16.5; 32 rows 9.6, 9.3, 11.0, 12.9, 13.9, 13.1, 21, 25.9, 19.4).  Not by a captured step's bound: over
        # few keys the four waves' parts are the slower form whatever the bound (32 rows, bound 1,500, one wave's parts and four waves'
        # over 60 keys 7.9, 9.6, 300 9.2, 10.6, 1,000 15.3, 15.3).
        if wide and not joined and SOME_DECODE_UNITS <= units < MANY_DECODE_UNITS:
            if SHARED_DECODE_KEYS <= bound <= WHOLE_UNIT_BYTES // (4 * head_dim):
                return ops.TILE_WAVES, dict(target_waves=cus, min_keys=bound + 1)
            if batch.static_plan is None and units * bound >= SOME_DECODE_KEYS:
                return ops.TILE_WAVES, dict(target_waves=cus, min_keys=32 * ops.TILE_WAVES)
        # Many pairs fill the GPU by themselves: the same form with the keys whole or in large parts
        # (64 sequences x 2 heads x 256 keys: 9.2 us against 11.1 us with one wave per part).  A second part pays for
        # its merge where a unit has more to read than MANY_PART_BYTES (64 x 2 heads of 128, us, whole against two
        # parts: 512 keys 12.5, 15.5; 1,024 keys 20.2, 21.5; 1,200 keys 24.7, 24.1; 1,536 keys 29.6, 28.0; 48 x 2
        # heads: 700 keys 14.8, 15.7; 1,024 keys 19.8, 18.8; 64 x 2 heads of 64: 1,280 keys 14.1, 16.5; the two parts
        # joined by a workgroup a row).  A captured step's bound is the longest context it may ever see: a limit of
        # WIDE_DECODE_KEYS and more has the form above, with 1,000 keys as with many (64 x 2 heads of 128 over 1,000 keys:
        # 19 us at a bound of 1,000, 22 at 4,096).
        if wide and units >= MANY_DECODE_UNITS and bound >= SHARED_DECODE_KEYS:
            return ops.TILE_WAVES, dict(target_waves=4 * cus // ops.TILE_WAVES,
                                        min_keys=max(512, MANY_PART_BYTES // (4 * head_dim)))
        # Otherwise one wave per part, parts down to one block of 32 keys (8 x 256 keys: 7.3 us in 8 parts,
        # 10.2 us in 2; 8 x 512 keys: 8.1 us in 16 parts, 10.6 us in 4) ...
        if bound >= SPLIT_DECODE_KEYS:
            # (joined: shares of 128 keys and less only while all of them are fewer than the units; one row of 16 heads on 2 over
            # 1,000 keys at a bound of 32,768 14.3 -> 11.8 us, over 32,000 20.5 -> 19.7; 8 rows over 800 keys 13.2 -> 12.0, 16 over 400 13.9 -> 12.7)
            most = min(4 * cus, max(cus, units * (bound // 128))) if joined else 4 * cus
            # (a few pairs at a limit that gives more parts than the product takes: four waves a part, and as many parts as its threads read
            # in whole turns, a power of two; with a merge of their own and so, a bound of 32,768, over 300 / 8,000 / 32,000 keys, 8 heads
            # of 128 on 1, 4 rows 15.3, 20.3, 30.9 -> 11.1, 17.3, 29.4 us, 5 rows 15.2, 21.2, 35.1 -> 10.8, 16.0, 30.7; of 64 14.1, 18.4, 27.5
            # -> 10.0, 12.5, 19.8; 16 heads on 2, 3 rows 15.7, 21.8, 38.0 -> 10.8, 15.9, 31.3.  85 parts of 3 rows 23.8 over 16,000, 64 20.1)
            if joined and plan_splits(units, bound, most, SPLIT_MIN_KEYS)[0] > room:
                if wide:
                    return ops.TILE_WAVES, dict(target_waves=units << (cus // units).bit_length() - 1, min_keys=64)
                most = 4 * cus
            return 1, dict(target_waves=most, min_keys=SPLIT_MIN_KEYS)
        # ... and below some 200 keys, where the merge costs more than it saves, four waves that share a
        # sequence's few blocks inside one workgroup instead of one wave that takes them in turn
        # (8 x 128 keys: 6.5 against 6.9 us, 8 x 160: 7 against 11)
        return (ops.TILE_WAVES if wide and bound >= SHARED_DECODE_KEYS else 1), dict(target_waves=4 * cus, min_keys=bound + 1)

    def shares_taken(rows: int) -> int:
        return MERGE_SHARES >> (rows - 1).bit_length() if unmerged and rows == batch.tokens else 0

    def leave(n_splits: int, rows: int) -> bool:
        return 1 < n_splits <= shares_taken(rows)

    plan = batch.static_plan
    longest_dev = None
    if plan is not None:
        # a captured step: grids are fixed, lengths live on the device.  Its first sequences bring one token
        # each (tile i is sequence i, no tile lists); the sizes of the keys' parts follow the step's longest
        # context, which the device knows, within the bound the step was captured for
        max_keys = plan.max_keys if window is None else min(plan.max_keys, window + 64)
        longest_dev = plan.max_context
        decode_rows = batch.sequences if plan.decode_rows is None else plan.decode_rows
        joined = wide and not eight and 0 < decode_rows <= JOINED_DECODE_ROWS and decode_rows < batch.sequences
        if decode_rows and not joined:
            decode_waves, split_options = decode_form(max_keys, decode_rows * num_kv_heads, shares_taken(decode_rows))
            units = decode_rows * num_kv_heads
            n_splits, _ = plan_splits(units, max_keys, **split_options)
            if n_splits > 1 and decode_waves > 1:
                # (the device sizes the parts: as many as asked for, where the bound's own would come out fewer, as 1,040 keys in 8 of
                # 160 do: 8 rows of 28 heads on 4 over 1,000 keys 19.7 us in 7, 19.3 in 8)
                n_splits = min(split_options["target_waves"] // units, max_keys // split_options["min_keys"])
            part_o = part_ml = None
            if n_splits > 1:
                part_o, part_ml = _workspaces(qkv.device, units * n_splits, 16 * decode_tiles, head_dim)
            ops.paged_attention_mfma(qkv, qkv.stride(0), view.k_pool, view.v_pool, view.block_table, None,
                                     None, decode_rows, *common, tokens_per_tile=1, row_tiles=decode_tiles,
                                     n_splits=n_splits, max_context_dev=longest_dev, part_o=part_o, part_ml=part_ml,
                                     tile_waves=decode_waves, merge=not leave(n_splits, decode_rows))
            if leave(n_splits, decode_rows):
                return Shares(part_o, part_ml, n_splits, 16 * decode_tiles)
        if decode_rows == batch.sequences:
            return out
        n_tiles = 0  # (of the eager decode form below)
    else:
        tile_seq, tile_q0, n_tiles = batch.tiles(1, decode=True)
        # A few single tokens beside prompt portions: one launch (and one merge) of the prompt form for all
        # sequences instead of two of each (8 decode rows and a 64-token portion of the 3B shape: 4.84 -> 4.49 ms
        # a step; 32 rows over 3,000 keys and 256 tokens: 8.9 -> 8.2 ms; with 64 such rows the forms are level)
        # (not beside the form of eight waves, where a tile of one token would leave six of them idle)
        joined = wide and not eight and 0 < n_tiles <= JOINED_DECODE_ROWS and n_tiles < batch.sequences
    if n_tiles and not joined:
        decode_waves, split_options = decode_form(max_keys, n_tiles * num_kv_heads, shares_taken(n_tiles))
        n_splits, per_split = plan_splits(n_tiles * num_kv_heads, max_keys, **split_options)
        part_o = part_ml = None
        if n_splits > 1:
            part_o, part_ml = _workspaces(qkv.device, n_tiles * num_kv_heads * n_splits, 16 * decode_tiles, head_dim)
        ops.paged_attention_mfma(qkv, qkv.stride(0), view.k_pool, view.v_pool, view.block_table, tile_seq, tile_q0,
                                 n_tiles, *common, tokens_per_tile=1, row_tiles=decode_tiles, n_splits=n_splits,
                                 keys_per_split=per_split, part_o=part_o, part_ml=part_ml, tile_waves=decode_waves,
                                 merge=not leave(n_splits, n_tiles))
        if leave(n_splits, n_tiles):
            return Shares(part_o, part_ml, n_splits, 16 * decode_tiles)
    if wide:
        # the prompt forms: waves share a tile's keys.  More rows per tile re-use each key more often,
        # fewer tiles leave compute units idle: the most rows that still give most units a workgroup, where a
        # short portion behind a long context also has its keys cut (256 tokens behind 3,840 keys, 2 kv heads:
        # 34 us with 64 rows per tile and four parts, 48 us with 16 rows per tile and the keys whole)
        if eight:
            tile_waves, row_tiles = ops.PROMPT_WAVES, lds_row_tiles
        else:
            tile_waves = ops.TILE_WAVES
            row_tiles = 4 if head_dim <= 128 else 1
            while row_tiles > 1 and -(-prompt_tokens * group // (16 * row_tiles)) * num_kv_heads * cuts < 0.75 * cus:
                row_tiles //= 2
    else:
        # one wave per tile; fewer rows where that would leave SIMDs without a wave (about a thousand
        # waves fill the GPU) or where the accumulators of a wide head would spill
        tile_waves = 1
        row_tiles = 2 if head_dim > 128 else 4
        while row_tiles > 1 and (prompt_tokens * group // (16 * row_tiles)) * num_kv_heads < 4 * cus:
            row_tiles //= 2
    while 16 * row_tiles < group:
        row_tiles *= 2
    per_tile = (16 * row_tiles) // group
    tile_seq, tile_q0, n_tiles = batch.tiles(per_tile, decode=None if joined else False)
    if n_tiles:
        # few tiles and many keys: parts of the keys, about as many workgroups as compute units
        n_splits, per_split, part_o, part_ml = 1, 0, None, None
        wanted = min(cuts, int(cus / (n_tiles * num_kv_heads) + 0.5))
        if wanted > 1:
            per_split = -(-(-(-max_keys // wanted)) // 128) * 128
            n_splits = -(-max_keys // per_split)
        if n_splits > 1:
            part_o, part_ml = _workspaces(qkv.device, n_tiles * num_kv_heads * n_splits, 16 * row_tiles, head_dim)
        else:
            per_split = 0
        ops.paged_attention_mfma(qkv, qkv.stride(0), view.k_pool, view.v_pool, view.block_table, tile_seq, tile_q0,
                                 n_tiles, *common, tokens_per_tile=per_tile, row_tiles=row_tiles,
                                 n_splits=n_splits, keys_per_split=per_split, part_o=part_o, part_ml=part_ml,
                                 tile_waves=tile_waves, max_context_dev=longest_dev if n_splits > 1 else None)
    return out


# Float32: contexts up to which single tokens take the prompt form too (a workgroup's two blocks of 64 keys in turn cost
# less than the second kernel that joins blocks)
F32_WHOLE_KEYS = 128
F32_CUT_TILES = 0.6  # tiles a compute unit up to which prompts' tiles may be cut into blocks
F32_CUT_BYTES = 64 << 20  # ... and the bytes that their blocks may take


def attend_f32(qkv: torch.Tensor, batch, view, num_heads: int, num_kv_heads: int, head_dim: int,
               window: Optional[int], scale: float) -> torch.Tensor:
    """Attention in true float32 on the matrix cores: single tokens in blocks of keys (a wave each, joined behind),
    prompt portions a workgroup per 64 rows, or in blocks too where there are few such tiles of many blocks."""
    out = torch.empty((batch.tokens, num_heads * head_dim), dtype=qkv.dtype, device=qkv.device)
    group = num_heads // num_kv_heads
    per_tile = ops.F32_TILE_ROWS // group
    cus = ops.compute_units()
    plan = batch.static_plan
    bound = plan.max_keys if plan is not None else batch.max_context
    common = (batch.seq_slot, batch.seq_start, batch.seq_q_len, batch.q_start_loc, out, num_heads, num_kv_heads, head_dim,
              window, scale)

    def run(tiles: tuple, tokens: int, whole: bool = False, decode: bool = False) -> None:
        tile_seq, tile_q0, n_tiles = tiles
        blocks = -(-bound // ops.F32_BLOCK_KEYS)
        if window is not None:  # (a window may begin inside a block)
            blocks = min(blocks, -(-(window + tokens) // ops.F32_BLOCK_KEYS) + 1)
        rows = tokens * group
        block_bytes = num_kv_heads * rows * (head_dim + 2) * 4
        # Whole tiles take some 8.3 us a block of the longest tile, tiles in blocks 0.055 us a block of all of them and 8 more
        # (the parts' way through memory), over 256 units (us, whole against in blocks, 16 heads of 128 on 2: a prompt of
        # 130 tokens 30, 24; 256 tokens 39, 31; 517 tokens 79, 66; 1,024 tokens 138, 160; 8 prompts of 64 tokens 16, 36; 8 of
        # 128 25, 68; 14 heads of 64 on 2: 600 tokens 51, 40)
        units = F32_CUT_TILES * cus - n_tiles * num_kv_heads
        launch = functools.partial(ops.paged_attention_f32, qkv, qkv.stride(0), view.k_pool, view.v_pool, view.block_table,
                                   tile_seq, tile_q0, n_tiles, *common, tokens)
        if whole or (tokens > 1 and (blocks * units <= F32_CUT_TILES * cus
                                     or n_tiles * blocks * block_bytes > F32_CUT_BYTES)):
            launch()
            return
        places, capacity, rounds = n_tiles * blocks, 0, 1
        if places * block_bytes > ops.F32_WORKSPACE_BYTES:
            # Sequences of very different lengths, or a captured step whose bound is far above its contexts: the tiles'
            # blocks lie packed, as many as the keys that are there need (64 sequences of 100 / 1,000 keys in a step captured
            # for 131,072: 23 / 51 us, where workspaces of 64 MB that three tiles of 2,048 blocks at a time shared took 370 / 403
            # and the generic kernel 35 / 298).
            # The host counts an eager step's rounds; of a captured step it knows none, so one round runs, and
            # whole tiles what begins behind it (millions of cached tokens in one step).
            capacity = max(blocks, ops.F32_WORKSPACE_BYTES // block_bytes - blocks)
            places = capacity + blocks
            if plan is None:
                size, sight = ops.F32_BLOCK_KEYS, batch.max_context if window is None else window
                taken = [(start + min(first + tokens, n) - 1) // size - max(0, start + first + 1 - sight) // size + 1
                         for start, n in zip(batch.host_starts, batch.host_q_lens) if (n == 1) == decode
                         for first in range(0, n, tokens)]
                rounds = -(-sum(taken) // capacity)
        part_o = torch.empty(places * num_kv_heads * rows * head_dim, dtype=torch.float32, device=qkv.device)
        part_ml = torch.empty(places * num_kv_heads * rows * 2, dtype=torch.float32, device=qkv.device)
        waves = n_tiles * num_kv_heads * -(-rows // 16)  # (some 16 waves a unit; more blocks than that are taken in turn)
        for turn in range(rounds):
            launch(turns=min(blocks, max(1, -(-16 * cus // waves))), blocks=blocks, part_o=part_o, part_ml=part_ml,
                   capacity=capacity, round=turn)
        if capacity and plan is not None:
            launch(capacity=capacity, blocks=blocks, round=rounds)

    single = batch.sequences if plan is not None and plan.decode_rows is None else plan.decode_rows if plan is not None else None
    if bound <= F32_WHOLE_KEYS:
        run((None, None, batch.sequences) if single == batch.sequences else batch.tiles(per_tile, decode=None), per_tile, whole=True)
        return out
    tiles = (None, None, single) if single is not None else batch.tiles(1, decode=True)
    if tiles[2]:
        run(tiles, 1, decode=True)
    if single != batch.sequences:
        tiles = batch.tiles(per_tile, decode=False)
        if tiles[2]:
            run(tiles, per_tile)
    return out


def _workspaces(device: torch.device, units: int, rows: int, head_dim: int) -> tuple[torch.Tensor, torch.Tensor]:
    return (torch.empty(units * rows * head_dim, dtype=torch.float32, device=device),
            torch.empty(units * rows * 2, dtype=torch.float32, device=device))


register_part("mixer", "attention", Attention)
