"""Python faces of the HIP entry points.

Every function checks on the host what the kernel and its grid assume (device,
dtype, contiguity, shapes, index ranges that are known on the host) and raises
``ValueError`` with the offending value otherwise: a kernel is never launched
on operands it was not written for.  Kernels run on torch's current stream.
"""

from __future__ import annotations

import contextlib
import functools
import math

from typing import Optional

import torch

from .library import load_library

F32, BF16 = 0, 1
_CODES = {torch.float32: F32, torch.bfloat16: BF16}
_ERRORS = {1: "bad argument (a size or option the kernel does not take)", 2: "kernel launch failed",
           3: "more than the entry point's fixed scratch memory holds", 4: "the library's device memory was not found"}


class KernelError(RuntimeError):
    pass


_COMPUTE_UNITS: dict[int, int] = {}


def compute_units(device: "torch.device | int | None" = None) -> int:
    """Compute units of the GPU the kernels run on, asked of the device once (the plans that spread
    workgroups over the units are made from it); 256, an MI355X's, where no GPU is visible."""
    if device is None and _COMPUTE_UNITS:  # (asked several times a layer)
        known = _COMPUTE_UNITS.get(torch._C._cuda_getDevice())
        if known is not None:
            return known
    if not torch.cuda.is_available():
        return 256
    index = torch.cuda.current_device() if device is None else torch.device(device).index if not isinstance(device, int) else device
    index = torch.cuda.current_device() if index is None else index
    if index not in _COMPUTE_UNITS:
        _COMPUTE_UNITS[index] = torch.cuda.get_device_properties(index).multi_processor_count
    return _COMPUTE_UNITS[index]


def _code(dtype: torch.dtype) -> int:
    try:
        return _CODES[dtype]
    except KeyError:
        raise ValueError(f"kernels take float32 or bfloat16, got {dtype}") from None


def _gpu(name: str, tensor: torch.Tensor, dtype: Optional[torch.dtype] = None, dims: Optional[int] = None) -> None:
    if not tensor.is_cuda:
        raise ValueError(f"{name} must live on the GPU, is on {tensor.device}")
    if not tensor.is_contiguous():
        raise ValueError(f"{name} must be contiguous")
    if dtype is not None:
        if not (tensor.dtype == dtype):
            raise ValueError(f"{name} must be {dtype}, is {tensor.dtype}")
    if dims is not None:
        if not (tensor.dim() == dims):
            raise ValueError(f"{name} must have {dims} dims, has shape {tuple(tensor.shape)}")


# Arguments go to the library as plain Python numbers: the entry points' argument types are declared
# when the library is loaded (kernels/library.py), and ctypes converts them itself.
def _ptr(tensor: Optional[torch.Tensor]) -> Optional[int]:
    return None if tensor is None else tensor.data_ptr()


def _stream() -> int:
    # the raw handle of torch's current stream (also the capturing one), without building a Stream object
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _run(name: str, code: int) -> None:
    if code != 0:
        raise KernelError(f"{name}: {_ERRORS.get(code, f'error {code}')}")


_i = int
_f = float


def _row_view(name: str, t: torch.Tensor, shape: tuple, dtypes: tuple) -> None:
    """A GPU matrix whose rows are in one piece each and may lie apart."""
    if not (t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.dtype in dtypes and tuple(t.shape) == tuple(shape)
            and (t.shape[0] <= 1 or t.stride(0) >= t.shape[1])):
        raise ValueError(f"{name} must be a {list(shape)} GPU view with unit inner stride in one of {dtypes}, is "
                         f"{tuple(t.shape)} {t.dtype} with strides {t.stride()}")


def _ld(t: torch.Tensor) -> int:
    """The distance of a view's rows (a single row has none of its own)."""
    return t.stride(0) if t.shape[0] > 1 else max(t.stride(0), t.shape[1])


def _check_pools(k_pool: torch.Tensor, v_pool: torch.Tensor, dtype: torch.dtype, kv_heads: int,
                 head_dim: int) -> int:
    """Keys [pages, Hkv, page_size, D], values transposed [pages, Hkv, D, page_size]; returns page_size."""
    _gpu("k_pool", k_pool, dtype, 4)
    _gpu("v_pool", v_pool, dtype, 4)
    pages, heads, page_size, dim = k_pool.shape
    if not (heads == kv_heads and dim == head_dim):
        raise ValueError(f"k_pool {tuple(k_pool.shape)} does not match Hkv={kv_heads}, D={head_dim}")
    if not (tuple(v_pool.shape) == (pages, kv_heads, head_dim, page_size)):
        raise ValueError(f"v_pool {tuple(v_pool.shape)} must be {(pages, kv_heads, head_dim, page_size)}")
    return page_size


# ---------------------------------------------------------------------------
def embed(table: torch.Tensor, ids: torch.Tensor, out: Optional[torch.Tensor] = None,
          feed: Optional[torch.Tensor] = None, pool: Optional[torch.Tensor] = None, scale: float = 1.0,
          rows: Optional[torch.Tensor] = None, ids_out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[t] = float32(table[ids[t]]) * scale``; ids int32 [T] (already checked against the vocabulary).
    With ``feed`` (int32 [T]) and ``pool`` (int32): row t takes ``pool[feed[t]]`` as its id where
    ``feed[t] >= 0`` (tokens another kernel left on the device; ``feed[t]`` must index ``pool``).
    ``rows`` ([T, hidden] in the table's dtype; a view whose rows lie apart is fine) also takes the same values, rounded
    to that dtype.  ``ids_out`` (int32 [T]) takes every row's token as it was taken."""
    _gpu("table", table, dims=2)
    _gpu("ids", ids, torch.int32, 1)
    vocab, hidden = table.shape
    tokens = ids.shape[0]
    if feed is not None:
        _gpu("feed", feed, torch.int32, 1)
        if pool is None or feed.shape[0] < tokens:
            raise ValueError("feed needs a pool and one entry per token")
        _gpu("pool", pool, torch.int32, 1)
    if out is None:
        out = torch.empty((tokens, hidden), dtype=torch.float32, device=table.device)
    _gpu("out", out, torch.float32, 2)
    if not (out.shape == (tokens, hidden)):
        raise ValueError(f"out must be {(tokens, hidden)}, is {tuple(out.shape)}")
    if rows is not None:
        _row_view("rows", rows, (tokens, hidden), (table.dtype,))
    if ids_out is not None:
        _gpu("ids_out", ids_out, torch.int32, 1)
        if ids_out.shape[0] != tokens:
            raise ValueError(f"ids_out must be [{tokens}]")
    _run("cie_embed", load_library().cie_embed(_stream(), _i(_code(table.dtype)), _ptr(table), _ptr(ids), _ptr(feed),
                                               _ptr(pool if feed is not None else None), _ptr(out), _ptr(rows),
                                               _ld(rows) if rows is not None else 0, _i(tokens), _i(hidden), _i(vocab),
                                               _f(scale), _ptr(ids_out)))
    return out


def embed_normed(table: torch.Tensor, ids: torch.Tensor, weight: torch.Tensor, eps: float,
                 feed: Optional[torch.Tensor] = None, pool: Optional[torch.Tensor] = None, scale: float = 1.0,
                 next_weight: Optional[torch.Tensor] = None, ids_out: Optional[torch.Tensor] = None
                 ) -> tuple[torch.Tensor, Optional[torch.Tensor]]:
    """The embedding's rows (as :func:`embed` takes them) under an RMS norm, as a float32 stream [T, hidden], and, with
    ``next_weight`` (float32 [hidden]), the RMS norm of that stream under it, in the table's dtype."""
    _gpu("table", table, dims=2)
    _gpu("ids", ids, torch.int32, 1)
    vocab, hidden = table.shape
    tokens = ids.shape[0]
    if feed is not None:
        _gpu("feed", feed, torch.int32, 1)
        if pool is None or feed.shape[0] < tokens:
            raise ValueError("feed needs a pool and one entry per token")
        _gpu("pool", pool, torch.int32, 1)
    for name, w in (("weight", weight), ("next_weight", next_weight)):
        if w is not None:
            _gpu(name, w, torch.float32, 1)
            if w.shape[0] != hidden:
                raise ValueError(f"{name} must be [{hidden}], is {tuple(w.shape)}")
    if hidden > MAX_NORM_WIDTH or not eps > 0:
        raise ValueError(f"rows of {hidden} numbers (at most {MAX_NORM_WIDTH}), eps {eps}")
    if ids_out is not None:
        _gpu("ids_out", ids_out, torch.int32, 1)
        if ids_out.shape[0] != tokens:
            raise ValueError(f"ids_out must be [{tokens}]")
    out = torch.empty((tokens, hidden), dtype=torch.float32, device=table.device)
    normed = torch.empty((tokens, hidden), dtype=table.dtype, device=table.device) if next_weight is not None else None
    _run("cie_embed_normed", load_library().cie_embed_normed(
        _stream(), _i(_code(table.dtype)), _ptr(table), _ptr(ids), _ptr(feed), _ptr(pool if feed is not None else None),
        _ptr(weight), _ptr(out), _ptr(ids_out), _ptr(next_weight), _ptr(normed), _i(tokens), _i(hidden), _i(vocab), _f(scale),
        _f(eps)))
    return out, normed


def table_rows(plan: torch.Tensor, rows: int, table: torch.Tensor) -> None:
    """Write entries of ``rows`` rows of a block table: ``plan`` (int32) holds (row, first entry, how many, where they begin in
    ``plan``) of each, and the entries behind them.  The caller vouches for the places."""
    _gpu("plan", plan, torch.int32, 1)
    _gpu("table", table, torch.int32, 2)
    if not (1 <= rows and plan.shape[0] >= 4 * rows):
        raise ValueError(f"a plan of {plan.shape[0]} numbers does not describe {rows} rows")
    _run("cie_table_rows", load_library().cie_table_rows(_stream(), _ptr(plan), _i(rows), _ptr(table), _i(table.shape[1])))


def clear_rows(states: torch.Tensor, slots: torch.Tensor, most_bytes: int) -> None:
    """Zero rows ``slots`` (int32) of every state in ``states`` (int64 [n, 2]: its address, a multiple of 16, and the bytes of a
    row, the largest of which is ``most_bytes``).  The caller vouches for addresses and slots."""
    _gpu("states", states, torch.int64, 2)
    _gpu("slots", slots, torch.int32, 1)
    if not (states.shape[0] >= 1 and states.shape[1] == 2 and slots.shape[0] >= 1 and most_bytes >= 2):
        raise ValueError(f"states {tuple(states.shape)}, slots {tuple(slots.shape)}, {most_bytes} bytes")
    _run("cie_clear_rows", load_library().cie_clear_rows(
        _stream(), _ptr(states), _i(states.shape[0]), _ptr(slots), _i(slots.shape[0]), _i(most_bytes)))


STEP_ROWS = 128  # rows of a captured decode step whose numbers travel as a kernel's arguments


def step_rows(values: "array.array", n: int, size: int, fed: bool, max_context: int, pad_slot: int, token_ids: torch.Tensor,
              positions: torch.Tensor, seq_start: torch.Tensor, seq_slot: torch.Tensor, token_feed: torch.Tensor,
              max_context_at: torch.Tensor, result_at: Optional[torch.Tensor] = None, result: Optional[torch.Tensor] = None) -> None:
    """Write what changes between two replays of a captured decode step of ``size`` rows: ``values`` (a host array of C ints)
    holds its ``n`` tokens, positions and slots and, if ``fed``, the places of the token pool they are taken from.  Rows beyond
    ``n`` become padding on ``pad_slot``.  ``result_at`` (int64 [1]) takes the address of ``result``, which the step's last product
    writes to."""
    if (result_at is None) != (result is None) or (result_at is not None and not (
            result_at.is_cuda and result_at.dtype == torch.int64 and result_at.numel() == 1 and result.is_cuda)):
        raise ValueError("a result and the place of its address come together")
    if not (values.typecode == "i" and values.itemsize == 4 and len(values) == (4 if fed else 3) * n and 0 <= n <= size <= STEP_ROWS):
        raise ValueError(f"{len(values)} numbers for {n} of {size} rows")
    for at, least in ((token_ids, size), (positions, size), (seq_start, size), (seq_slot, size), (token_feed, size), (max_context_at, 1)):
        if not (at.is_cuda and at.dtype == torch.int32 and at.is_contiguous() and at.numel() >= least):
            raise ValueError(f"a place of {size} int32 numbers is {tuple(at.shape)} {at.dtype}")
    _run("cie_step_rows", load_library().cie_step_rows(
        _stream(), values.buffer_info()[0], _i(n), _i(size), _i(fed), _i(max_context), _i(pad_slot), _ptr(token_ids), _ptr(positions),
        _ptr(seq_start), _ptr(seq_slot), _ptr(token_feed), _ptr(max_context_at), _ptr(result_at), _ptr(result)))


def _result_at(out_at: torch.Tensor) -> None:
    if not (out_at.is_cuda and out_at.dtype == torch.int64 and out_at.numel() == 1):
        raise ValueError("the place of a result's address is one int64 number on the GPU")


MAX_NORM_WIDTH = 16384  # a row of the norm kernels is held in 64 KB of LDS as float32


def add_rmsnorm(residual: torch.Tensor, branch: Optional[torch.Tensor], weight: torch.Tensor, eps: float,
                out_dtype: torch.dtype, rows: Optional[torch.Tensor] = None,
                out: Optional[torch.Tensor] = None, parts: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``residual += branch`` (if given; written back unless ``rows``), then RMS-normalise.

    residual float32 [T, H]; branch and the result in ``out_dtype``; weight [H]
    in ``out_dtype`` or float32.  ``parts`` (float32 [P, T, H]) join the residual too, one after the other.  With ``rows`` (int32 [n]) only those rows are
    produced, in that order, and the residual is left as it is."""
    _gpu("residual", residual, torch.float32, 2)
    tokens, hidden = residual.shape
    _gpu("weight", weight, dims=1)
    if not (weight.shape[0] == hidden):
        raise ValueError(f"weight must be [{hidden}], is {tuple(weight.shape)}")
    if not (weight.dtype in (out_dtype, torch.float32)):
        raise ValueError(f"weight dtype {weight.dtype} does not fit {out_dtype}")
    if not (hidden <= MAX_NORM_WIDTH):
        raise ValueError(f"hidden size {hidden} exceeds the norm kernel's {MAX_NORM_WIDTH}")
    if not (eps > 0):
        raise ValueError(f"eps must be positive, is {eps}")
    if branch is not None:
        _gpu("branch", branch, out_dtype, 2)
        if not (branch.shape == residual.shape):
            raise ValueError(f"branch {tuple(branch.shape)} vs residual {tuple(residual.shape)}")
    if parts is not None:
        _gpu("parts", parts, torch.float32, 3)
        if not (parts.shape[1:] == residual.shape):
            raise ValueError(f"parts {tuple(parts.shape)} vs residual {tuple(residual.shape)}")
    if rows is not None:
        _gpu("rows", rows, torch.int32, 1)
        n_out = rows.shape[0]
    else:
        n_out = tokens
    if out is None:
        out = torch.empty((n_out, hidden), dtype=out_dtype, device=residual.device)
    _gpu("out", out, out_dtype, 2)
    if not (out.shape == (n_out, hidden)):
        raise ValueError(f"out must be {(n_out, hidden)}, is {tuple(out.shape)}")
    _run("cie_add_rmsnorm", load_library().cie_add_rmsnorm(
        _stream(), _i(_code(out_dtype)), _i(_code(weight.dtype)), _ptr(residual), _ptr(branch), _ptr(weight),
        _ptr(out), _ptr(rows), _i(n_out), _i(hidden), _f(eps), _i(0 if rows is not None else 1), _ptr(parts),
        _i(0 if parts is None else parts.shape[0]), _i(tokens)))
    return out


def rmsnorm_from_sumsq(residual: torch.Tensor, sumsq: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """bf16 RMSNorm of float32 rows whose partial sums of squares ``sumsq`` [rows, parts] are known."""
    _gpu("residual", residual, torch.float32, 2)
    rows, hidden = residual.shape
    _gpu("sumsq", sumsq, torch.float32, 2)
    if not (sumsq.shape[0] >= rows):
        raise ValueError(f"sumsq has {sumsq.shape[0]} rows for {rows}")
    _gpu("weight", weight, dims=1)
    if not (weight.shape[0] == hidden and weight.dtype in (torch.bfloat16, torch.float32)):
        raise ValueError("norm weight does not fit")
    if not (eps > 0):
        raise ValueError(f"eps must be positive, is {eps}")
    out = torch.empty((rows, hidden), dtype=torch.bfloat16, device=residual.device)
    _run("cie_rmsnorm_from_sumsq", load_library().cie_rmsnorm_from_sumsq(
        _stream(), _i(_code(weight.dtype)), _ptr(residual), _ptr(sumsq), _i(sumsq.shape[1]), _ptr(weight), _ptr(out),
        _i(rows), _i(hidden), _f(eps)))
    return out


def rope_kv_write(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                  seq_of_token: torch.Tensor, seq_slot: torch.Tensor, block_table: torch.Tensor,
                  k_pool: torch.Tensor, v_pool: torch.Tensor, q_heads: int, kv_heads: int, head_dim: int,
                  rotate: bool = True, write_kv: bool = True, rotary_dim: Optional[int] = None) -> None:
    """Rotate q (in place) and k, write k and v of every token into its cache slot.

    qkv [T, (Hq+2Hkv)*D]; the first ``rotary_dim`` dimensions of every head rotate (all of them if
    ``None``), dimension i with i + rotary_dim/2, the rest pass through; cos/sin float32
    [max_position, rotary_dim/2]; key pool [pages, Hkv, page_size, D] and value pool
    [pages, Hkv, D, page_size] in qkv's dtype; block_table int32 [slots, width]."""
    _gpu("qkv", qkv, dims=2)
    tokens = qkv.shape[0]
    if not (qkv.shape[1] == (q_heads + 2 * kv_heads) * head_dim):
        raise ValueError(f"qkv row is {qkv.shape[1]}, heads say {(q_heads + 2 * kv_heads) * head_dim}")
    rotary_dim = head_dim if rotary_dim is None else rotary_dim
    if rotate and not (0 < rotary_dim <= head_dim and rotary_dim % 2 == 0):
        raise ValueError(f"rotary_dim must be even and at most the head size {head_dim}, is {rotary_dim}")
    for name, table in (("cos", cos), ("sin", sin)):
        _gpu(name, table, torch.float32, 2)
        if rotate and not (table.shape[1] == rotary_dim // 2):
            raise ValueError(f"{name} must be [max_position, {rotary_dim // 2}]")
    if not (cos.shape == sin.shape):
        raise ValueError("cos and sin tables differ in shape")
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= tokens):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {tokens} tokens")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    _gpu("block_table", block_table, torch.int32, 2)
    page_size = _check_pools(k_pool, v_pool, qkv.dtype, kv_heads, head_dim)
    _run("cie_rope_kv_write", load_library().cie_rope_kv_write(
        _stream(), _i(_code(qkv.dtype)), _ptr(qkv), _ptr(cos), _ptr(sin), _ptr(positions), _ptr(seq_of_token),
        _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]), _ptr(k_pool), _ptr(v_pool), _i(tokens),
        _i(q_heads), _i(kv_heads), _i(head_dim), _i(rotary_dim if rotate else 0), _i(page_size),
        _i(1 if rotate else 0), _i(1 if write_kv else 0)))


def silu_mul(gate_up: torch.Tensor, out: Optional[torch.Tensor] = None, row_sumsq: Optional[torch.Tensor] = None,
             hidden: int = 0, eps: float = 0.0) -> torch.Tensor:
    """``silu(gate_up[:, :I]) * gate_up[:, I:]`` for gate_up [T, 2I].  With ``row_sumsq``
    [T, parts] (partial sums of squares of rows of ``hidden`` values) both halves of
    row t are first multiplied by ``rsqrt(sum(row_sumsq[t]) / hidden + eps)``: the
    1/rms that the rows of the product behind ``gate_up`` lacked."""
    _gpu("gate_up", gate_up, dims=2)
    tokens, twice = gate_up.shape
    if not (twice % 2 == 0):
        raise ValueError(f"gate_up row must be even, is {twice}")
    inter = twice // 2
    if out is None:
        out = torch.empty((tokens, inter), dtype=gate_up.dtype, device=gate_up.device)
    _gpu("out", out, gate_up.dtype, 2)
    if not (out.shape == (tokens, inter)):
        raise ValueError(f"out must be {(tokens, inter)}, is {tuple(out.shape)}")
    parts = 0
    if row_sumsq is not None:
        _gpu("row_sumsq", row_sumsq, torch.float32, 2)
        if not (row_sumsq.shape[0] >= tokens and hidden > 0 and eps > 0):
            raise ValueError("row_sumsq needs a row per token, the rows' width and a positive eps")
        parts = row_sumsq.shape[1]
    _run("cie_silu_mul", load_library().cie_silu_mul(_stream(), _i(_code(gate_up.dtype)), _ptr(gate_up),
                                                     _ptr(out), _i(tokens), _i(inter), _ptr(row_sumsq), _i(parts),
                                                     _i(hidden), _f(eps)))
    return out


def paged_attention_generic(q: torch.Tensor, q_row_stride: int, k_pool: torch.Tensor, v_pool: torch.Tensor,
                            block_table: torch.Tensor, positions: torch.Tensor, seq_of_token: torch.Tensor,
                            seq_slot: torch.Tensor, tokens: int, q_heads: int, kv_heads: int, head_dim: int,
                            window: Optional[int], scale: float,
                            out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Attention of each token over its request's cached keys (its own included).

    ``q`` is any tensor whose row ``t`` holds the token's q heads in its first
    ``q_heads*head_dim`` elements, rows ``q_row_stride`` elements apart (the
    fused qkv buffer qualifies).  Returns [tokens, q_heads*head_dim]."""
    if not (q.is_cuda and q.dim() == 2 and q.stride(1) == 1 and q.stride(0) == q_row_stride):
        raise ValueError(f"q must be 2-d on the GPU with unit inner stride and row stride {q_row_stride}")
    if not (q.shape[0] >= tokens and q.shape[1] >= q_heads * head_dim):
        raise ValueError(f"q {tuple(q.shape)} too small")
    if not (q_heads % kv_heads == 0):
        raise ValueError(f"{q_heads} query heads are no multiple of {kv_heads} key heads")
    if not (head_dim % 8 == 0 and head_dim <= 256):
        raise ValueError(f"head_dim must be a multiple of 8 up to 256, is {head_dim}")
    if not (q_row_stride % 8 == 0):
        raise ValueError(f"q row stride must be a multiple of 8, is {q_row_stride}")
    _check_pools(k_pool, v_pool, q.dtype, kv_heads, head_dim)
    _gpu("block_table", block_table, torch.int32, 2)
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= tokens):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {tokens} tokens")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    if out is None:
        out = torch.empty((tokens, q_heads * head_dim), dtype=q.dtype, device=q.device)
    _gpu("out", out, q.dtype, 2)
    if not (out.shape == (tokens, q_heads * head_dim)):
        raise ValueError(f"out is {tuple(out.shape)}")
    _run("cie_paged_attention_generic", load_library().cie_paged_attention_generic(
        _stream(), _i(_code(q.dtype)), _ptr(q), _i(q_row_stride), _ptr(k_pool), _ptr(v_pool), _ptr(block_table),
        _i(block_table.shape[1]), _ptr(positions), _ptr(seq_of_token), _ptr(seq_slot), _ptr(out), _i(tokens),
        _i(q_heads), _i(kv_heads), _i(head_dim), _i(k_pool.shape[2]), _i(window or 0), _f(scale)))
    return out


F32_HEAD_DIMS = (32, 64, 96, 128)  # head sizes of the float32 attention on the matrix cores
F32_TILE_ROWS = 64   # (token, head) rows of its tiles
F32_BLOCK_KEYS = 64  # keys of its blocks
# the most bytes that the workspace of a float32 product or attention takes (an engine sets as much aside)
F32_WORKSPACE_BYTES = 256 << 20


def paged_attention_f32(q: torch.Tensor, q_row_stride: int, k_pool: torch.Tensor, v_pool: torch.Tensor,
                        block_table: torch.Tensor, tile_seq: Optional[torch.Tensor], tile_q0: Optional[torch.Tensor],
                        n_tiles: int, seq_slot: torch.Tensor, seq_start: torch.Tensor, seq_q_len: torch.Tensor,
                        q_start_loc: torch.Tensor, out: torch.Tensor, q_heads: int, kv_heads: int, head_dim: int,
                        window: Optional[int], scale: float, tokens_per_tile: int, turns: int = 0, blocks: int = 0,
                        part_o: Optional[torch.Tensor] = None, part_ml: Optional[torch.Tensor] = None,
                        capacity: int = 0, round: int = 0) -> None:
    """True float32 attention on the matrix cores: tile i holds
    up to ``tokens_per_tile`` tokens of sequence ``tile_seq[i]`` from its ``tile_q0[i]``-th token of this step on (both
    ``None``: tile i starts sequence i).  Rows of other tokens of ``out`` are left alone.  ``turns=0``: a workgroup to a
    tile and key head.  Otherwise that many waves to 16 rows of a tile, which take its blocks of 64 keys in turn and leave
    them in workspaces, of ``blocks`` blocks a tile (as many as any tile's keys need), that a second kernel joins.  Both
    give a row the same bits.  ``capacity``: the tiles' blocks lie one behind the other instead, each tile with as many as
    its keys need, in workspaces of ``capacity + blocks`` blocks; the call runs the tiles that begin in the ``round``-th
    ``capacity`` of them, or, with ``turns=0``, there and behind it."""
    if not (q.is_cuda and q.dtype == torch.float32 and q.dim() == 2 and q.stride(1) == 1 and q.stride(0) == q_row_stride):
        raise ValueError("q must be a float32 GPU matrix with unit inner stride")
    if not (q.shape[1] >= q_heads * head_dim and q_row_stride % 4 == 0):
        raise ValueError(f"q {tuple(q.shape)} does not fit")
    if head_dim not in F32_HEAD_DIMS or q_heads % kv_heads:
        raise ValueError(f"head_dim must be one of {F32_HEAD_DIMS}, is {head_dim}, and {kv_heads} key heads divide {q_heads}")
    group = q_heads // kv_heads
    if not (1 <= tokens_per_tile and tokens_per_tile * group <= F32_TILE_ROWS):
        raise ValueError(f"{tokens_per_tile} tokens of {group} heads do not fit {F32_TILE_ROWS} rows")
    page_size = _check_pools(k_pool, v_pool, torch.float32, kv_heads, head_dim)
    if not (page_size >= 4 and page_size & (page_size - 1) == 0):
        raise ValueError(f"page size must be a power of two >= 4, is {page_size}")
    _gpu("block_table", block_table, torch.int32, 2)
    if (tile_seq is None) != (tile_q0 is None):
        raise ValueError("tile_seq and tile_q0 come together, or neither (tile i is then the first tile of sequence i)")
    for name, meta in (("tile_seq", tile_seq), ("tile_q0", tile_q0)):
        if meta is not None:
            _gpu(name, meta, torch.int32, 1)
            if not (meta.shape[0] >= n_tiles):
                raise ValueError(f"{name} has {meta.shape[0]} entries for {n_tiles} tiles")
    if tile_seq is None and seq_q_len.shape[0] < n_tiles:
        raise ValueError(f"{n_tiles} tiles for {seq_q_len.shape[0]} sequences")
    for name, meta in (("seq_slot", seq_slot), ("seq_start", seq_start), ("seq_q_len", seq_q_len),
                       ("q_start_loc", q_start_loc)):
        _gpu(name, meta, torch.int32, 1)
    _gpu("out", out, torch.float32, 2)
    if not (out.shape[1] == q_heads * head_dim and out.shape[0] <= q.shape[0]):
        raise ValueError(f"out is {tuple(out.shape)}")
    rows = tokens_per_tile * group
    if turns:
        if part_o is None or part_ml is None or blocks < 1:
            raise ValueError("attention in blocks needs its workspaces")
        _gpu("part_o", part_o, torch.float32)
        _gpu("part_ml", part_ml, torch.float32)
        units = (capacity + blocks if capacity else n_tiles * blocks) * kv_heads * rows
        if not (part_o.numel() >= units * head_dim and part_ml.numel() >= units * 2):
            raise ValueError("attention workspaces are too small")
    _run("cie_paged_attention_f32", load_library().cie_paged_attention_f32(
        _stream(), _ptr(q), _i(q_row_stride), _ptr(k_pool), _ptr(v_pool), _ptr(block_table), _i(block_table.shape[1]),
        _ptr(tile_seq), _ptr(tile_q0), _i(n_tiles), _ptr(seq_slot), _ptr(seq_start), _ptr(seq_q_len),
        _ptr(q_start_loc), _ptr(out), _ptr(part_o), _ptr(part_ml), _i(rows), _i(blocks), _i(capacity), _i(round), _i(turns), _i(q_heads),
        _i(kv_heads), _i(head_dim), _i(page_size), _i(window or 0), _f(scale), _i(tokens_per_tile)))


MFMA_HEAD_DIMS = (32, 64, 96, 128, 256)
TILE_WAVES = 4  # waves per workgroup of the prompt form of the matrix-core attention
PROMPT_WAVES = 8  # ... and of its form with tiles of 128 rows whose keys and values go through LDS


def paged_attention_mfma(q: torch.Tensor, q_row_stride: int, k_pool: torch.Tensor, v_pool: torch.Tensor,
                         block_table: torch.Tensor, tile_seq: Optional[torch.Tensor], tile_q0: Optional[torch.Tensor],
                         n_tiles: int,
                         seq_slot: torch.Tensor, seq_start: torch.Tensor, seq_q_len: torch.Tensor,
                         q_start_loc: torch.Tensor, out: torch.Tensor, q_heads: int, kv_heads: int, head_dim: int,
                         window: Optional[int], scale: float, tokens_per_tile: int, row_tiles: int,
                         n_splits: int = 1, keys_per_split: int = 0,
                         max_context_dev: Optional[torch.Tensor] = None,
                         part_o: Optional[torch.Tensor] = None, part_ml: Optional[torch.Tensor] = None,
                         tile_waves: int = 1, merge: bool = True) -> None:
    """Matrix-core attention (bf16) for the tiles ``(tile_seq[i], tile_q0[i])``: tile i
    holds up to ``tokens_per_tile`` tokens of sequence ``tile_seq[i]`` from its
    ``tile_q0[i]``-th token of this step on (both ``None``: tile i starts sequence i, as in
    a step of single tokens; one dependent load less).  Rows of other tokens of ``out`` are left alone.
    With ``n_splits > 1`` every tile's keys are cut into parts of ``keys_per_split``
    (a multiple of 32; or, with ``max_context_dev``, derived on the device from the
    step's longest context) and merged through the workspaces.  ``tile_waves=4`` gives
    every tile (and every part of its keys) a workgroup of four waves that take the
    blocks of 32 keys in turn; it needs pages of at least 16 keys.  ``tile_waves=8`` (heads of up to
    128 dimensions) is the form whose waves share the tile's keys and values through LDS: with
    ``row_tiles=8`` tiles of 128 rows and eight waves, with ``row_tiles=4`` tiles of 64 rows and four
    waves, two such workgroups to a compute unit.  ``merge=False`` (several parts, not with ``tile_waves=8``) leaves the
    parts in the workspaces for :func:`merge_project` and ``out`` as it is."""
    if not (
        q.is_cuda and q.dtype == torch.bfloat16 and q.dim() == 2 and q.stride(1) == 1 and q.stride(0) == q_row_stride
    ):
        raise ValueError("q must be a bf16 GPU matrix with unit inner stride")
    if not (q.shape[1] >= q_heads * head_dim and q_row_stride % 8 == 0):
        raise ValueError(f"q {tuple(q.shape)} does not fit")
    if not (head_dim in MFMA_HEAD_DIMS):
        raise ValueError(f"head_dim must be one of {MFMA_HEAD_DIMS}, is {head_dim}")
    if not (q_heads % kv_heads == 0):
        raise ValueError(f"{q_heads} query heads are no multiple of {kv_heads} key heads")
    group = q_heads // kv_heads
    if not (row_tiles in (1, 2, 4, 8) and 1 <= tokens_per_tile and tokens_per_tile * group <= 16 * row_tiles):
        raise ValueError(f"{tokens_per_tile} tokens of {group} heads do not fit {row_tiles} row tiles")
    page_size = _check_pools(k_pool, v_pool, torch.bfloat16, kv_heads, head_dim)
    if not (page_size >= 4 and page_size & (page_size - 1) == 0):
        raise ValueError(f"page size must be a power of two >= 4, is {page_size}")
    _gpu("block_table", block_table, torch.int32, 2)
    if (tile_seq is None) != (tile_q0 is None):
        raise ValueError("tile_seq and tile_q0 come together, or neither (tile i is then the first tile of sequence i)")
    for name, meta in (("tile_seq", tile_seq), ("tile_q0", tile_q0)):
        if meta is None:
            continue
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= n_tiles):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {n_tiles} tiles")
    if tile_seq is None and seq_q_len.shape[0] < n_tiles:
        raise ValueError(f"{n_tiles} tiles for {seq_q_len.shape[0]} sequences")
    for name, meta in (("seq_slot", seq_slot), ("seq_start", seq_start), ("seq_q_len", seq_q_len),
                       ("q_start_loc", q_start_loc)):
        _gpu(name, meta, torch.int32, 1)
    _gpu("out", out, torch.bfloat16, 2)
    if not (out.shape[1] == q_heads * head_dim and out.shape[0] <= q.shape[0]):
        raise ValueError(f"out is {tuple(out.shape)}")
    if not (1 <= n_splits <= 65535):
        raise ValueError(f"n_splits {n_splits} out of range")
    if not (
        (tile_waves == 1 and row_tiles <= 4)
        or (tile_waves == TILE_WAVES and scale > 0 and page_size >= 16 and row_tiles <= 4
            and (row_tiles == 1 or head_dim <= 128))
        or (tile_waves == PROMPT_WAVES and scale > 0 and page_size >= 16 and row_tiles in (4, 8) and head_dim <= 128)
    ):
        raise ValueError(f"tile_waves {tile_waves} with {n_splits} splits, {row_tiles} row tiles, head size {head_dim}, "
                         f"pages of {page_size}")
    if n_splits > 1:
        rows = 16 * row_tiles
        if not (part_o is not None and part_ml is not None):
            raise ValueError("split attention needs its workspaces")
        _gpu("part_o", part_o, torch.float32)
        _gpu("part_ml", part_ml, torch.float32)
        units = n_tiles * kv_heads * n_splits
        if not (part_o.numel() >= units * rows * head_dim and part_ml.numel() >= units * rows * 2):
            raise ValueError("attention workspaces are too small")
        if max_context_dev is not None:
            _gpu("max_context_dev", max_context_dev, torch.int32)
        else:
            if not (keys_per_split > 0 and keys_per_split % 32 == 0):
                raise ValueError(f"keys_per_split {keys_per_split} must be a multiple of 32")
    if not merge and (n_splits == 1 or tile_waves == PROMPT_WAVES):
        raise ValueError("only parts of the keys, and not those of the form through LDS, can be left unmerged")
    _run("cie_paged_attention_mfma", load_library().cie_paged_attention_mfma(
        _stream(), _ptr(q), _i(q_row_stride), _ptr(k_pool), _ptr(v_pool), _ptr(block_table),
        _i(block_table.shape[1]), _ptr(tile_seq), _ptr(tile_q0), _ptr(seq_slot), _ptr(seq_start), _ptr(seq_q_len),
        _ptr(q_start_loc), _ptr(out), _ptr(part_o), _ptr(part_ml), _i(n_tiles), _i(q_heads), _i(kv_heads),
        _i(head_dim), _i(page_size), _i(window or 0), _f(scale), _i(n_splits), _i(tokens_per_tile), _i(row_tiles),
        _i(keys_per_split), _ptr(max_context_dev), _i(tile_waves), _i(merge)))


MERGE_PROJECT_ROWS = 16   # one row tile
MERGE_PROJECT_SLICE = 128  # k of a workgroup


def merge_project(part_o: torch.Tensor, part_ml: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
                  residual: torch.Tensor, q_heads: int, kv_heads: int, head_dim: int, n_splits: int, tile_rows: int,
                  tiles: Optional[int] = None) -> None:
    """``residual += merged @ weight.T + bias`` (float32, in place, atomic adds), where row m of ``merged`` is the attention of
    tile m, whose one token's ``n_splits`` parts :func:`paged_attention_mfma` left in the workspaces (``merge=False``;
    ``tile_rows``: rows of its tiles).  ``weight`` is [N, q_heads * head_dim] in bf16."""
    _gpu("weight", weight, torch.bfloat16, 2)
    n, k = weight.shape
    _gpu("residual", residual, torch.float32, 2)
    m = residual.shape[0]
    if not (1 <= m <= MERGE_PROJECT_ROWS and residual.shape[1] == n):
        raise ValueError(f"residual {tuple(residual.shape)} for a weight of {n} rows; at most {MERGE_PROJECT_ROWS} rows")
    if not (kv_heads >= 1 and q_heads % kv_heads == 0 and tile_rows >= q_heads // kv_heads and head_dim % 4 == 0
            and k == q_heads * head_dim and k % MERGE_PROJECT_SLICE == 0 and weight.data_ptr() % 16 == 0):
        raise ValueError(f"{q_heads} heads of {head_dim} on {kv_heads} and a weight {tuple(weight.shape)} do not fit")
    _gpu("part_o", part_o, torch.float32)
    _gpu("part_ml", part_ml, torch.float32)
    units = m * kv_heads * n_splits * tile_rows
    if not (n_splits >= 1 and part_o.numel() >= units * head_dim and part_ml.numel() >= units * 2
            and part_o.data_ptr() % 16 == 0 and part_ml.data_ptr() % 8 == 0):
        raise ValueError("attention workspaces are too small, or off a 16-byte line")
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if bias.shape[0] != n:
            raise ValueError(f"bias must be [{n}]")
    if tiles is None:  # (128 columns a workgroup while every one has a unit of its own; else 512, fewer that merge the same shares)
        tiles = 4 if -(-n // MERGE_PROJECT_SLICE) * (k // MERGE_PROJECT_SLICE) > compute_units() else 1
    _run("cie_merge_project", load_library().cie_merge_project(
        _stream(), _ptr(part_o), _ptr(part_ml), _ptr(weight), _ptr(bias), _ptr(residual), _i(m), _i(n), _i(q_heads),
        _i(kv_heads), _i(head_dim), _i(n_splits), _i(tile_rows), _i(tiles)))


F32_STRETCH = 1024  # k that one workgroup takes where the float32 product cuts K


def f32_bands(rows: int, columns: int, k: int) -> tuple[int, int]:
    """(bands, rows of a band) in which the float32 product with K in stretches takes its rows: as few bands, in multiples
    of the tiles' 64 rows, as keep the stretches' sums of one within ``F32_WORKSPACE_BYTES`` (7B down of 1,500 rows: two
    bands of 768 instead of 409 MB)."""
    most = max(64, F32_WORKSPACE_BYTES // (-(-k // F32_STRETCH) * columns * 4) // 64 * 64)
    bands = -(-rows // most)
    return bands, -(-(-(-rows // bands)) // 64) * 64


def plan_gemm_f32(rows: int, columns: int, k: int) -> int:
    """Which form of the float32 product runs (the numbers of ``cie_gemm_f32``): 0 few rows, 1 tiles of 64 x 64, 2 such
    tiles with K cut in stretches.  Up to 16 rows the first, bound by the weight's stream; beyond that the one whose
    turns over the units take least, in us as measured on MI355X: a turn of workgroups of 32 rows and 16 columns takes
    9.5 per 2,048 k (eight waves; 3.9 where K is up to 1,024 and four waves do), a tile 21.5 per 1,000 k when alone on its
    unit and 17.5 behind another, a stretch 19 and the join behind it 10, a band.  (N = K = 2,048: 64 / 128 rows 13 / 23 in
    the first, 47 / 48 in the second, 28 / 29 in the third form; N 22,016: 101 / 177, 81 / 115, 69 / 125; N 2,048, K
    11,008: 53 / 106, 236 / 237, 52 / 75.)"""
    if rows <= 16:
        return 0
    units = compute_units()
    turns = -(-(-(-rows // 32) * -(-columns // 16)) // units)
    few = 3 + turns * (3.9 if k <= 1024 else 9.5 * -(-k // 2048))
    tiles = -(-rows // 64) * -(-columns // 64)
    whole = 2 + k / 1000 * (21.5 + 17.5 * (-(-tiles // units) - 1))
    stretches = -(-k // F32_STRETCH)
    cut = whole
    if stretches > 1 and 64 * stretches * columns * 4 <= F32_WORKSPACE_BYTES:
        bands, band = f32_bands(rows, columns, k)
        cut = bands * (10 + 19 * -(-(band // 64 * -(-columns // 64) * stretches) // units))
    return 0 if few <= min(whole, cut) else 1 if whole <= cut else 2


def gemm_f32(a: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
             out: Optional[torch.Tensor] = None, gate: bool = False, form: Optional[int] = None) -> torch.Tensor:
    """True float32 ``a @ weight.T + bias``; a [M, K] (rows may be strided), weight [N, K].  ``gate``: the gated unit of
    the product's halves instead, ``silu(first N / 2 columns) * (the others)`` (no bias).  ``form``: one of the kernel's
    forms instead of the planned one (every form gives a row the same bits)."""
    if not (a.is_cuda and a.dtype == torch.float32 and a.dim() == 2 and a.stride(1) == 1):
        raise ValueError("a must be a float32 GPU matrix with unit inner stride")
    _gpu("weight", weight, torch.float32, 2)
    m, k = a.shape
    n = weight.shape[0]
    if not (weight.shape[1] == k):
        raise ValueError(f"a is [{m},{k}] but weight is {tuple(weight.shape)}")
    if gate and (bias is not None or n % 2):
        raise ValueError("a gated unit takes an even number of weight rows and no bias")
    if bias is not None:
        _gpu("bias", bias, torch.float32, 1)
        if not (bias.shape[0] == n):
            raise ValueError(f"bias must be [{n}]")
    width = n // 2 if gate else n
    if out is None:
        out = torch.empty((m, width), dtype=torch.float32, device=a.device)
    _gpu("out", out, torch.float32, 2)
    if not (out.shape == (m, width)):
        raise ValueError(f"out must be {(m, width)}")
    lda = a.stride(0) if m > 1 else max(a.stride(0), k)
    if form is None:
        form = plan_gemm_f32(m, n, k)
    band, parts = m, None
    if form == 2 and m:
        _, band = f32_bands(m, n, k)
        parts = torch.empty((-(-k // F32_STRETCH), min(m, band), n), dtype=torch.float32, device=a.device)
    for first in range(0, max(m, 1), max(band, 1)):
        _run("cie_gemm_f32", load_library().cie_gemm_f32(
            _stream(), _ptr(a) + 4 * first * lda, _ptr(weight), _ptr(bias), _ptr(out) + 4 * first * width, _ptr(parts),
            _i(min(band, m - first)), _i(n), _i(k), _i(lda), _i(width), _i(bool(gate)), _i(form), _i(compute_units(a.device))))
    return out


# Rows up to which a float32 product takes the norm in front, the rotation or the add into the stream along (every workgroup makes
# the norm of as many rows).  Decode steps of 12 layers, kernels of their own and joined, us: 3B 4 sequences, eight steps 12,061,
# 11,211; 0.5B 8 sequences, four steps 3,586, 3,442; 16 sequences, with kernels for as many rows, 3,757, 3,770.
F32_FEW_ROWS = 8
F32_NORM_WIDTH = 8192  # ... the widest rows whose norm it makes,
F32_NORM_SEGMENT, F32_NORM_SEGMENTS = 512, 32  # and how many segments of a row in all, which lie in LDS


def folds_norm_f32(stream: torch.Tensor) -> bool:
    """Whether :func:`gemm_f32_normed` and :func:`gemm_f32_qkv_rope` take this float32 stream."""
    rows, width = stream.shape
    return (1 <= rows <= F32_FEW_ROWS and 8 <= width <= F32_NORM_WIDTH and width % 8 == 0
            and rows * -(-width // F32_NORM_SEGMENT) <= F32_NORM_SEGMENTS and stream.is_cuda
            and stream.dtype == torch.float32 and stream.is_contiguous() and stream.data_ptr() % 16 == 0)


def _check_normed_f32(stream: torch.Tensor, norm_weight: torch.Tensor, eps: float, weight: torch.Tensor,
                      bias: Optional[torch.Tensor]) -> tuple[int, int, int]:
    if not (stream.dim() == 2 and folds_norm_f32(stream)):
        raise ValueError(f"the product makes the norm of 1 to {F32_FEW_ROWS} contiguous float32 rows of up to {F32_NORM_WIDTH} "
                         f"numbers (a multiple of 8; {F32_NORM_SEGMENTS} segments of {F32_NORM_SEGMENT} in all) on a 16-byte "
                         f"line itself, not of {tuple(stream.shape)}")
    _gpu("weight", weight, torch.float32, 2)
    _gpu("norm_weight", norm_weight, torch.float32, 1)
    m, k = stream.shape
    n = weight.shape[0]
    if not (weight.shape[1] == k and norm_weight.shape[0] == k and eps > 0):
        raise ValueError(f"weight {tuple(weight.shape)} and norm weight {tuple(norm_weight.shape)} do not fit rows of K={k}")
    if weight.data_ptr() % 16 or norm_weight.data_ptr() % 16:
        raise ValueError("operands must be 16-byte aligned")
    if bias is not None:
        _gpu("bias", bias, torch.float32, 1)
        if not (bias.shape[0] == n):
            raise ValueError(f"bias must be [{n}]")
    return m, n, k


def gemm_f32_normed(stream: torch.Tensor, norm_weight: torch.Tensor, eps: float, weight: torch.Tensor) -> torch.Tensor:
    """The gated unit of :func:`gemm_f32` of the RMS norm of ``stream``'s few rows, made inside the product: the bits are those of
    :func:`add_rmsnorm` followed by the product."""
    m, n, k = _check_normed_f32(stream, norm_weight, eps, weight, None)
    if n % 2:
        raise ValueError("a gated unit takes an even number of weight rows")
    out = torch.empty((m, n // 2), dtype=torch.float32, device=stream.device)
    _run("cie_gemm_f32_normed", load_library().cie_gemm_f32_normed(
        _stream(), _ptr(stream), _ptr(norm_weight), _f(eps), _ptr(weight), _ptr(out), _i(m), _i(n), _i(k), _i(n // 2),
        _i(compute_units(stream.device))))
    return out


def gemm_f32_into(a: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], into: torch.Tensor) -> None:
    """``into += a @ weight.T + bias`` for up to ``F32_FEW_ROWS`` rows, in the bits of :func:`gemm_f32` and an add behind it."""
    if not (a.is_cuda and a.dtype == torch.float32 and a.dim() == 2 and a.stride(1) == 1):
        raise ValueError("a must be a float32 GPU matrix with unit inner stride")
    _gpu("weight", weight, torch.float32, 2)
    _gpu("into", into, torch.float32, 2)
    m, k = a.shape
    n = weight.shape[0]
    if not (weight.shape[1] == k and into.shape == (m, n) and m <= F32_FEW_ROWS):
        raise ValueError(f"a is [{m},{k}], weight {tuple(weight.shape)}, into {tuple(into.shape)}; up to {F32_FEW_ROWS} rows")
    if bias is not None:
        _gpu("bias", bias, torch.float32, 1)
        if not (bias.shape[0] == n):
            raise ValueError(f"bias must be [{n}]")
    lda = a.stride(0) if m > 1 else max(a.stride(0), k)
    _run("cie_gemm_f32_into", load_library().cie_gemm_f32_into(
        _stream(), _ptr(a), _ptr(weight), _ptr(bias), _ptr(into), _i(m), _i(n), _i(k), _i(lda), _i(n), _i(compute_units(a.device))))


def gemm_f32_at(a: torch.Tensor, weight: torch.Tensor, out_at: torch.Tensor) -> None:
    """``a @ weight.T`` of up to ``F32_FEW_ROWS`` rows into the contiguous float32 [M, N] whose address ``out_at`` (int64 [1], on
    the GPU) holds when the kernel runs (the caller vouches for it), with the bits of :func:`gemm_f32`."""
    _result_at(out_at)
    _gpu("weight", weight, torch.float32, 2)
    (m, k), n = a.shape, weight.shape[0]
    if not (a.is_cuda and a.dtype == torch.float32 and a.stride(1) == 1 and weight.shape[1] == k and 1 <= m <= F32_FEW_ROWS):
        raise ValueError(f"a {tuple(a.shape)} vs weight {tuple(weight.shape)}, up to {F32_FEW_ROWS} float32 rows with unit inner stride")
    _run("cie_gemm_f32_at", load_library().cie_gemm_f32_at(
        _stream(), _ptr(a), _ptr(weight), _ptr(out_at), _i(m), _i(n), _i(k), _i(a.stride(0) if m > 1 else max(a.stride(0), k)),
        _i(compute_units(a.device))))


def gemm_f32_qkv_rope(stream: torch.Tensor, norm_weight: torch.Tensor, eps: float, weight: torch.Tensor,
                      bias: Optional[torch.Tensor], cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                      seq_of_token: torch.Tensor, seq_slot: torch.Tensor, block_table: torch.Tensor, k_pool: torch.Tensor,
                      v_pool: torch.Tensor, q_heads: int, kv_heads: int, head_dim: int, rotate: bool = True,
                      write_kv: bool = True, rotary_dim: Optional[int] = None) -> torch.Tensor:
    """The q/k/v product of :func:`gemm_f32_normed` with the rotation and the cache write of :func:`rope_kv_write` in its
    epilogue, in their bits (heads of a size in steps of 16, of which the first ``rotary_dim`` dimensions, a number in steps
    of 16 too, rotate; all without it).  Returns [M, N] whose query columns hold the
    rotated queries; the others are not written."""
    m, n, k = _check_normed_f32(stream, norm_weight, eps, weight, bias)
    if head_dim % 16 or n != (q_heads + 2 * kv_heads) * head_dim:
        raise ValueError(f"weight has {n} rows, heads say {(q_heads + 2 * kv_heads) * head_dim}, of {head_dim} (in steps of 16)")
    rotary_dim = head_dim if rotary_dim is None else rotary_dim
    if not (0 < rotary_dim <= head_dim and rotary_dim % 16 == 0):
        raise ValueError(f"rotary_dim must be in steps of 16 up to {head_dim}, is {rotary_dim}")
    for name, table in (("cos", cos), ("sin", sin)):
        _gpu(name, table, torch.float32, 2)
        if rotate and not (table.shape[1] == rotary_dim // 2):
            raise ValueError(f"{name} must be [max_position, {rotary_dim // 2}]")
    if not (cos.shape == sin.shape):
        raise ValueError("cos and sin tables differ in shape")
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= m):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {m} rows")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    _gpu("block_table", block_table, torch.int32, 2)
    page_size = _check_pools(k_pool, v_pool, torch.float32, kv_heads, head_dim)
    out = torch.empty((m, n), dtype=torch.float32, device=weight.device)
    _run("cie_gemm_f32_normed_rope", load_library().cie_gemm_f32_normed_rope(
        _stream(), _ptr(stream), _ptr(norm_weight), _f(eps), _ptr(weight), _ptr(bias), _ptr(out), _i(m), _i(n), _i(k), _ptr(cos),
        _ptr(sin), _ptr(positions), _ptr(seq_of_token), _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]), _ptr(k_pool),
        _ptr(v_pool), _i(q_heads), _i(kv_heads), _i(head_dim), _i(rotary_dim), _i(page_size), _i(bool(rotate)), _i(bool(write_kv)),
        _i(compute_units(weight.device))))
    return out


EPI_BF16, EPI_F32, EPI_SILU, EPI_RESID, EPI_PARTIAL = 0, 1, 2, 3, 4
EPI_ATOMIC = 7  # (the shared-rows form: parts of K add into a float32 stream with atomic adds)
FUSED_TARGET_WAVES = 2048
FUSED_MAX_ROWS = 64  # rows one workgroup of ``gemm_fused`` takes; more rows run as more workgroup rows
FUSED_PAIR_WORKGROUPS = 256  # workgroups that must remain when workgroups of many rows take two column tiles


FUSED_SHORT_K = 1024  # of which four waves have all in flight at once (two slices of 128 each; one with four row tiles)
FUSED_LONG_K = 4096   # from which more than 16 rows may run as blocks of 16


BLOCK_START = 4  # of a workgroup, in the time that 16 rows or columns of a slice take it
BLOCK_WAITS = 1.25  # ... a slice of four row tiles behind another, which have one in flight


def _row_blocks(rows: int, row_tiles: int, column_tiles: int, groups: int, units: int, k: int, whole: bool = True) -> float:
    """What a product of more than 16 rows takes, in the time that 16 rows or columns take a workgroup: it reads its columns of
    the weight and its rows of A, and more workgroups than units take turns.  Of a short K the start counts too (q/k/v, 50 rows
    x 10,240, K 136 6.7 us in blocks of 64 rows, 10.2 of 32; 121 x 5,120, K 88 6.5, 9.8), four row tiles wait for the second of a wave's slices
    (83 x 5,120, K 520 9.4, 7.8), and the q/k/v product, which hides a start behind the workgroup beside it, does not take ``whole`` turns
    only."""
    turns = groups * -(-rows // (16 * row_tiles)) / units
    turns = math.ceil(turns) if whole or k > FUSED_SHORT_K else max(1.0, turns)
    if k > FUSED_SHORT_K:
        return turns * (column_tiles + row_tiles)
    slices = -(-k // 512)  # of a wave
    return turns * (BLOCK_START + slices * (column_tiles + row_tiles) * (BLOCK_WAITS if row_tiles == 4 and slices > 1 else 1.0))


@functools.lru_cache(maxsize=4096)
def _plan_row_blocks(rows: int, tiles: int, k: int, units: int) -> tuple[int, int]:
    """(row tiles, waves) of a workgroup with one column tile.  Four waves where they have all of K in flight, or where there are
    workgroups for two on a unit (96 rows x 2,816, K 2,048 12.0 us, a tenth more with eight)."""
    row_tiles = min((4, 2, 1) if k >= FUSED_LONG_K else (4, 2), key=lambda r: _row_blocks(rows, r, 1, tiles, units, k))
    fills = tiles * -(-rows // (16 * row_tiles)) * 4 >= FUSED_TARGET_WAVES
    short = k < FUSED_SHORT_K if row_tiles == 4 else k <= FUSED_SHORT_K
    return row_tiles, 4 if fills or short else 8


def plan_fused(rows: int, column_tiles: int, k: int) -> tuple[int, int, int]:
    """(row tiles, waves per workgroup, column tiles per workgroup) of ``gemm_fused``
    for ``rows`` rows, ``column_tiles`` tiles of 16 columns and a K of ``k``.  16, 32 or 64 rows per workgroup (more rows: more workgroups,
    each streaming the weight again).  With more than 16 rows a workgroup takes
    two column tiles if that still leaves enough workgroups (each activation
    value a wave loads then meets two weight tiles), else as many rows as have the units read least (``_row_blocks``).  MI355X, us, up to 64 rows a workgroup and as many as are taken:
    2,048 x 2,048 64 rows 9.7, 7.7 (128 and 256 workgroups), 128 rows 9.7 either way; 896 x 896 64 rows 6.7, 4.8, 128 6.8, 4.9;
    1,024 x 4,096 64 rows 14.5, 9.4; 2,304 x 2,304 64 rows 10.2 either way, 96 14.0, 11.1; 4,096 x 1,024 32 rows with eight and four
    waves 7.3, 6.3.  Up to 16 rows as many waves share K as it
    takes to fill the GPU, each with at least one 128-wide slice."""
    pair = column_tiles >= 2 * FUSED_PAIR_WORKGROUPS
    if rows > 16 and not pair:
        return *_plan_row_blocks(rows, column_tiles, k, compute_units()), 1
    row_tiles = 1 if rows <= 16 else 2 if rows <= 32 else 4
    pair = pair and row_tiles > 1
    groups = (-(-column_tiles // 2) if pair else column_tiles) * -(-rows // FUSED_MAX_ROWS)
    waves = 1 if row_tiles == 1 else 4
    while waves < 8 and groups * waves < FUSED_TARGET_WAVES and waves * 2 * 128 <= k:
        waves *= 2
    return row_tiles, waves, 2 if pair else 1


def gemm_fused(weight: torch.Tensor, epilogue: int, a: torch.Tensor, bias: Optional[torch.Tensor] = None,
               residual_out: Optional[torch.Tensor] = None, sumsq_out: Optional[torch.Tensor] = None,
               plan: Optional[tuple[int, int, int]] = None,
               norm_weight: Optional[torch.Tensor] = None, scaled_out: Optional[torch.Tensor] = None,
               row_sumsq: Optional[torch.Tensor] = None, eps: float = 0.0,
               act_out: Optional[torch.Tensor] = None, out_at: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """Few-row matrix product ``a @ weight.T`` (bf16 operands, float32 sums) fused
    with its neighbour.  ``epilogue``: ``EPI_BF16`` / ``EPI_F32`` return
    ``a W^T + bias``; ``EPI_SILU`` (weight = gate rows over up rows) returns
    ``silu(gate) * up`` [M, N/2]; ``EPI_RESID`` adds the product
    into ``residual_out`` (float32 [M, N]) and returns the partial sums of
    squares of its new rows [M, ceil(N/16)].  (Partial products of a cut K: :func:`gemm_shared_rows`.)
    An RMSNorm between an ``EPI_RESID`` product and an ``EPI_SILU`` product of up to 16
    rows can ride along: with ``norm_weight`` (float32 [N]) and ``scaled_out`` (bf16
    [M, N]) the former also writes the new residual times the weight, and the latter,
    given these rows as ``a`` with ``row_sumsq`` (the former's result) and ``eps``,
    multiplies its sums by each row's ``rsqrt(mean square + eps)`` before the SiLU.
    ``act_out`` (bf16 [M, n], rows may lie apart; ``EPI_BF16``): the last n columns go there, squared behind relu, and the
    result that comes back holds the columns in front of them.  ``out_at`` (int64 [1] on the GPU; ``EPI_F32``): the result goes
    to the contiguous float32 [M, N] whose address it holds when the kernel runs (the caller vouches for it), and none comes back."""
    _gpu("weight", weight, torch.bfloat16, 2)
    n, k = weight.shape
    if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.stride(1) == 1):
        raise ValueError("a must be a bf16 GPU matrix with unit inner stride")
    m = a.shape[0]
    if not (m >= 1 and a.shape[1] == k):
        raise ValueError(f"a {tuple(a.shape)} vs K={k}")
    lda = a.stride(0) if m > 1 else max(a.stride(0), k)
    if not (k % 8 == 0 and lda % 8 == 0):
        raise ValueError(f"K and the row stride must be multiples of 8, are {k} and {lda}")
    if not (a.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0):
        raise ValueError("operands must be 16-byte aligned")
    device = weight.device
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if not (bias.shape[0] == n and epilogue != EPI_SILU):
            raise ValueError("bias does not fit")
    columns = n // 2 if epilogue == EPI_SILU else n
    row_tiles, waves, column_tiles = plan or plan_fused(m, -(-columns // 16), k)
    if epilogue == EPI_SILU:
        column_tiles = 1 if row_tiles == 1 else 2  # always a gate tile with its up tile
    if not (
        row_tiles in (1, 2, 4) and waves in ((1, 2, 4, 8) if row_tiles == 1 else (4, 8))
        and column_tiles in ((1,) if row_tiles == 1 else (1, 2))
    ):
        raise ValueError(f"plan {(row_tiles, waves, column_tiles)} is not one the kernel has")
    residual = sumsq = None
    split, act_ld = n, 0
    if act_out is not None:
        split = n - act_out.shape[1]
        if epilogue != EPI_BF16 or not 0 < split < n:
            raise ValueError("columns that pass through an activation are the last ones of a bf16 result, and not all of it")
        _row_view("act_out", act_out, (m, n - split), (torch.bfloat16,))
        act_ld = _ld(act_out)
    if epilogue == EPI_BF16:
        out = torch.empty((m, split), dtype=torch.bfloat16, device=device)
    elif epilogue == EPI_F32:
        out = torch.empty((m, n), dtype=torch.float32, device=device) if out_at is None else None
    elif epilogue == EPI_SILU:
        if not (n % 2 == 0):
            raise ValueError(f"the SiLU epilogue needs an even N, got {n}")
        out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=device)
    elif epilogue == EPI_RESID:
        if not (residual_out is not None):
            raise ValueError("the residual epilogue needs the residual to add into")
        _gpu("residual_out", residual_out, torch.float32, 2)
        if not (residual_out.shape == (m, n)):
            raise ValueError(f"residual_out {tuple(residual_out.shape)} vs {(m, n)}")
        parts = -(-n // 16)
        if sumsq_out is None:
            sumsq_out = torch.empty((m, parts), dtype=torch.float32, device=device)
        _gpu("sumsq_out", sumsq_out, torch.float32, 2)
        if not (sumsq_out.shape[0] >= m and sumsq_out.shape[1] == parts):
            raise ValueError(f"sumsq_out {tuple(sumsq_out.shape)} must be [>= {m}, {parts}]")
        out, residual, sumsq = sumsq_out, residual_out, sumsq_out
    else:
        raise ValueError(f"unknown epilogue {epilogue}")
    if (norm_weight is None) != (scaled_out is None) or (scaled_out is not None and epilogue != EPI_RESID):
        raise ValueError("a scaled copy needs the norm's weight, its own rows and the residual epilogue")
    if scaled_out is not None:
        _gpu("norm_weight", norm_weight, torch.float32, 1)
        _gpu("scaled_out", scaled_out, torch.bfloat16, 2)
        if not (norm_weight.shape[0] == n and scaled_out.shape == (m, n)):
            raise ValueError(f"norm_weight {tuple(norm_weight.shape)} / scaled_out {tuple(scaled_out.shape)} vs {(m, n)}")
    if out_at is not None:
        _result_at(out_at)
        if epilogue != EPI_F32:
            raise ValueError("only a float32 result goes to an address on the device")
    parts_in = 0
    if row_sumsq is not None:
        _gpu("row_sumsq", row_sumsq, torch.float32, 2)
        if not (epilogue == EPI_SILU and row_tiles == 1 and m <= 16 and row_sumsq.shape[0] >= m and eps > 0):
            raise ValueError("rows that lack their scale go to the SiLU epilogue of up to 16 rows, with a positive eps")
        parts_in = row_sumsq.shape[1]
    _run("cie_gemm_fused", load_library().cie_gemm_fused(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(bias), _ptr(None if epilogue == EPI_RESID else out),
        _ptr(residual), _ptr(sumsq), _i(m), _i(n), _i(k), _i(epilogue), _i(row_tiles), _i(waves), _i(column_tiles),
        _ptr(norm_weight), _ptr(scaled_out), _ptr(row_sumsq), _i(parts_in), _f(eps), _i(split), _ptr(act_out), act_ld, _ptr(out_at)))
    return out


SHARED_ROWS_MAX = 128  # rows of the form whose waves share the rows of A


def gemm_shared_rows(weight: torch.Tensor, epilogue: int, a: torch.Tensor, bias: Optional[torch.Tensor] = None,
                     column_tiles: int = 2, waves: int = 4, k_parts: int = 1,
                     row_sumsq: Optional[torch.Tensor] = None, eps: float = 0.0,
                     add_into: Optional[torch.Tensor] = None, out_at: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``a @ weight.T`` for 17 to 128 rows (it takes fewer too) in the form whose four waves per
    workgroup own columns and share each slice of ``a`` through LDS: ``EPI_BF16`` or ``EPI_F32`` (+ bias),
    ``EPI_SILU`` (weight = gate rows over up rows; with ``row_sumsq`` and ``eps`` the rows of ``a``
    lack their ``rsqrt(mean square + eps)``, as in :func:`gemm_fused`) or ``EPI_PARTIAL``
    (``k_parts`` float32 partial products [k_parts, M, N], bias in part 0) or ``EPI_ATOMIC``
    (each of the ``k_parts`` parts of K adds its products into ``add_into``, float32 [M, N], with the
    hardware's atomic float add: no partial products to sum afterwards, and no fixed order of the sums;
    ``add_into`` comes back).  ``column_tiles`` tiles of 16 columns per wave, ``waves`` waves per workgroup.
    ``out_at`` (``EPI_F32``): as in :func:`gemm_fused`."""
    _gpu("weight", weight, torch.bfloat16, 2)
    n, k = weight.shape
    if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.stride(1) == 1):
        raise ValueError("a must be a bf16 GPU matrix with unit inner stride")
    m = a.shape[0]
    if not (1 <= m <= SHARED_ROWS_MAX and a.shape[1] == k):
        raise ValueError(f"a {tuple(a.shape)} vs K={k} and at most {SHARED_ROWS_MAX} rows")
    lda = a.stride(0) if m > 1 else max(a.stride(0), k)
    if not (k % 8 == 0 and lda % 8 == 0 and a.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0):
        raise ValueError(f"K and the row stride must be multiples of 8 (are {k}, {lda}) and the operands 16-byte aligned")
    if epilogue not in (EPI_BF16, EPI_F32, EPI_SILU, EPI_PARTIAL, EPI_ATOMIC):
        raise ValueError(f"epilogue {epilogue} is not one this form has")
    if epilogue == EPI_F32:
        column_tiles = 2
    if not (1 <= k_parts <= 64 and (k_parts == 1 or epilogue in (EPI_PARTIAL, EPI_ATOMIC))):
        raise ValueError(f"k_parts {k_parts} does not fit the epilogue")
    if (epilogue == EPI_ATOMIC) != (add_into is not None):
        raise ValueError("the atomic epilogue, and only it, adds into a stream that the caller gives")
    if add_into is not None:
        _gpu("add_into", add_into, torch.float32, 2)
        if not (tuple(add_into.shape) == (m, n) and add_into.is_contiguous()):
            raise ValueError(f"add_into is {tuple(add_into.shape)}, the product [{m}, {n}]")
    if epilogue == EPI_SILU:
        column_tiles = 2
        if n % 2 or bias is not None:
            raise ValueError("the SiLU epilogue needs an even N and no bias")
    if column_tiles not in (1, 2) or waves not in (2, 3, 4):
        raise ValueError(f"column_tiles {column_tiles} not in (1, 2), or waves {waves} not in (2, 3, 4)")
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if bias.shape[0] != n:
            raise ValueError(f"bias must be [{n}]")
    parts_in = 0
    if row_sumsq is not None:
        _gpu("row_sumsq", row_sumsq, torch.float32, 2)
        if not (epilogue == EPI_SILU and row_sumsq.shape[0] >= m and eps > 0):
            raise ValueError("rows that lack their scale go to the SiLU epilogue, with a positive eps")
        parts_in = row_sumsq.shape[1]
    device = weight.device
    if out_at is not None:
        _result_at(out_at)
        if epilogue != EPI_F32:
            raise ValueError("only a float32 result goes to an address on the device")
        out = None
    elif epilogue == EPI_BF16:
        out = torch.empty((m, n), dtype=torch.bfloat16, device=device)
    elif epilogue == EPI_F32:
        out = torch.empty((m, n), dtype=torch.float32, device=device)
    elif epilogue == EPI_SILU:
        out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=device)
    elif epilogue == EPI_ATOMIC:
        out = add_into
    else:
        out = torch.empty((k_parts, m, n), dtype=torch.float32, device=device)
    _run("cie_gemm_shared_rows", load_library().cie_gemm_shared_rows(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(bias), _ptr(out), _i(m), _i(n), _i(k), _i(epilogue),
        _i(column_tiles), _i(waves), _i(k_parts), _ptr(row_sumsq), _i(parts_in), _f(eps), _ptr(out_at)))
    return out


BESIDE_ROWS = 16  # of two products in one launch


def _beside_rows(name: str, a: torch.Tensor, weight: torch.Tensor) -> int:
    """The row stride of one of two products' rows, checked."""
    _gpu(f"weight of {name}", weight, torch.bfloat16, 2)
    if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.stride(1) == 1 and a.shape[1] == weight.shape[1]
            and 1 <= a.shape[0] <= BESIDE_ROWS):
        raise ValueError(f"{name} {tuple(a.shape)} must be up to {BESIDE_ROWS} bf16 rows with unit inner stride as long as the weight's")
    lda = a.stride(0) if a.shape[0] > 1 else max(a.stride(0), a.shape[1])
    if a.shape[1] % 8 or lda % 8 or a.data_ptr() % 16 or weight.data_ptr() % 16:
        raise ValueError(f"{name}: K and the row stride must be multiples of 8 and the operands 16-byte aligned")
    return lda


def gemm_silu_beside(weight: torch.Tensor, a: torch.Tensor, weight2: torch.Tensor, a2: torch.Tensor, bias2: Optional[torch.Tensor],
                     waves: int = 4) -> tuple[torch.Tensor, torch.Tensor]:
    """Two products of up to ``BESIDE_ROWS`` rows in one launch: ``silu(gate) * up`` of ``a`` (``weight``: gate rows over up rows)
    and ``a2 @ weight2.T + bias2``, in bf16."""
    lda, lda2 = _beside_rows("a", a, weight), _beside_rows("a2", a2, weight2)
    (n, k), n2, m = weight.shape, weight2.shape[0], a.shape[0]
    if weight2.shape[1] != k or a2.shape[0] != m or n % 2 or waves not in (2, 3, 4):
        raise ValueError(f"products {tuple(a.shape)} x {tuple(weight.shape)} and {tuple(a2.shape)} x {tuple(weight2.shape)}, {waves} waves")
    if bias2 is not None:
        _gpu("bias2", bias2, torch.bfloat16, 1)
        if bias2.shape[0] != n2:
            raise ValueError(f"bias2 must be [{n2}]")
    out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=a.device)
    out2 = torch.empty((m, n2), dtype=torch.bfloat16, device=a.device)
    _run("cie_gemm_silu_beside", load_library().cie_gemm_silu_beside(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(out), _ptr(a2), _i(lda2), _ptr(weight2), _ptr(bias2), _ptr(out2), _i(m), _i(n),
        _i(n2), _i(k), _i(waves)))
    return out, out2


def gemm_parts_beside(weight: torch.Tensor, a: torch.Tensor, parts: int, weight2: torch.Tensor, a2: torch.Tensor,
                      parts2: int) -> torch.Tensor:
    """The float32 partial sums [parts + parts2, M, N] of ``a @ weight.T + a2 @ weight2.T``, up to ``BESIDE_ROWS`` rows, in one
    launch: ``parts`` parts of the first product's K, ``parts2`` of the second's."""
    lda, lda2 = _beside_rows("a", a, weight), _beside_rows("a2", a2, weight2)
    (n, k), m = weight.shape, a.shape[0]
    if weight2.shape[0] != n or a2.shape[0] != m or parts < 1 or parts2 < 1 or parts + parts2 > 64:
        raise ValueError(f"products {tuple(a.shape)} x {tuple(weight.shape)} and {tuple(a2.shape)} x {tuple(weight2.shape)} in {parts}, {parts2} parts")
    out = torch.empty((parts + parts2, m, n), dtype=torch.float32, device=a.device)
    _run("cie_gemm_parts_beside", load_library().cie_gemm_parts_beside(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _i(k), _i(parts), _ptr(a2), _i(lda2), _ptr(weight2), _i(weight2.shape[1]),
        _i(parts2), _ptr(out), _i(m), _i(n)))
    return out


def gemm_shared_rows_normed(stream: torch.Tensor, norm_weight: torch.Tensor, eps: float, weight: torch.Tensor,
                            waves: int = 4) -> torch.Tensor:
    """:func:`gemm_shared_rows` with ``EPI_SILU`` over the RMSNorm of up to ``FOLDED_NORM_ROWS`` float32 rows, which the product
    makes itself."""
    _gpu("weight", weight, torch.bfloat16, 2)
    n, k = weight.shape
    _gpu("stream", stream, torch.float32, 2)
    _gpu("norm_weight", norm_weight, torch.float32, 1)
    m = stream.shape[0]
    if not (folds_norm(m, k) and stream.shape[1] == k and norm_weight.shape[0] == k and n % 2 == 0 and eps > 0 and waves in (2, 3, 4)):
        raise ValueError(f"{tuple(stream.shape)} rows, a norm of {norm_weight.shape[0]} and a weight {tuple(weight.shape)} do not fit")
    if stream.data_ptr() % 16 or norm_weight.data_ptr() % 16 or weight.data_ptr() % 16:
        raise ValueError("operands must be 16-byte aligned")
    out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=weight.device)
    _run("cie_gemm_shared_rows_normed", load_library().cie_gemm_shared_rows_normed(
        _stream(), _ptr(stream), _ptr(norm_weight), _f(eps), _ptr(weight), _ptr(out), _i(m), _i(n), _i(k), _i(waves)))
    return out


_WORKSPACES: dict[torch.device, torch.Tensor] = {}
LIBRARY_WORKSPACE_BYTES = 64 << 20
# Products of at least this many rows, in steps of 256 (full prompt portions), and of a power of two of rows
# from 32 on (the buckets of captured decode steps) are the shapes that recur: they time the library's
# candidate algorithms at their first call and keep the fastest; others take its first choice.
LIBRARY_TUNE_ROWS = 512
# Row counts whose products time every algorithm the library has, not only the heuristic's candidates (a few
# seconds for each shape, once in a process).  An engine names the sizes of its full prompt portions around its
# own steps (:func:`library_search`); outside of that nothing is searched, so one engine's choice does not
# reach another's steps.
_search_rows: frozenset = frozenset()


@contextlib.contextmanager
def library_search(rows):
    """While the block runs, library products of these row counts time every algorithm at a shape's first call."""
    global _search_rows
    previous, _search_rows = _search_rows, frozenset(rows)
    try:
        yield
    finally:
        _search_rows = previous


def _tune_level(rows: int) -> int:
    """How the library's algorithm for products of this many rows is chosen: 0 its first choice, 1 its candidates timed, 2 all
    its algorithms timed."""
    if rows >= LIBRARY_TUNE_ROWS and rows in _search_rows:
        return 2
    if (rows >= LIBRARY_TUNE_ROWS and rows % 256 == 0) or (rows >= 32 and rows & (rows - 1) == 0):
        return 1
    return 0


def gemm_library(a: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
                 out_dtype: torch.dtype = torch.bfloat16) -> Optional[torch.Tensor]:
    """``a @ weight.T + bias`` through the vendor library (hipBLASLt) with the
    descriptors and the chosen algorithm of every shape kept after its first call:
    bf16 operands and bias, float32 sums, bf16 result, or without bias a float32
    result.  For products with many rows.  Returns ``None`` if the library has no algorithm for the shape."""
    _gpu("weight", weight, torch.bfloat16, 2)
    n, k = weight.shape
    if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.stride(1) == 1):
        raise ValueError("a must be a bf16 GPU matrix with unit inner stride")
    m = a.shape[0]
    if not (m >= 1 and a.shape[1] == k):
        raise ValueError(f"a {tuple(a.shape)} vs K={k}")
    lda = a.stride(0) if m > 1 else max(a.stride(0), k)
    if out_dtype not in (torch.bfloat16, torch.float32) or (out_dtype == torch.float32 and bias is not None):
        raise ValueError(f"the result is bf16, or float32 without bias; asked for {out_dtype} with{'' if bias is not None else 'out'} bias")
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if bias.shape[0] != n:
            raise ValueError(f"bias must be [{n}]")
    device = weight.device
    workspace = _WORKSPACES.get(device)
    if workspace is None:
        # cleared once: algorithms that meet through flags in the workspace leave them cleared after each call
        workspace = _WORKSPACES[device] = torch.zeros(LIBRARY_WORKSPACE_BYTES, dtype=torch.uint8, device=device)
    out = torch.empty((m, n), dtype=out_dtype, device=device)
    code = load_library().cie_gemm_library(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(bias), _ptr(out), _i(m), _i(n), _i(k),
        _i(1 if out_dtype == torch.float32 else 0), _ptr(workspace), workspace.numel(),
        _i(_tune_level(m)))
    if code == 1:
        return None
    _run("cie_gemm_library", code)
    return out


QKV_SPLIT_PAIRS_BELOW = 128  # (of up to 16 rows: below this many pairs of tiles, one tile a workgroup)


FOLDED_NORM_ROWS = 16      # the most rows whose norm the q/k/v product makes itself: one tile of rows
# (norm kernel + product against the product that makes its norm, us in a captured chain: 3B shape 1 / 8 / 16 rows
# 9.0 / 10.6 / 10.9 against 7.1 / 7.9 / 8.9; 7B 13.3 / 15.2 / 16.0 against 11.3 / 12.8 / 14.2; 14B 21.1 / 22.3 /
# 23.4 against 18.9 / 20.2 / 22.0; 0.5B 7.0 / 8.3 / 8.5 against 5.7 / 6.6 / 7.4.  Every workgroup makes the rows
# anew, which costs it about 1 us: the rows are read in whole 256-byte segments, four rows a load, and pass through
# the wave's staging area; with every lane reading the values of its own matrix operand it cost 2 to 6 us and lost
# from the 7B width on.)


def folds_norm(rows: int, k: int) -> bool:
    """Whether ``gemm_qkv_rope`` takes ``folded=`` for this many rows of ``k`` values."""
    return 1 <= rows <= FOLDED_NORM_ROWS and k >= 8 and k % 8 == 0


TILE_BF16, TILE_SILU, TILE_RESID, TILE_PARTS = 0, 1, 2, 3
TILE_ATOMIC = 5  # (only straight into LDS: parts of K add into a float32 stream with atomic adds)
TILE_SHAPES = ((64, 64), (128, 64), (128, 128), (128, 256))  # columns x rows of a workgroup's tile
# ... of the kernel whose operands go straight into LDS (K a multiple of 64)
DIRECT_SHAPES = ((64, 64), (96, 64), (96, 128), (128, 64), (128, 128), (128, 192), (128, 256), (192, 128), (192, 192),
                 (192, 256), (256, 128), (256, 160), (256, 256))
DIRECT_FEW_SHAPES = DIRECT_SHAPES[:5]  # ... where its parts add atomically, or its rows are scaled
DIRECT_SLICE = 64
DIRECT_NUMBERS = 1 << 31  # an operand holds fewer numbers (their places are 32-bit numbers of bytes)


def direct_fits(rows: int, n: int, k: int, lda: int) -> bool:
    """Whether the kernel that loads straight into LDS takes a product of these sizes."""
    return k % DIRECT_SLICE == 0 and n * k < DIRECT_NUMBERS and rows * lda < DIRECT_NUMBERS


def _tile_rows(a: torch.Tensor, weight: torch.Tensor) -> tuple[int, int, int, int]:
    """(rows, columns, K, row stride) of a product that goes to the tile kernel, checked."""
    _gpu("weight", weight, torch.bfloat16, 2)
    if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.stride(1) == 1):
        raise ValueError("a must be a bf16 GPU matrix with unit inner stride")
    m, k = a.shape
    n = weight.shape[0]
    lda = a.stride(0) if m > 1 else max(a.stride(0), k)
    if not (m >= 1 and weight.shape[1] == k and k % 8 == 0 and lda % 8 == 0):
        raise ValueError(f"a {tuple(a.shape)} with row stride {lda} and weight {tuple(weight.shape)}: K and the stride are multiples of 8")
    if a.data_ptr() % 16 or weight.data_ptr() % 16:
        raise ValueError("operands must be 16-byte aligned")
    return m, n, k, lda


def _check_tile_shape(columns: int, rows: int, direct: bool, m: int, n: int, k: int, lda: int, few: bool = False) -> None:
    shapes = DIRECT_FEW_SHAPES if few else DIRECT_SHAPES if direct else TILE_SHAPES
    if (columns, rows) not in shapes:
        raise ValueError(f"tiles are one of {shapes}, not {(columns, rows)}")
    if direct and not direct_fits(m, n, k, lda):
        raise ValueError(f"{m} x {n} x {k} with row stride {lda}: K is a multiple of {DIRECT_SLICE}, an operand below 2^31 numbers")


def gemm_tiles(weight: torch.Tensor, epilogue: int, a: torch.Tensor, columns: int, rows: int,
               bias: Optional[torch.Tensor] = None, into: Optional[torch.Tensor] = None, parts: int = 1,
               direct: bool = False) -> torch.Tensor:
    """``a @ weight.T + bias`` in bfloat16 for some hundred rows, in tiles of ``columns`` x ``rows``: the bf16 result, its
    gated unit (``TILE_SILU``), added in place to the float32 stream ``into`` (``TILE_RESID``), or K in ``parts`` parts
    whose float32 sums come back as [parts, M, N] (``TILE_PARTS``).  ``direct``: by the kernel that loads its operands
    straight into LDS (``DIRECT_SHAPES``; K a multiple of 64); there the parts may also add themselves into ``into``
    (``TILE_ATOMIC``: in no fixed order)."""
    if epilogue == TILE_ATOMIC and not direct:
        raise ValueError("parts add themselves into the stream only in the kernel that loads straight into LDS")
    m, n, k, lda = _tile_rows(a, weight)
    _check_tile_shape(columns, rows, direct, m, n, k, lda, epilogue == TILE_ATOMIC)
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if not (bias.shape[0] == n and epilogue != TILE_SILU):
            raise ValueError("bias does not fit")
    if epilogue in (TILE_RESID, TILE_ATOMIC):
        _gpu("into", into, torch.float32, 2)
        if not (into.shape == (m, n) and into.data_ptr() % 16 == 0):
            raise ValueError(f"into must be {(m, n)}, is {tuple(into.shape)}")
        out = into
    elif epilogue == TILE_PARTS:
        out = torch.empty((parts, m, n), dtype=torch.float32, device=a.device)
    else:
        out = torch.empty((m, n // 2 if epilogue == TILE_SILU else n), dtype=torch.bfloat16, device=a.device)
    entry = "cie_gemm_direct" if direct else "cie_gemm_tiles"
    _run(entry, getattr(load_library(), entry)(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(bias), _ptr(out), _i(out.shape[-1]), _i(m), _i(n), _i(k), _i(epilogue),
        _i(columns), _i(rows), _i(parts)))
    return out


def gemm_tiles_silu_scaled(weight: torch.Tensor, a: torch.Tensor, columns: int, rows: int, row_sumsq: torch.Tensor,
                           eps: float) -> torch.Tensor:
    """The gated unit of :func:`gemm_tiles` (``direct``) of rows that lack their 1/rms, which it applies to its sums:
    ``row_sumsq`` [M, parts] holds partial sums of squares of the stream's rows (as ``gemm_fused`` takes them)."""
    m, n, k, lda = _tile_rows(a, weight)
    _check_tile_shape(columns, rows, True, m, n, k, lda, True)
    _gpu("row_sumsq", row_sumsq, torch.float32, 2)
    if not (n % 2 == 0 and row_sumsq.shape[0] == m and row_sumsq.shape[1] >= 1 and eps > 0 and row_sumsq.data_ptr() % 16 == 0):
        raise ValueError(f"row_sumsq {tuple(row_sumsq.shape)} does not fit {m} rows, or the weight's {n} rows are no pairs")
    out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=a.device)
    _run("cie_gemm_direct_silu_scaled", load_library().cie_gemm_direct_silu_scaled(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(out), _i(n // 2), _i(m), _i(n), _i(k), _i(columns), _i(rows),
        _ptr(row_sumsq), _i(row_sumsq.shape[1]), _f(eps)))
    return out


def gemm_tiles_rope(weight: torch.Tensor, a: torch.Tensor, bias: Optional[torch.Tensor], cos: torch.Tensor,
                    sin: torch.Tensor, positions: torch.Tensor, seq_of_token: torch.Tensor, seq_slot: torch.Tensor,
                    block_table: torch.Tensor, k_pool: torch.Tensor, v_pool: torch.Tensor, q_heads: int, kv_heads: int,
                    head_dim: int, columns: int, rows: int, rotate: bool = True, write_kv: bool = True,
                    direct: bool = False) -> torch.Tensor:
    """What :func:`gemm_qkv_rope` does, for some hundred rows in tiles of ``columns`` x ``rows`` (``direct``: as in
    :func:`gemm_tiles`)."""
    m, n, k, lda = _tile_rows(a, weight)
    _check_tile_shape(columns, rows, direct, m, n, k, lda)
    if head_dim % 32 or n != (q_heads + 2 * kv_heads) * head_dim:
        raise ValueError(f"tiles of {columns} x {rows}, heads of {head_dim}, {n} weight rows do not fit")
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if not (bias.shape[0] == n):
            raise ValueError("bias does not fit")
    for name, table in (("cos", cos), ("sin", sin)):
        _gpu(name, table, torch.float32, 2)
        if rotate and not (table.shape[1] == head_dim // 2 and table.data_ptr() % 16 == 0 and cos.shape == sin.shape):
            raise ValueError(f"{name} must be [max_position, {head_dim // 2}]")
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= m):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {m} rows")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    _gpu("block_table", block_table, torch.int32, 2)
    page_size = _check_pools(k_pool, v_pool, torch.bfloat16, kv_heads, head_dim)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=a.device)
    entry = "cie_gemm_direct_rope" if direct else "cie_gemm_tiles_rope"
    _run(entry, getattr(load_library(), entry)(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(bias), _ptr(out), _i(m), _i(n), _i(k), _i(columns), _i(rows),
        _ptr(cos), _ptr(sin), _ptr(positions), _ptr(seq_of_token), _ptr(seq_slot), _ptr(block_table),
        _i(block_table.shape[1]), _ptr(k_pool), _ptr(v_pool), _i(q_heads), _i(kv_heads), _i(head_dim), _i(page_size),
        _i(1 if rotate else 0), _i(1 if write_kv else 0)))
    return out


@functools.lru_cache(maxsize=4096)
def _plan_qkv_row_blocks(rows: int, pairs: int, k: int, units: int) -> tuple[int, int, bool]:
    # (the waves of the plain product, so that both cut K alike: four keep too little of a long K in flight for four row tiles, and
    # one row tile gained with the pair only)
    _, waves = _plan_row_blocks(rows, 2 * pairs, k, units)
    forms = ((2, 1), (2, 2)) if waves == 4 and k > FUSED_SHORT_K else ((4, 1), (4, 2), (2, 1), (2, 2)) + (((1, 2),) if waves == 8 else ())
    row_tiles, tiles = min(forms, key=lambda f: _row_blocks(rows, f[0], f[1], 2 * pairs // f[1], units, k, whole=False))
    return row_tiles, 4 if row_tiles <= 2 and k <= FUSED_SHORT_K else waves, tiles == 1


def plan_qkv_rope(rows: int, pairs: int, k: int, folded: bool = False) -> tuple[int, int, bool]:
    """(row tiles, waves per workgroup, whether a workgroup takes one tile of 16 columns and not a pair) of ``gemm_qkv_rope``
    for ``pairs`` pairs of tiles.  Up to 16 rows: one tile where the pairs leave half of the units without a workgroup (80 pairs
    8.1 -> 7.2 us), but for a short K, of which a pair's four waves have all in flight too, and read the rows once for twice the columns
    (``folded``: with the norm made in the product, one tile and a pair: 1,152 x 896 1 row 5.8, 5.2, 8 6.5 either way, 16 7.5, 7.0; 3,072 x
    1,024 6.5, 6.1, 7.6 either way, 8.6, 8.0; 2,048 x 1,536 6.8, 8.1; without it a pair gains up to a K of 512, 2 to 5 %, and loses beyond,
    3,072 x 824, 16 rows 6.1, 6.6).  Beyond, as :func:`plan_fused` (MI355X, us, up to 64 rows a workgroup, one tile up to 64 rows and fewer than
    128 pairs, and what is taken: 2,560 x 2,048 48 rows 9.8, 8.7, 64 10.1, 9.3, 96 11.7, 9.4; 1,152 x 896 64 rows 7.8, 5.7, 96
    8.9, 5.7; 3,072 x 2,048 64 rows 10.6, 9.6)."""
    if rows > 16:
        return _plan_qkv_row_blocks(rows, pairs, k, compute_units())
    _, waves, _ = plan_fused(rows, pairs, k)
    few = pairs < QKV_SPLIT_PAIRS_BELOW
    return 1, min(waves, 4) if few else waves, few and k > (FUSED_SHORT_K if folded else FUSED_SHORT_K // 2)


def gemm_qkv_rope(weight: torch.Tensor, a: Optional[torch.Tensor], bias: Optional[torch.Tensor], cos: torch.Tensor,
                  sin: torch.Tensor, positions: torch.Tensor, seq_of_token: torch.Tensor, seq_slot: torch.Tensor,
                  block_table: torch.Tensor, k_pool: torch.Tensor, v_pool: torch.Tensor, q_heads: int,
                  kv_heads: int, head_dim: int, rotate: bool = True, write_kv: bool = True,
                  waves: Optional[int] = None, folded: Optional[tuple] = None,
                  blocks: Optional[tuple[int, bool]] = None) -> torch.Tensor:
    """The q/k/v product of a few rows (64 per workgroup) fused with what ``rope_kv_write`` does:
    ``a @ weight.T + bias`` for weight [(Hq+2Hkv)*D, K], queries and keys rotated
    by each row's position, keys and values written into the cache.  Returns the
    buffer [M, (Hq+2Hkv)*D] whose query columns hold the rotated queries (its key
    and value columns are not written).  Same results as ``gemm_fused`` followed
    by ``rope_kv_write``.  Head sizes in steps of 32.

    ``folded=(residual, norm_weight, eps)`` instead of ``a`` (``folds_norm`` says for which sizes): the rows
    are the RMSNorm of ``residual`` (float32 [M, K], float32 weight), made inside the product: a lane makes
    the values of its matrix operand from the stream, and the rows' 1/rms multiplies the sums.

    ``blocks``: (row tiles, one tile a workgroup) instead of the planned ones."""
    _gpu("weight", weight, torch.bfloat16, 2)
    n, k = weight.shape
    if folded is not None:
        residual, norm_weight, eps = folded
        _gpu("residual", residual, torch.float32, 2)
        _gpu("norm_weight", norm_weight, torch.float32, 1)
        m = residual.shape[0]
        if a is not None or not folds_norm(m, k):
            raise ValueError(f"the product makes the norm of up to {FOLDED_NORM_ROWS} rows itself, not of {m} rows "
                             f"of {k}; and then takes no rows")
        if not (residual.shape == (m, k) and norm_weight.shape == (k,) and eps > 0):
            raise ValueError(f"residual {tuple(residual.shape)}, weight {tuple(norm_weight.shape)} do not fit rows of K={k}")
        if not (residual.is_contiguous() and norm_weight.is_contiguous()
                and residual.data_ptr() % 16 == 0 and norm_weight.data_ptr() % 16 == 0):
            raise ValueError("residual and weight must be contiguous and 16-byte aligned")
        lda = k
    else:
        if not (a.is_cuda and a.dtype == torch.bfloat16 and a.dim() == 2 and a.stride(1) == 1):
            raise ValueError("a must be a bf16 GPU matrix with unit inner stride")
        m = a.shape[0]
        if not (m >= 1 and a.shape[1] == k):
            raise ValueError(f"a {tuple(a.shape)}: rows of K={k}")
        lda = a.stride(0) if m > 1 else max(a.stride(0), k)
        if not (a.data_ptr() % 16 == 0):
            raise ValueError("operands must be 16-byte aligned")
    if not (k % 8 == 0 and lda % 8 == 0):
        raise ValueError(f"K and the row stride must be multiples of 8, are {k} and {lda}")
    if not (weight.data_ptr() % 16 == 0):
        raise ValueError("operands must be 16-byte aligned")
    if not (head_dim % 32 == 0):
        raise ValueError(f"the fused rotation takes head sizes in steps of 32, not {head_dim}")
    if not (n == (q_heads + 2 * kv_heads) * head_dim):
        raise ValueError(f"weight has {n} rows, heads say {(q_heads + 2 * kv_heads) * head_dim}")
    if bias is not None:
        _gpu("bias", bias, torch.bfloat16, 1)
        if not (bias.shape[0] == n):
            raise ValueError("bias does not fit")
    for name, table in (("cos", cos), ("sin", sin)):
        _gpu(name, table, torch.float32, 2)
        if not (table.shape[1] == head_dim // 2):
            raise ValueError(f"{name} must be [max_position, {head_dim // 2}]")
    if not (cos.shape == sin.shape):
        raise ValueError("cos and sin tables differ in shape")
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= m):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {m} rows")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    _gpu("block_table", block_table, torch.int32, 2)
    page_size = _check_pools(k_pool, v_pool, torch.bfloat16, kv_heads, head_dim)
    row_tiles, planned, one_tile = plan_qkv_rope(m, n // 32, k, folded is not None)
    waves = planned if waves is None else waves
    if blocks is not None:
        row_tiles, one_tile = blocks
    if not (row_tiles in ((1,) if m <= 16 else (1, 2, 4)) and waves in ((1, 2, 4, 8) if row_tiles == 1 else (4, 8))):
        raise ValueError(f"{waves} waves per workgroup and {row_tiles} row tiles with {m} rows is not a form the kernel has")
    out = torch.empty((m, n), dtype=torch.bfloat16, device=weight.device)
    if folded is not None:
        _run("cie_gemm_qkv_rope_folded_norm", load_library().cie_gemm_qkv_rope_folded_norm(
            _stream(), _ptr(residual), _ptr(norm_weight), _f(eps),
            _ptr(weight), _ptr(bias), _ptr(out), _i(m), _i(n), _i(k), _i(waves), _i(one_tile), _ptr(cos), _ptr(sin), _ptr(positions),
            _ptr(seq_of_token), _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]), _ptr(k_pool), _ptr(v_pool),
            _i(q_heads), _i(kv_heads), _i(head_dim), _i(page_size), _i(1 if rotate else 0), _i(1 if write_kv else 0)))
        return out
    _run("cie_gemm_qkv_rope", load_library().cie_gemm_qkv_rope(
        _stream(), _ptr(a), _i(lda), _ptr(weight), _ptr(bias), _ptr(out), _i(m), _i(n), _i(k), _i(row_tiles), _i(waves), _i(one_tile),
        _ptr(cos), _ptr(sin), _ptr(positions), _ptr(seq_of_token), _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]),
        _ptr(k_pool), _ptr(v_pool), _i(q_heads), _i(kv_heads), _i(head_dim), _i(page_size),
        _i(1 if rotate else 0), _i(1 if write_kv else 0)))
    return out


ARGMAX_CHUNK = 2048


def sample(logits: torch.Tensor, temperature: Optional[torch.Tensor] = None,
           uniform: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """One token per row of float32 logits: argmax where the row's temperature
    is 0 (or none is given), else a draw with the row's uniform number."""
    _gpu("logits", logits, torch.float32, 2)
    rows, vocab = logits.shape
    if temperature is None and vocab >= 4 * ARGMAX_CHUNK:
        if out is None:
            out = torch.empty((rows,), dtype=torch.int32, device=logits.device)
        chunks = -(-vocab // ARGMAX_CHUNK)
        chunk_val = torch.empty(rows * chunks, dtype=torch.float32, device=logits.device)
        chunk_idx = torch.empty(rows * chunks, dtype=torch.int32, device=logits.device)
        _run("cie_argmax", load_library().cie_argmax(_stream(), _ptr(logits), _ptr(chunk_val), _ptr(chunk_idx),
                                                     _ptr(out), _i(rows), _i(vocab), _i(vocab), _i(ARGMAX_CHUNK)))
        return out
    if temperature is not None:
        _gpu("temperature", temperature, torch.float32, 1)
        if not (uniform is not None):
            raise ValueError("temperature sampling needs the uniform numbers")
        _gpu("uniform", uniform, torch.float32, 1)
        if not (temperature.shape[0] == rows and uniform.shape[0] == rows):
            raise ValueError("one temperature and one uniform per row")
    if out is None:
        out = torch.empty((rows,), dtype=torch.int32, device=logits.device)
    _gpu("out", out, torch.int32, 1)
    if not (out.shape[0] == rows):
        raise ValueError(f"out must be [{rows}]")
    if temperature is not None and vocab >= 4 * ARGMAX_CHUNK:
        # a row is taken by many workgroups (one per row reads a vocabulary of 150,000 in a quarter of a millisecond)
        parts = -(-vocab // ARGMAX_CHUNK)
        part_val = torch.empty(rows * parts, dtype=torch.float32, device=logits.device)
        part_idx = torch.empty(rows * parts, dtype=torch.int32, device=logits.device)
        part_sum = torch.empty(rows * parts, dtype=torch.float32, device=logits.device)
        _run("cie_sample_parts", load_library().cie_sample_parts(
            _stream(), _ptr(logits), _ptr(temperature), _ptr(uniform), _ptr(part_val), _ptr(part_idx), _ptr(part_sum),
            _ptr(out), _i(rows), _i(vocab), _i(vocab), _i(ARGMAX_CHUNK)))
        return out
    _run("cie_sample", load_library().cie_sample(_stream(), _ptr(logits), _ptr(temperature), _ptr(uniform),
                                                 _ptr(out), _i(rows), _i(vocab), _i(vocab)))
    return out


# ---------------------------------------------------------------------------
# A stream that is averaged over the depth, block-diagonal products, compressed keys, recurrent mixers
def depth_stream(x: torch.Tensor, branch_a: Optional[torch.Tensor] = None, branch_b: Optional[torch.Tensor] = None,
                 mult: float = 1.0, history: Optional[torch.Tensor] = None, newest: int = -1,
                 weights: Optional[torch.Tensor] = None, gains: tuple = (), out_dtype: torch.dtype = torch.float32,
                 eps: float = 1e-6, want_stream: bool = True, parts: Optional[torch.Tensor] = None):
    """One layer boundary of a stream whose layers add two parallel branches and whose next input is a weighted
    average of what the embedding and every layer so far left:

    ``v = x + mult * (branch_a + branch_b)`` (float32; without branches ``v = x``; ``parts`` [P, T, H] float32:
    their sum, in order, is one more branch, or all there is); ``history[newest] = v``;
    with ``weights`` (float32 [terms]) ``v = sum_j weights[j] * history[j]``; then for every gain ``g`` in
    ``gains`` (up to two) the rows ``v / sqrt(mean(v^2) + eps) * g`` in ``out_dtype``.

    x float32 [T, H]; branches [T, H] in ``out_dtype``; history float32 [layers + 1, T, H].  Returns
    ``(stream or None, [normed rows per gain])``; the stream is a new tensor (``want_stream``) unless nothing changed it."""
    _gpu("x", x, torch.float32, 2)
    rows, hidden = x.shape
    if hidden > MAX_NORM_WIDTH:
        raise ValueError(f"rows of up to {MAX_NORM_WIDTH} numbers, not {hidden}")
    for name, branch in (("branch_a", branch_a), ("branch_b", branch_b)):
        if branch is not None:
            _gpu(name, branch, out_dtype, 2)
            if branch.shape != x.shape:
                raise ValueError(f"{name} {tuple(branch.shape)} vs the stream {tuple(x.shape)}")
    if branch_b is not None and branch_a is None:
        raise ValueError("a second branch needs a first")
    if parts is not None:
        _gpu("parts", parts, torch.float32, 3)
        if tuple(parts.shape[1:]) != (rows, hidden):
            raise ValueError(f"parts {tuple(parts.shape)} for a stream of {tuple(x.shape)}")
    terms, stride = 0, 0
    if history is not None:
        _gpu("history", history, torch.float32, 3)
        if tuple(history.shape[1:]) != (rows, hidden) or not -1 <= newest < history.shape[0]:
            raise ValueError(f"history {tuple(history.shape)} does not hold rows of {tuple(x.shape)} at {newest}")
        stride = rows * hidden
    elif newest >= 0:
        raise ValueError("a place in the history needs the history")
    if weights is not None:
        _gpu("weights", weights, torch.float32, 1)
        terms = weights.shape[0]
        if history is None or terms > history.shape[0]:
            raise ValueError(f"{terms} weights for a history of {0 if history is None else history.shape[0]}")
    if len(gains) > 2 or not eps > 0:
        raise ValueError("at most two norms, and a positive eps")
    changed = branch_a is not None or parts is not None or terms > 0
    stream = torch.empty_like(x) if (want_stream and changed) else None
    outs = [torch.empty((rows, hidden), dtype=out_dtype, device=x.device) for _ in gains]
    g = [float(v) for v in gains] + [0.0, 0.0]
    _run("cie_depth_stream", load_library().cie_depth_stream(
        _stream(), _i(_code(out_dtype)), _ptr(x), _ptr(branch_a), _ptr(branch_b), _f(mult), _ptr(history), stride,
        _i(newest), _ptr(weights), _i(terms), _ptr(stream), _ptr(outs[0] if outs else None), _f(g[0]),
        _ptr(outs[1] if len(outs) > 1 else None), _f(g[1]), _i(rows), _i(hidden), _f(eps), _ptr(parts),
        _i(0 if parts is None else parts.shape[0])))
    return (stream if stream is not None else (x if want_stream else None)), outs


def block_linear(a: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
                 a_block: Optional[int] = None, out: Optional[torch.Tensor] = None, out_offset: int = 0,
                 c_block: Optional[int] = None, out_dtype: Optional[torch.dtype] = None,
                 gate: Optional[torch.Tensor] = None, gate_offset: int = 0, a_offset: int = 0) -> torch.Tensor:
    """A block-diagonal product: ``out[m, b, :] = a[m, b, :] @ weight[b].T (+ bias[b])``, times
    ``sigmoid(gate[m, b, :])`` if a gate is given.

    ``a`` [M, >= a_offset + (B-1) * a_block + K] with unit inner stride (block b's K numbers start at column
    ``a_offset + b * a_block``; ``a_block`` defaults to K); ``weight`` [B, N, K]; ``bias`` [B, N].  The result goes to
    columns ``out_offset + b * c_block`` (``c_block`` defaults to N) of ``out``, a new [M, B * N] tensor of ``out_dtype``
    (float32 or ``a``'s type) if none is given.  ``gate`` is laid out like the default result from its column
    ``gate_offset`` on.  float32 sums in one fixed order; float32 operands give a true float32 product."""
    _gpu("weight", weight, a.dtype, 3)
    blocks, n, k = weight.shape
    if not (a.is_cuda and a.dim() == 2 and a.stride(1) == 1 and a.dtype in _CODES):
        raise ValueError("a must be a float32 or bfloat16 GPU matrix with unit inner stride")
    a_block = k if a_block is None else a_block
    m = a.shape[0]
    if a_offset < 0 or a_block < 0 or a.shape[1] < a_offset + (blocks - 1) * a_block + k:
        raise ValueError(f"a {tuple(a.shape)} does not hold {blocks} blocks of {k} numbers {a_block} apart from {a_offset}")
    lda = a.stride(0) if m > 1 else max(a.stride(0), a.shape[1])
    if bias is not None:
        _gpu("bias", bias, a.dtype, 2)
        if tuple(bias.shape) != (blocks, n):
            raise ValueError(f"bias must be {(blocks, n)}")
    c_block = n if c_block is None else c_block
    if out is None:
        out_dtype = out_dtype or a.dtype
        out = torch.empty((m, out_offset + (blocks - 1) * c_block + n), dtype=out_dtype, device=a.device)
    if not (out.is_cuda and out.dim() == 2 and out.stride(1) == 1 and out.shape[0] == m
            and out.dtype in (torch.float32, a.dtype)):
        raise ValueError("out must be a GPU matrix of float32 or a's type with a row per row of a")
    if out_offset < 0 or c_block < n or out.shape[1] < out_offset + (blocks - 1) * c_block + n:
        raise ValueError(f"out {tuple(out.shape)} does not hold {blocks} blocks of {n} results {c_block} apart from {out_offset}")
    ldc = out.stride(0) if m > 1 else max(out.stride(0), out.shape[1])
    ldg = 0
    if gate is not None:
        if not (gate.is_cuda and gate.dim() == 2 and gate.stride(1) == 1 and gate.dtype == a.dtype and gate.shape[0] == m
                and gate.shape[1] >= gate_offset + blocks * n):
            raise ValueError("the gate must be a matrix of a's type with a row per row of a and a number per result")
        ldg = gate.stride(0) if m > 1 else max(gate.stride(0), gate.shape[1])
    esz_a, esz_c = a.element_size(), out.element_size()
    _run("cie_block_linear", load_library().cie_block_linear(
        _stream(), _i(_code(a.dtype)), _i(1 if out.dtype == torch.float32 else 0), a.data_ptr() + a_offset * esz_a, lda,
        a_block, _ptr(weight), _ptr(bias), out.data_ptr() + out_offset * esz_c, ldc, c_block,
        None if gate is None else gate.data_ptr() + gate_offset * esz_a, ldg, n, _i(m), _i(n), _i(k), _i(blocks)))
    return out


def latent_rows(proj: torch.Tensor, weight: torch.Tensor, heads: int, plain: int, turned: int, latent: int,
                width: int, eps: float, rotary: Optional[tuple[torch.Tensor, torch.Tensor]], positions: torch.Tensor,
                seq_of_token: torch.Tensor, seq_slot: torch.Tensor, block_table: torch.Tensor, k_pool: torch.Tensor,
                v_pool: torch.Tensor, write_kv: bool = True) -> torch.Tensor:
    """What lies between the joint projection and the attention kernels of a layer whose keys are compressed
    (``csrc/latent.hip``).  ``proj`` [T, heads * (plain + turned) + latent + turned].  Returns the query rows
    ``[T, heads * width]``: per head its turned part, turned by the token's position, room for its folded plain part,
    and zeros.  Writes every token's cache entry, key ``[turned part | normed latent | zeros]`` and value
    ``[zeros | normed latent | zeros]``, where ``write_kv``.  ``rotary``: (cos, sin) float32 [max_position, turned / 2],
    or ``None`` where nothing turns; pools as for ``rope_kv_write`` with one head of ``width``."""
    if not (proj.is_cuda and proj.dim() == 2 and proj.stride(1) == 1 and proj.dtype in _CODES):
        raise ValueError("proj must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens = proj.shape[0]
    if proj.shape[1] != heads * (plain + turned) + latent + turned or width < turned + latent:
        raise ValueError(f"proj {tuple(proj.shape)} does not fit {heads} heads of {plain}+{turned} and a latent of {latent}+{turned}")
    _gpu("weight", weight, dims=1)
    if weight.shape[0] != latent or weight.dtype not in (proj.dtype, torch.float32):
        raise ValueError("the latent's norm weight does not fit")
    cos = sin = None
    if rotary is not None:
        cos, sin = rotary
        if turned <= 0 or turned % 2:
            raise ValueError(f"the turned part must be even, is {turned}")
        for name, table in (("cos", cos), ("sin", sin)):
            _gpu(name, table, torch.float32, 2)
            if not (table.shape[1] == turned // 2):
                raise ValueError(f"{name} must be [max_position, {turned // 2}]")
        if not (cos.shape == sin.shape):
            raise ValueError("cos and sin tables differ in shape")
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= tokens):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {tokens} tokens")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    _gpu("block_table", block_table, torch.int32, 2)
    page_size = _check_pools(k_pool, v_pool, proj.dtype, 1, width)
    rows = torch.empty((tokens, heads * width), dtype=proj.dtype, device=proj.device)
    ldp = proj.stride(0) if tokens > 1 else max(proj.stride(0), proj.shape[1])
    _run("cie_latent_rows", load_library().cie_latent_rows(
        _stream(), _i(_code(proj.dtype)), _i(_code(weight.dtype)), _ptr(proj), ldp, _ptr(weight), _ptr(rows), _ptr(cos),
        _ptr(sin), _i(turned if rotary is not None else 0), _ptr(positions), _ptr(seq_of_token), _ptr(seq_slot),
        _ptr(block_table), _i(block_table.shape[1]), _ptr(k_pool), _ptr(v_pool), _i(page_size), _i(1 if write_kv else 0),
        _i(tokens), _i(heads), _i(plain), _i(turned), _i(latent), _i(width), _f(eps)))
    return rows


def latent_down(proj: torch.Tensor, q_off: int, q_rank: int, c_off: int, q_weight: Optional[torch.Tensor],
                c_weight: torch.Tensor, latent: int, turned: int, rotary: Optional[tuple], positions: torch.Tensor,
                seq_of_token: torch.Tensor, seq_slot: torch.Tensor, block_table: torch.Tensor, k_pool: torch.Tensor,
                v_pool: torch.Tensor, eps: float, write_kv: bool = True) -> Optional[torch.Tensor]:
    """Behind the down projections of a layer whose keys are compressed (``csrc/latent.hip``): the query latent
    (``q_rank`` numbers from column ``q_off`` of ``proj``; 0: none) under its RMS norm comes back as [T, q_rank]; the key
    latent (``latent`` numbers from ``c_off``) under its own and the shared key part behind it (``turned`` numbers, turned
    by the position) go to the token's place in the cache: keys ``[turned | latent | zeros]``, values ``[latent | zeros]``.
    ``rotary = (cos, sin, rot, neighbours)`` or ``None``; norm weights float32."""
    if not (proj.is_cuda and proj.dim() == 2 and proj.stride(1) == 1 and proj.dtype in _CODES):
        raise ValueError("proj must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens = proj.shape[0]
    if min(q_off, q_rank, c_off) < 0 or proj.shape[1] < max(q_off + q_rank, c_off + latent + turned):
        raise ValueError(f"proj {tuple(proj.shape)} does not hold latents of {q_rank} and {latent}+{turned} at {q_off}, {c_off}")
    for name, w, size in (("q_weight", q_weight if q_rank else None, q_rank), ("c_weight", c_weight, latent)):
        if w is not None:
            _gpu(name, w, torch.float32, 1)
            if w.shape[0] != size:
                raise ValueError(f"{name} must be [{size}], is {tuple(w.shape)}")
    if q_rank and q_weight is None:
        raise ValueError("the query latent's norm has a weight")
    width, value_width = k_pool.shape[3], v_pool.shape[2]
    page_size = _check_kv_pools(k_pool, v_pool, proj.dtype, 1, width, value_width)
    if width < latent + turned or value_width < latent:
        raise ValueError(f"cache entries of {width} and {value_width} do not hold a latent of {latent} and {turned} turned numbers")
    cos, sin, rot, neighbours = _check_rotary(rotary, turned)
    _gpu("block_table", block_table, torch.int32, 2)
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < tokens:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {tokens} tokens")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    q_latent = torch.empty((tokens, q_rank), dtype=proj.dtype, device=proj.device) if q_rank else None
    _run("cie_latent_down", load_library().cie_latent_down(
        _stream(), _i(_code(proj.dtype)), _ptr(proj), _ld(proj), _i(q_off), _i(q_rank), _i(c_off), _ptr(q_weight), _ptr(c_weight),
        _ptr(q_latent), _ptr(cos), _ptr(sin), _i(rot), _i(1 if neighbours else 0), _ptr(positions), _ptr(seq_of_token),
        _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]), _ptr(k_pool), _ptr(v_pool), _i(tokens), _i(latent),
        _i(turned), _i(width), _i(value_width), _i(page_size), _f(eps), _i(1 if write_kv else 0)))
    return q_latent


def _check_rotary(rotary: Optional[tuple], most: int) -> tuple:
    if rotary is None:
        return None, None, 0, False
    cos, sin, rot, neighbours = rotary
    if rot < 2 or rot % 2 or rot > most:
        raise ValueError(f"{rot} turning numbers of {most}: even, at least 2, at most all of them")
    for name, table in (("cos", cos), ("sin", sin)):
        _gpu(name, table, torch.float32, 2)
        if table.shape[1] != rot // 2:
            raise ValueError(f"{name} {tuple(table.shape)} does not hold {rot // 2} pairs per position")
    return cos, sin, rot, neighbours


def latent_queries(q: torch.Tensor, heads: int, plain: int, turned: int, latent: int, width: int, rotary: Optional[tuple],
                   positions: torch.Tensor) -> torch.Tensor:
    """Query rows [T, heads * width] for entries ``[turned | latent | zeros]`` from ``q`` [T, heads * (plain + turned)]:
    each head's turned part, turned by the position, and the zeros; the room between them is left for the folded part."""
    _row_view("q", q, (q.shape[0], heads * (plain + turned)), tuple(_CODES))
    tokens = q.shape[0]
    if width < turned + latent:
        raise ValueError(f"rows of {width} do not hold {turned} + {latent} numbers")
    cos, sin, rot, neighbours = _check_rotary(rotary, turned)
    _gpu("positions", positions, torch.int32, 1)
    if positions.shape[0] < tokens:
        raise ValueError("one position per token")
    rows = torch.empty((tokens, heads * width), dtype=q.dtype, device=q.device)
    _run("cie_latent_queries", load_library().cie_latent_queries(
        _stream(), _i(_code(q.dtype)), _ptr(q), _ld(q), _ptr(cos), _ptr(sin), _i(rot), _i(1 if neighbours else 0),
        _ptr(positions), _ptr(rows), _i(tokens), _i(heads), _i(plain), _i(turned), _i(latent), _i(width)))
    return rows


RETENTION_ROWS = (4, 8, 16, 32)  # rows of a head's memory that one thread keeps in registers
RETENTION_SLICE = 64             # value columns of a head that one workgroup takes
RETENTION_LDS_FLOATS = 15 * 1024
RETENTION_ACTIVATIONS = {None: 0, "silu": 1}   # what queries, keys and values pass through on their way in
RETENTION_GATES = {"silu": 0, "sigmoid": 1}    # the function of the gate columns that multiplies the read-out
RETENTION_BLOCKS_FROM = 16       # tokens a sequence (on average) from which the walk goes in blocks on the matrix cores
RETENTION_BLOCKS_MAX_DIM = 160   # ... for heads whose queries, keys and values of a block fit the LDS
RETENTION_BLOCKS_MAX_BYTES = 2 << 30  # ... and whose blocks' sums fit this much scratch memory


def plan_retention(dim: int, vdim: int, units: int = 1) -> tuple[int, int, int, int, int]:
    """(rows per thread, groups of threads, parts of the rows, value columns per workgroup, tokens per chunk) of
    the retention kernel for heads of ``dim`` x ``vdim`` when ``units`` (sequence, head) pairs run: a workgroup takes
    up to 64 value columns and a part of a head's rows, as many parts as give every compute unit a workgroup;
    workgroups of up to 512 threads."""
    if dim < 1 or vdim < 1 or units < 1:
        raise ValueError("head sizes must be positive")
    piece = min(vdim, RETENTION_SLICE)
    slices = -(-vdim // piece)
    most_groups = max(1, 512 // (-(-piece // 8) * 8))
    parts = max(1, min(compute_units() // (units * slices), -(-dim // 4)))
    parts = max(parts, -(-dim // (most_groups * RETENTION_ROWS[-1])))  # (no more rows than a workgroup can keep)
    share = -(-dim // parts)  # rows of a part
    rows = next((r for r in RETENTION_ROWS if -(-share // r) <= most_groups), None)
    if rows is None:
        raise ValueError(f"heads of {dim} x {vdim} do not fit the retention kernel's registers")
    groups = -(-share // rows)
    parts = -(-dim // (groups * rows))
    per_token = 2 * groups * rows + piece + groups * piece
    threads = -(-piece * groups // 64) * 64
    # (what a chunk holds must fit the LDS, and what a thread fetches ahead of a chunk its registers:
    # six 16-byte pieces of queries and keys and twelve values).  Long chunks: the next chunk's numbers are on
    # their way from memory for as long as the walk over the current one takes.
    chunk = min(48, RETENTION_LDS_FLOATS // per_token, 6 * threads * 4 // (2 * groups * rows), 12 * threads // piece)
    if chunk < 1 or threads > 512:
        raise ValueError(f"heads of {dim} x {vdim} do not fit the retention kernel's LDS")
    return rows, groups, parts, piece, chunk


RETENTION_STEP_THREADS = 1024  # of a workgroup; no more columns and rows of a head either (csrc/recurrent.hip)
RETENTION_STEP_ROWS = 8        # that a thread keeps, four columns each


def steps_retention(tokens: int, sequences: int, dim: int, vdim: int, norm_span: int) -> bool:
    """Whether a step goes to the kernel that turns, walks, norms and gates a head in one workgroup: one token a
    sequence, a norm over single heads, and heads whose memory a workgroup's registers hold in 16-byte pieces.  (Faster
    than the three kernels wherever it runs: heads of 4 x 72 to 256 x 128, 1 to 128 sequences, 1.7 to 3.5 times.)"""
    return (tokens == sequences and norm_span == 1 and vdim % 4 == 0 and max(dim, vdim) <= RETENTION_STEP_THREADS
            and vdim // 4 * -(-dim // RETENTION_STEP_ROWS) <= RETENTION_STEP_THREADS)


def retention(proj: torch.Tensor, offsets: tuple[int, int, int, int], cos: Optional[torch.Tensor],
              sin: Optional[torch.Tensor], rot: int, decay: torch.Tensor, state: torch.Tensor, seq_slot: torch.Tensor,
              positions: torch.Tensor, q_start_loc: torch.Tensor, sequences: int, heads: int, dim: int, vdim: int,
              eps: float, key_scale: float, longest_position: int, activation: Optional[str] = None,
              norm_span: int = 1, norm_weight: Optional[torch.Tensor] = None, gate: str = "silu") -> torch.Tensor:
    """Retention over a step's tokens (``csrc/recurrent.hip``; ``positions`` int32 [T] are the tokens' own).
    ``proj`` [T, ...] holds each token's queries, keys
    (heads x dim), values and gates (heads x vdim) from the columns ``offsets`` on; ``state`` float32
    [slots, heads, dim, vdim] is read and written at the sequences' slots; cos/sin float32 [positions, rot/2]
    must reach ``longest_position``.  ``activation="silu"``: queries, keys and values pass through silu on their way
    in.  The read-out is divided by its root mean square over runs of ``norm_span`` heads (1: each head alone;
    ``heads``: the token's whole row), multiplied by ``norm_weight`` (float32 [heads * vdim]) where given, and by
    ``silu`` or ``sigmoid`` (``gate``) of the gate columns.  Steps of ``RETENTION_BLOCKS_FROM`` tokens a sequence and more
    walk in blocks of 32 tokens on the matrix cores in float32 (heads of up to ``RETENTION_BLOCKS_MAX_DIM`` numbers a key,
    scratch of up to ``RETENTION_BLOCKS_MAX_BYTES``), others token by token, one token a sequence in one kernel
    (``steps_retention``): the same sums in another order.
    Returns [T, heads * vdim] in ``proj``'s type."""
    if activation not in RETENTION_ACTIVATIONS or gate not in RETENTION_GATES:
        raise ValueError(f"activation is one of {list(RETENTION_ACTIVATIONS)}, gate one of {list(RETENTION_GATES)}")
    if norm_span < 1 or heads % norm_span:
        raise ValueError(f"the norm's runs of {norm_span} heads do not divide {heads} heads")
    if norm_weight is not None:
        _gpu("norm_weight", norm_weight, torch.float32, 1)
        if norm_weight.shape[0] != heads * vdim:
            raise ValueError(f"norm_weight must be [{heads * vdim}], is {tuple(norm_weight.shape)}")
    if not (proj.is_cuda and proj.dim() == 2 and proj.stride(1) == 1 and proj.dtype in _CODES):
        raise ValueError("proj must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens = proj.shape[0]
    q_off, k_off, v_off, g_off = offsets
    if max(q_off + heads * dim, k_off + heads * dim, v_off + heads * vdim, g_off + heads * vdim) > proj.shape[1]:
        raise ValueError(f"proj {tuple(proj.shape)} does not hold the heads at {offsets}")
    if rot:
        for name, table in (("cos", cos), ("sin", sin)):
            _gpu(name, table, torch.float32, 2)
            if table.shape[1] != rot // 2 or table.shape[0] <= longest_position:
                raise ValueError(f"{name} {tuple(table.shape)} does not reach position {longest_position} with {rot // 2} pairs")
    _gpu("decay", decay, torch.float32, 1)
    _gpu("state", state, torch.float32, 4)
    if decay.shape[0] != heads or tuple(state.shape[1:]) != (heads, dim, vdim):
        raise ValueError(f"decay {tuple(decay.shape)} / state {tuple(state.shape)} do not fit {heads} heads of {dim} x {vdim}")
    for name, meta, least in (("seq_slot", seq_slot, sequences), ("positions", positions, tokens),
                              ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries, {least} are needed")
    ldp = proj.stride(0) if tokens > 1 else max(proj.stride(0), proj.shape[1])
    if steps_retention(tokens, sequences, dim, vdim, norm_span) and state.data_ptr() % 16 == 0:
        out = torch.empty((tokens, heads * vdim), dtype=proj.dtype, device=proj.device)
        _run("cie_retention_step", load_library().cie_retention_step(
            _stream(), _i(_code(proj.dtype)), _ptr(proj), ldp, _i(q_off), _i(k_off), _i(v_off),
            _i(g_off), _ptr(cos if rot else None), _ptr(sin if rot else None), _i(rot), _ptr(decay), _ptr(state),
            _ptr(seq_slot), _ptr(positions), _ptr(q_start_loc), _ptr(out), _i(sequences), _i(heads), _i(dim), _i(vdim),
            _f(eps), _f(key_scale), _i(RETENTION_ACTIVATIONS[activation]), _ptr(norm_weight), _i(RETENTION_GATES[gate])))
        return out
    rows, groups, parts, piece, chunk = plan_retention(dim, vdim, max(1, sequences * heads))
    # sequences that bring many tokens (prompts' portions) walk in blocks of 32 tokens on the matrix cores, float32
    # operands and sums, every block's own sums at once and only the memory itself in order; steps of few tokens a
    # sequence walk token by token.  (The same sums in another order.)
    padded, vdim16 = -(-dim // 16) * 16, -(-vdim // 16) * 16
    places = tokens // 32 + sequences + 1
    blocks = (tokens >= RETENTION_BLOCKS_FROM * max(sequences, 1) and dim <= RETENTION_BLOCKS_MAX_DIM
              and places * heads * padded * vdim16 * 4 <= RETENTION_BLOCKS_MAX_BYTES)
    sums = None
    if blocks:
        rows, groups, parts = 16, 1, padded // 16
        sums = torch.empty((places, heads, padded, vdim16), dtype=torch.float32, device=proj.device)
    turned = torch.empty((tokens, heads, 2, parts * groups * rows), dtype=torch.float32, device=proj.device)
    raw = torch.empty((2 if blocks else parts, tokens, heads * vdim), dtype=torch.float32, device=proj.device)
    out = torch.empty((tokens, heads * vdim), dtype=proj.dtype, device=proj.device)
    _run("cie_retention", load_library().cie_retention(
        _stream(), _i(_code(proj.dtype)), _ptr(proj), ldp, _i(q_off), _i(k_off), _i(v_off), _i(g_off),
        _ptr(cos if rot else None), _ptr(sin if rot else None), _i(rot), _ptr(decay), _ptr(state), _ptr(seq_slot),
        _ptr(positions), _ptr(q_start_loc), _ptr(turned), _ptr(raw), _ptr(out), _i(tokens), _i(sequences), _i(heads), _i(dim), _i(vdim),
        _i(rows), _i(groups), _i(parts), _i(piece), _i(chunk), _f(eps), _f(key_scale),
        _i(RETENTION_ACTIVATIONS[activation]), _i(norm_span), _ptr(norm_weight), _i(RETENTION_GATES[gate]),
        _i(1 if blocks else 0), _ptr(sums)))
    return out


MAX_CONV_TAPS = 16
MAX_SCAN_SEGMENTS = 64


def causal_conv(x: torch.Tensor, taps_w: torch.Tensor, bias: Optional[torch.Tensor], past: torch.Tensor,
                seq_of_token: torch.Tensor, seq_slot: torch.Tensor, q_start_loc: torch.Tensor,
                activation: Optional[str] = None, out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """Per channel, ``out[t] = act(sum_j taps_w[c, j] * x[t - (taps - 1) + j] + bias[c])`` within each sequence; the
    inputs before the step come from ``past`` (float32 [slots, max(taps - 1, 1), C], oldest first; zeros for a new
    sequence).  x [T, C] (a view with unit inner stride), taps_w [C, taps].  ``activation``: ``None`` or ``"silu"``;
    ``out_dtype``: x's type, or float32."""
    if not (x.is_cuda and x.dim() == 2 and x.stride(1) == 1 and x.dtype in _CODES):
        raise ValueError("x must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens, channels = x.shape
    _gpu("taps_w", taps_w, x.dtype, 2)
    taps = taps_w.shape[1]
    if taps_w.shape[0] != channels or not 1 <= taps <= MAX_CONV_TAPS:
        raise ValueError(f"taps {tuple(taps_w.shape)} for {channels} channels (up to {MAX_CONV_TAPS} taps)")
    if bias is not None:
        _gpu("bias", bias, x.dtype, 1)
        if bias.shape[0] != channels:
            raise ValueError(f"bias must be [{channels}]")
    _gpu("past", past, torch.float32, 3)
    if tuple(past.shape[1:]) != (max(taps - 1, 1), channels):
        raise ValueError(f"past {tuple(past.shape)} must be [slots, {max(taps - 1, 1)}, {channels}]")
    for name, meta in (("seq_of_token", seq_of_token), ("seq_slot", seq_slot), ("q_start_loc", q_start_loc)):
        _gpu(name, meta, torch.int32, 1)
    if seq_of_token.shape[0] < tokens:
        raise ValueError("one sequence index per token")
    if activation not in RETENTION_ACTIVATIONS or out_dtype not in (None, x.dtype, torch.float32):
        raise ValueError(f"activation {activation!r} / out_dtype {out_dtype} are none the convolution has")
    out = torch.empty((tokens, channels), dtype=out_dtype or x.dtype, device=x.device)
    ldx = x.stride(0) if tokens > 1 else max(x.stride(0), channels)
    _run("cie_causal_conv", load_library().cie_causal_conv(
        _stream(), _i(_code(x.dtype)), _ptr(x), ldx, _ptr(taps_w), _ptr(bias), _ptr(past), _ptr(seq_of_token),
        _ptr(seq_slot), _ptr(q_start_loc), _ptr(out), _i(tokens), _i(channels), _i(taps),
        _i(RETENTION_ACTIVATIONS[activation]), _i(1 if out.dtype == torch.float32 else 0)))
    return out


def conv_keep(x: torch.Tensor, past: torch.Tensor, seq_slot: torch.Tensor, q_start_loc: torch.Tensor, sequences: int,
              taps: int) -> None:
    """Moves a causal convolution's state on by a step's inputs ``x`` [T, C]: of what ``past`` (float32 [slots,
    max(taps - 1, 1), C]) held and the step's rows, the last ``taps - 1`` stay.  Runs behind the convolution."""
    if not (x.is_cuda and x.dim() == 2 and x.stride(1) == 1 and x.dtype in _CODES):
        raise ValueError("x must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens, channels = x.shape
    _gpu("past", past, torch.float32, 3)
    if tuple(past.shape[1:]) != (max(taps - 1, 1), channels) or not 1 <= taps <= MAX_CONV_TAPS:
        raise ValueError(f"past {tuple(past.shape)} must be [slots, {max(taps - 1, 1)}, {channels}]")
    for name, meta, least in (("seq_slot", seq_slot, sequences), ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {sequences} sequences")
    ldx = x.stride(0) if tokens > 1 else max(x.stride(0), channels)
    _run("cie_conv_keep", load_library().cie_conv_keep(_stream(), _i(_code(x.dtype)), _ptr(x), ldx, _ptr(past),
                                                       _ptr(seq_slot), _ptr(q_start_loc), _i(sequences), _i(channels),
                                                       _i(taps)))


def gated_recurrence(y_pre: torch.Tensor, x_in: torch.Tensor, u: torch.Tensor, gates: torch.Tensor, block_width: int,
                     rate: torch.Tensor, state: torch.Tensor, past: torch.Tensor, seq_slot: torch.Tensor,
                     q_start_loc: torch.Tensor, sequences: int, taps: int, segments: int = 1) -> torch.Tensor:
    """The gated linear recurrence of ``csrc/recurrent.hip`` over a step's tokens: per channel
    ``a = exp(rate * sigmoid(r))``, ``S = a * S + sqrt(1 - a^2) * sigmoid(i) * u``, ``out = S * gelu_tanh(y_pre)``,
    with r and i from ``gates`` (float32 [T, 2C], per block of ``block_width`` channels its r then its i).  ``state``
    float32 [slots, C]; ``past`` float32 [slots, max(taps - 1, 1), C] is moved on with the step's ``x_in``.
    ``segments`` (1 to 64) stretches of a sequence's tokens run side by side and are joined by the recurrence's
    own linearity (for long portions; the result differs from the walk in order by float32 rounding only)."""
    tokens, channels = u.shape
    for name, t in (("y_pre", y_pre), ("x_in", x_in)):
        if not (t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.dtype == u.dtype and tuple(t.shape) == (tokens, channels)):
            raise ValueError(f"{name} must be a [{tokens}, {channels}] view of u's type with unit inner stride")
    _gpu("u", u, dims=2)
    _gpu("gates", gates, torch.float32, 2)
    _gpu("rate", rate, torch.float32, 1)
    _gpu("state", state, torch.float32, 2)
    _gpu("past", past, torch.float32, 3)
    if (tuple(gates.shape) != (tokens, 2 * channels) or rate.shape[0] != channels or state.shape[1] != channels
            or tuple(past.shape[1:]) != (max(taps - 1, 1), channels) or channels % block_width
            or not 1 <= taps <= MAX_CONV_TAPS or not 1 <= segments <= MAX_SCAN_SEGMENTS):
        raise ValueError("gates, rate, state or past do not fit the channels")
    for name, meta, least in (("seq_slot", seq_slot, sequences), ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {sequences} sequences")
    out = torch.empty((tokens, channels), dtype=u.dtype, device=u.device)
    ld = lambda t: t.stride(0) if tokens > 1 else max(t.stride(0), channels)
    _run("cie_gated_recurrence", load_library().cie_gated_recurrence(
        _stream(), _i(_code(u.dtype)), _ptr(y_pre), ld(y_pre), _ptr(x_in), ld(x_in), _ptr(u), _ptr(gates),
        _i(block_width), _ptr(rate), _ptr(state), _ptr(past), _ptr(seq_slot), _ptr(q_start_loc), _ptr(out),
        _i(sequences), _i(channels), _i(taps), _i(segments)))
    return out


SCAN_CHUNK_WIDTHS = (64, 128, 256)  # of a block
SCAN_CHUNK_TOKENS = 64


def chunks_gated_recurrence(y_pre: torch.Tensor, u: torch.Tensor, weight: torch.Tensor, block_width: int, taps: int) -> bool:
    """Whether :func:`gated_recurrence_chunks` takes these: bfloat16, rows in 16-byte pieces."""
    return (u.dtype == weight.dtype == y_pre.dtype == torch.bfloat16 and block_width in SCAN_CHUNK_WIDTHS and u.shape[0] > 1
            and taps <= MAX_CONV_TAPS and y_pre.stride(0) % 8 == 0
            and u.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0 and y_pre.data_ptr() % 16 == 0)


def gated_recurrence_chunks(y_pre: torch.Tensor, x_in: torch.Tensor, u: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor,
                            rate: torch.Tensor, state: torch.Tensor, past: torch.Tensor, seq_of_token: torch.Tensor,
                            seq_slot: torch.Tensor, q_start_loc: torch.Tensor, sequences: int, taps: int) -> torch.Tensor:
    """``gated_recurrence`` with its gates' product ``block_linear(u, weight, bias)`` in front of it, over the step's flat tokens in
    chunks of ``SCAN_CHUNK_TOKENS`` (the result differs from the walk in order by float32 rounding only)."""
    tokens, channels = u.shape
    for name, t in (("y_pre", y_pre), ("x_in", x_in)):
        if not (t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.dtype == u.dtype and tuple(t.shape) == (tokens, channels)):
            raise ValueError(f"{name} must be a [{tokens}, {channels}] view of u's type with unit inner stride")
    _gpu("u", u, torch.bfloat16, 2)
    _gpu("weight", weight, torch.bfloat16, 3)
    _gpu("bias", bias, torch.bfloat16, 2)
    _gpu("rate", rate, torch.float32, 1)
    _gpu("state", state, torch.float32, 2)
    _gpu("past", past, torch.float32, 3)
    blocks, twice, width = weight.shape
    if (twice != 2 * width or blocks * width != channels or tuple(bias.shape) != (blocks, twice) or rate.shape[0] != channels
            or state.shape[1] != channels or tuple(past.shape[1:]) != (max(taps - 1, 1), channels)
            or past.shape[0] != state.shape[0] or not 1 <= taps <= MAX_CONV_TAPS or width not in SCAN_CHUNK_WIDTHS):
        raise ValueError("weight, bias, rate, state or past do not fit the channels")
    for name, meta, least in (("seq_of_token", seq_of_token, tokens), ("seq_slot", seq_slot, sequences),
                              ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {sequences} sequences of {tokens} tokens")
    out = torch.empty((tokens, channels), dtype=u.dtype, device=u.device)
    planes = torch.empty((2, tokens, channels), dtype=torch.float32, device=u.device)
    carry = torch.empty((-(-tokens // SCAN_CHUNK_TOKENS), 2, channels), dtype=torch.float32, device=u.device)
    ld = lambda t: t.stride(0) if tokens > 1 else max(t.stride(0), channels)
    _run("cie_gated_recurrence_chunks", load_library().cie_gated_recurrence_chunks(
        _stream(), _ptr(y_pre), ld(y_pre), _ptr(x_in), ld(x_in), _ptr(u), _ptr(weight), _ptr(bias), _i(width), _ptr(rate),
        _ptr(state), _ptr(past), _ptr(seq_of_token), _ptr(seq_slot), _ptr(q_start_loc), _ptr(out), _ptr(planes), _ptr(carry),
        _i(sequences), _i(tokens), _i(channels), _i(taps)))
    return out


SCAN_STEP_TAPS = 5         # of a convolution in front of the kernel of single tokens, at most
# ... and workgroups of 16 channels and 16 sequences a compute unit: blocks of up to so many numbers have little K for what a
# fifth costs (us, the two kernels and this one: 20 blocks of 128, 4.4 a unit 11.0, 12.1, 5 11.7, 13.5; 16 blocks of 128, 4 a unit
# 10.8, 10.0, 5 11.4, 12.8; 32 blocks of 64 10.8, 10.0 and 11.9, 13.1; 8 blocks of 256 12.7, 10.1 and 13.5, 13.1, 6 a unit 14.3,
# 14.5; 16 of 160 5 a unit 13.7, 10.6; 4 of 640 21.3, 19.2, 6.3 a unit 22.5, 24.5)
SCAN_STEP_WORKGROUPS, SCAN_STEP_NARROW, SCAN_STEP_WORKGROUPS_NARROW = 5, 128, 4


def steps_gated_recurrence(u: torch.Tensor, weight: torch.Tensor, sequences: int, block_width: int, taps: int) -> bool:
    """Whether the kernel that makes the gates and moves the states of single tokens is the faster one for these and takes
    them: bfloat16, blocks in 16-byte pieces."""
    groups = u.shape[1] // block_width * -(-block_width // 16) * -(-sequences // 16)
    most = SCAN_STEP_WORKGROUPS if block_width > SCAN_STEP_NARROW else SCAN_STEP_WORKGROUPS_NARROW
    return (u.dtype == torch.bfloat16 and weight.dtype == u.dtype and block_width % 8 == 0 and taps <= SCAN_STEP_TAPS
            and groups <= most * compute_units() and u.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)


def gated_recurrence_step(y_pre: torch.Tensor, x_in: torch.Tensor, u: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor,
                          rate: torch.Tensor, state: torch.Tensor, past: torch.Tensor, seq_slot: torch.Tensor,
                          q_start_loc: torch.Tensor, sequences: int, taps: int) -> torch.Tensor:
    """``gated_recurrence`` with its gates' product ``block_linear(u, weight, bias)`` (``weight``
    [blocks, 2 * block_width, block_width]) in one kernel, for a step in which no sequence brings more than one token
    (the caller's to know: of a sequence with more, only the first would be walked)."""
    tokens, channels = u.shape
    for name, t in (("y_pre", y_pre), ("x_in", x_in)):
        if not (t.is_cuda and t.dim() == 2 and t.stride(1) == 1 and t.dtype == u.dtype and tuple(t.shape) == (tokens, channels)):
            raise ValueError(f"{name} must be a [{tokens}, {channels}] view of u's type with unit inner stride")
    _gpu("u", u, torch.bfloat16, 2)
    _gpu("weight", weight, torch.bfloat16, 3)
    _gpu("bias", bias, torch.bfloat16, 2)
    _gpu("rate", rate, torch.float32, 1)
    _gpu("state", state, torch.float32, 2)
    _gpu("past", past, torch.float32, 3)
    blocks, twice, width = weight.shape
    if (twice != 2 * width or blocks * width != channels or tuple(bias.shape) != (blocks, twice) or rate.shape[0] != channels
            or state.shape[1] != channels or tuple(past.shape[1:]) != (max(taps - 1, 1), channels)
            or past.shape[0] != state.shape[0] or not 1 <= taps <= SCAN_STEP_TAPS or width % 8):
        raise ValueError("weight, bias, rate, state or past do not fit the channels")
    for name, meta, least in (("seq_slot", seq_slot, sequences), ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {sequences} sequences")
    out = torch.empty((tokens, channels), dtype=u.dtype, device=u.device)
    ld = lambda t: t.stride(0) if tokens > 1 else max(t.stride(0), channels)
    _run("cie_gated_recurrence_step", load_library().cie_gated_recurrence_step(
        _stream(), _ptr(y_pre), ld(y_pre), _ptr(x_in), ld(x_in), _ptr(u), _ptr(weight), _ptr(bias), _i(width), _ptr(rate),
        _ptr(state), _ptr(past), _ptr(seq_slot), _ptr(q_start_loc), _ptr(out), _i(sequences), _i(tokens), _i(channels),
        _i(taps)))
    return out


# ---------------------------------------------------------------------------
WALK_ROWS = (4, 8, 16, 32, 64)   # rows of a memory that one thread of the walk keeps in registers
WALK_MAX_ROWS = 1024
WALK_LDS_BYTES = 48 * 1024
WALK_AHEAD_FROM = 4              # tokens a sequence (on average) from which the walk fetches a chunk's operands a chunk ahead
WALK_BLOCKS_FROM = 16            # tokens a sequence (on average) from which the first form of the walk goes in blocks
WALK_BLOCKS_MAX_BYTES = 2 << 30  # ... while the blocks' sums fit this much scratch memory


def plan_memory_walk(rows: int, cols: int, time_form: bool, units: int = 1) -> tuple[int, int, int, int]:
    """(rows per thread, row groups, columns per workgroup, tokens staged at once) of ``memory_walk`` for a memory
    of ``rows`` x ``cols`` per head, of which ``units`` (sequences x heads) are walked at once.  Rows per thread and
    row groups follow from ``rows`` alone (they fix the order of the read-out's sums): few rows a thread, so that a
    prompt of one sequence still brings several waves to every compute unit.  The columns are cut into more
    workgroups while these are fewer than the compute units."""
    if not (1 <= rows <= WALK_MAX_ROWS and cols >= 1):
        raise ValueError(f"a memory of {rows} x {cols}: up to {WALK_MAX_ROWS} rows")
    per_thread = next(n for n in WALK_ROWS if 16 * n >= rows)
    groups = -(-rows // per_thread)
    slice_cols = 16
    while slice_cols < min(cols, 64) and 2 * slice_cols * groups <= 512:
        slice_cols *= 2
    while slice_cols > 16 and units * -(-cols // slice_cols) < 2 * compute_units():
        slice_cols //= 2
    per_token = groups * (per_thread + 4)
    floats = (4 if time_form else 2) * per_token + slice_cols + groups * slice_cols
    chunk = max(1, min(16, (WALK_LDS_BYTES - 64) // (4 * floats)))
    # (a thread fetches the next chunk's operands into registers while it walks this one: 8 numbers of each row
    # operand and 4 values a thread)
    threads = -(-slice_cols * groups // 64) * 64
    chunk = max(1, min(chunk, 8 * threads // (groups * per_thread), 4 * threads // slice_cols))
    return per_thread, groups, slice_cols, chunk


def memory_walk(decay: torch.Tensor, in_rows: torch.Tensor, out_rows: torch.Tensor, values: torch.Tensor,
                state: torch.Tensor, seq_slot: torch.Tensor, q_start_loc: torch.Tensor, sequences: int, heads: int,
                rows: int, cols: int, heads_per_group: int = 1, bonus: Optional[torch.Tensor] = None,
                value_scale: Optional[torch.Tensor] = None, skip: Optional[torch.Tensor] = None,
                read_first: bool = False, log_decay: Optional[torch.Tensor] = None,
                blocks: Optional[bool] = None) -> torch.Tensor:
    """The walk of ``csrc/memory_walk.hip`` over a step's tokens: per head a float32 memory ``S`` [rows, cols] in
    ``state`` [slots, heads, rows, cols], ``S <- decay * S + in (x) (value * value_scale)`` token by token, and the
    read-out ``y = S^T out + skip * value`` behind the update, or (``read_first``) ``y = (S + (bonus * in) (x) value)^T
    out`` in front of it.  All operands float32 views with unit inner stride: ``decay`` [T, heads] (one per head and
    token) or [T, heads * rows]; ``in_rows``, ``out_rows`` [T, (heads / heads_per_group) * rows]; ``values``
    [T, heads * cols]; ``bonus`` [heads, rows]; ``value_scale`` [T, heads]; ``skip`` [heads].  Returns y, float32
    [T, heads * cols].  With ``log_decay`` (float32 [T, heads], the decays' logarithms; the first form only) sequences
    that bring ``WALK_BLOCKS_FROM`` tokens and more on average are walked in blocks of 32 tokens on the matrix cores
    (``blocks``: force it or forbid it); the sums come in another order, a difference of float32 rounding."""
    tokens = values.shape[0]
    groups_of_heads = heads // heads_per_group
    if heads % heads_per_group:
        raise ValueError(f"{heads} heads in groups of {heads_per_group}")
    per_row = bool(read_first)  # (the read-out in front of the update comes with a decay per row, the other form with one per head)
    for name, t, width in (("decay", decay, heads * rows if per_row else heads), ("in_rows", in_rows, groups_of_heads * rows),
                           ("out_rows", out_rows, groups_of_heads * rows), ("values", values, heads * cols)):
        if not (t.is_cuda and t.dtype == torch.float32 and t.dim() == 2 and t.stride(1) == 1 and tuple(t.shape) == (tokens, width)):
            raise ValueError(f"{name} must be a float32 GPU view [{tokens}, {width}] with unit inner stride, is {tuple(t.shape)} {t.dtype}")
    _gpu("state", state, torch.float32, 4)
    if tuple(state.shape[1:]) != (heads, rows, cols):
        raise ValueError(f"state {tuple(state.shape)} does not hold {heads} memories of {rows} x {cols}")
    if bonus is not None:
        _gpu("bonus", bonus, torch.float32, 2)
        if tuple(bonus.shape) != (heads, rows) or not read_first:
            raise ValueError("the bonus is [heads, rows] and comes with a read-out in front of the update")
    ld_scale = 0
    if value_scale is not None:
        if not (value_scale.is_cuda and value_scale.dtype == torch.float32 and tuple(value_scale.shape) == (tokens, heads)
                and value_scale.stride(1) == 1):
            raise ValueError(f"value_scale must be float32 [{tokens}, {heads}]")
        ld_scale = value_scale.stride(0)
    if skip is not None:
        _gpu("skip", skip, torch.float32, 1)
        if skip.shape[0] != heads:
            raise ValueError(f"skip must be [{heads}]")
    for name, meta, least in (("seq_slot", seq_slot, sequences), ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {sequences} sequences")
    per_thread, row_groups, slice_cols, chunk = plan_memory_walk(rows, cols, per_row, sequences * heads)
    y = torch.empty((tokens, heads * cols), dtype=torch.float32, device=values.device)
    ld = lambda t: t.stride(0) if tokens > 1 else max(t.stride(0), t.shape[1])
    if blocks is None:
        blocks = tokens >= WALK_BLOCKS_FROM * max(sequences, 1)
    if blocks and log_decay is not None and not read_first and bonus is None and sequences > 0:
        padded, cols16 = -(-rows // 16) * 16, -(-cols // 16) * 16
        panel = min(cols16, 128)
        lds = 4 * (2 * 32 * (padded + 4) + 32 * (panel + 16 if panel % 32 == 0 else panel) + 32 * 36 + 36)
        places = tokens // 32 + sequences + 1
        scratch = places * heads * padded * cols16 * 4
        if lds <= 64 * 1024 and scratch <= WALK_BLOCKS_MAX_BYTES and tokens <= 32 * 65535:
            if not (log_decay.is_cuda and log_decay.dtype == torch.float32 and tuple(log_decay.shape) == (tokens, heads)
                    and log_decay.stride(1) == 1):
                raise ValueError(f"log_decay must be float32 [{tokens}, {heads}]")
            sums = torch.empty(places * heads * padded * cols16, dtype=torch.float32, device=values.device)
            totals = torch.empty(places * heads, dtype=torch.float32, device=values.device)
            _run("cie_memory_walk_blocks", load_library().cie_memory_walk_blocks(
                _stream(), _ptr(log_decay), ld(log_decay), _ptr(in_rows), ld(in_rows), _ptr(out_rows), ld(out_rows),
                _i(heads_per_group), _ptr(values), ld(values), _ptr(value_scale), ld_scale, _ptr(skip), _ptr(state),
                _ptr(seq_slot), _ptr(q_start_loc), _ptr(y), _ptr(sums), _ptr(totals), _i(tokens), _i(sequences), _i(heads),
                _i(rows), _i(cols)))
            return y
    _run("cie_memory_walk", load_library().cie_memory_walk(
        _stream(), _ptr(decay), ld(decay), _ptr(in_rows), ld(in_rows), _ptr(out_rows), ld(out_rows), _i(heads_per_group),
        _ptr(bonus), _ptr(values), ld(values), _ptr(value_scale), ld_scale, _ptr(skip), _ptr(state), _ptr(seq_slot),
        _ptr(q_start_loc), _ptr(y), _i(sequences), _i(heads), _i(rows), _i(cols), _i(per_thread), _i(row_groups),
        _i(slice_cols), _i(chunk), _i(1 if read_first else 0), _i(1 if tokens >= WALK_AHEAD_FROM * max(sequences, 1) else 0)))
    return y


def space_steps(raw: torch.Tensor, bias: torch.Tensor, a_log: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Step sizes and decays of a state-space layer: ``dt = softplus(raw + bias)``, ``exp(-exp(a_log) * dt)`` and the
    decay's logarithm ``-exp(a_log) * dt`` per token and head, all float32 [T, heads].  ``raw`` [T, heads] (a view
    with unit inner stride); bias, a_log float32."""
    if not (raw.is_cuda and raw.dim() == 2 and raw.stride(1) == 1 and raw.dtype in _CODES):
        raise ValueError("raw must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens, heads = raw.shape
    for name, t in (("bias", bias), ("a_log", a_log)):
        _gpu(name, t, torch.float32, 1)
        if t.shape[0] != heads:
            raise ValueError(f"{name} must be [{heads}]")
    made = torch.empty((3, tokens, heads), dtype=torch.float32, device=raw.device)
    ld = raw.stride(0) if tokens > 1 else max(raw.stride(0), heads)
    _run("cie_space_steps", load_library().cie_space_steps(_stream(), _i(_code(raw.dtype)), _ptr(raw), ld, _ptr(bias),
                                                           _ptr(a_log), _ptr(made[0]), _ptr(made[1]), _ptr(made[2]),
                                                           _i(tokens), _i(heads)))
    return made[0], made[1], made[2]


def shift_mix(h: torch.Tensor, before: torch.Tensor, mu: torch.Tensor, seq_of_token: torch.Tensor,
              seq_slot: torch.Tensor, q_start_loc: torch.Tensor) -> torch.Tensor:
    """``mixes[s, t] = h[t] + (h[t - 1] - h[t]) * mu[s]`` within each sequence, [n_mix, T, W] in h's type; the row in
    front of a step's first token comes from ``before`` (float32 [slots, W]; zeros for a new sequence), which
    ``time_decay`` moves on.  ``mu`` float32 [n_mix, W]."""
    if not (h.is_cuda and h.dim() == 2 and h.stride(1) == 1 and h.dtype in _CODES):
        raise ValueError("h must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens, width = h.shape
    _gpu("before", before, torch.float32, 2)
    _gpu("mu", mu, torch.float32, 2)
    if before.shape[1] != width or mu.shape[1] != width:
        raise ValueError(f"before {tuple(before.shape)} / mu {tuple(mu.shape)} do not fit rows of {width}")
    for name, meta in (("seq_of_token", seq_of_token), ("seq_slot", seq_slot), ("q_start_loc", q_start_loc)):
        _gpu(name, meta, torch.int32, 1)
    if seq_of_token.shape[0] < tokens:
        raise ValueError("one sequence index per token")
    mixes = torch.empty((mu.shape[0], tokens, width), dtype=h.dtype, device=h.device)
    ldh = h.stride(0) if tokens > 1 else max(h.stride(0), width)
    _run("cie_shift_mix", load_library().cie_shift_mix(_stream(), _i(_code(h.dtype)), _ptr(h), ldh, _ptr(before), _ptr(mu),
                                                       _ptr(seq_of_token), _ptr(seq_slot), _ptr(q_start_loc), _ptr(mixes),
                                                       _i(tokens), _i(width), _i(mu.shape[0])))
    return mixes


def time_decay(low: torch.Tensor, w2t: torch.Tensor, w0: torch.Tensor, h: torch.Tensor, before: torch.Tensor,
               seq_of_token: torch.Tensor, seq_slot: torch.Tensor, q_start_loc: torch.Tensor) -> torch.Tensor:
    """``exp(-exp(tanh(low) w2t + w0))``, float32 [T, C]: ``low`` float32 [T, rank], ``w2t`` [rank, C] in h's type
    (the second small product's weight, transposed), ``w0`` float32 [C].  Also leaves the last row of ``h`` of every
    sequence of the step in ``before`` (the token-shift state that ``shift_mix`` reads at the next step)."""
    _gpu("low", low, torch.float32, 2)
    tokens, rank = low.shape
    if not (h.is_cuda and h.dim() == 2 and h.stride(1) == 1 and h.dtype in _CODES and h.shape[0] == tokens):
        raise ValueError("h must be a float32 or bfloat16 GPU matrix with unit inner stride, a row per token")
    _gpu("w2t", w2t, h.dtype, 2)
    channels = w2t.shape[1]
    _gpu("w0", w0, torch.float32, 1)
    _gpu("before", before, torch.float32, 2)
    if w2t.shape[0] != rank or w0.shape[0] != channels or before.shape[1] != h.shape[1]:
        raise ValueError(f"w2t {tuple(w2t.shape)}, w0 {tuple(w0.shape)}, before {tuple(before.shape)} do not fit")
    for name, meta in (("seq_of_token", seq_of_token), ("seq_slot", seq_slot), ("q_start_loc", q_start_loc)):
        _gpu(name, meta, torch.int32, 1)
    decay = torch.empty((tokens, channels), dtype=torch.float32, device=low.device)
    ldh = h.stride(0) if tokens > 1 else max(h.stride(0), h.shape[1])
    _run("cie_time_decay", load_library().cie_time_decay(
        _stream(), _i(_code(h.dtype)), _ptr(low), _ptr(w2t), _ptr(w0), _ptr(decay), _i(tokens), _i(channels), _i(rank),
        _ptr(h), ldh, _ptr(before), _ptr(seq_of_token), _ptr(seq_slot), _ptr(q_start_loc), _i(h.shape[1])))
    return decay


def gated_group_norm(y: torch.Tensor, gate: Optional[torch.Tensor], weight: Optional[torch.Tensor], groups: int,
                     eps: float, out_dtype: torch.dtype, gate_first: bool) -> torch.Tensor:
    """The RMS norm of float32 rows ``y`` [T, W] in ``groups`` equal consecutive parts (each over its own root mean
    square), times ``weight`` (float32 [W], or one group's numbers for all groups alike), with ``silu(gate)`` multiplied in front of the norm (``gate_first``) or
    behind it.  ``gate`` [T, W] in ``out_dtype`` (a view with unit inner stride)."""
    _gpu("y", y, torch.float32, 2)
    tokens, width = y.shape
    if groups < 1 or width % groups or not eps > 0 or width + groups > MAX_NORM_WIDTH:
        raise ValueError(f"{groups} groups over rows of {width} with eps {eps}")
    ldg = 0
    if gate is not None:
        if not (gate.is_cuda and gate.dim() == 2 and gate.stride(1) == 1 and gate.dtype == out_dtype
                and tuple(gate.shape) == (tokens, width)):
            raise ValueError(f"gate must be a [{tokens}, {width}] view of {out_dtype} with unit inner stride")
        ldg = gate.stride(0) if tokens > 1 else max(gate.stride(0), width)
    weight_width = 0
    if weight is not None:
        _gpu("weight", weight, torch.float32, 1)
        weight_width = weight.shape[0]
        if weight_width not in (width, width // groups):
            raise ValueError(f"weight must be [{width}], or [{width // groups}] for every group alike")
    out = torch.empty((tokens, width), dtype=out_dtype, device=y.device)
    _run("cie_gated_group_norm", load_library().cie_gated_group_norm(
        _stream(), _i(_code(out_dtype)), _ptr(y), _ptr(gate), ldg, _ptr(weight), _i(weight_width), _ptr(out), _i(tokens),
        _i(width), _i(groups), _f(eps), _i(1 if gate_first else 0)))
    return out


# ---------------------------------------------------------------------------
def branch_norm_add(residual: torch.Tensor, branch: Optional[torch.Tensor], weight: torch.Tensor, eps: float,
                    out_dtype: torch.dtype, parts: Optional[torch.Tensor] = None, want_rows: bool = True,
                    branch_gate: Optional[torch.Tensor] = None, part_weight: Optional[torch.Tensor] = None,
                    branch2: Optional[torch.Tensor] = None, scales: tuple[float, float] = (1.0, 1.0),
                    next_weight: Optional[torch.Tensor] = None):
    """``residual += y / sqrt(mean(y^2) + eps) * weight`` with ``y = scales[0] * branch * sigmoid(branch_gate) +
    scales[1] * branch2 + sum_p part_weight[:, p] * parts[:, p]`` (whatever of it is given), row by row, in float32
    and in place.  ``branch``, ``branch2`` [T, H] float32 or ``out_dtype``; ``branch_gate`` float32 [T] (logits, any
    stride); ``parts`` float32 [T, P, H]; ``part_weight`` float32 [T, P]; ``weight`` float32 [H] as it multiplies.
    Returns the new stream rounded to ``out_dtype`` (``want_rows``), which is what a sublayer that reads the stream
    itself takes; with ``next_weight`` (float32 [H]) a pair of that and the RMS norm of the new stream under that
    weight, in ``out_dtype``."""
    _gpu("residual", residual, torch.float32, 2)
    tokens, hidden = residual.shape
    _gpu("weight", weight, torch.float32, 1)
    if not (weight.shape[0] == hidden and hidden <= MAX_NORM_WIDTH and eps > 0):
        raise ValueError(f"weight {tuple(weight.shape)}, hidden {hidden}, eps {eps} do not fit the norm kernel")
    if branch is None and parts is None and branch2 is None:
        raise ValueError("nothing to add")
    kinds = set()
    for name, t in (("branch", branch), ("branch2", branch2)):
        if t is not None:
            _gpu(name, t, dims=2)
            if not (t.shape == residual.shape and t.dtype in (torch.float32, out_dtype)):
                raise ValueError(f"{name} {tuple(t.shape)} {t.dtype} does not fit {tuple(residual.shape)} {out_dtype}")
            kinds.add(t.dtype)
    if len(kinds) > 1:
        raise ValueError("the two branches must be of one type")
    gate_stride = 1
    if branch_gate is not None:
        if not (branch_gate.is_cuda and branch_gate.dtype == torch.float32 and branch_gate.dim() == 1):
            raise ValueError("branch_gate must be a float32 GPU vector")
        if branch is None or branch_gate.shape[0] != tokens:
            raise ValueError("a gate comes with a branch, one logit per row")
        gate_stride = max(branch_gate.stride(0), 1)
    n_parts = 0
    if parts is not None:
        _gpu("parts", parts, torch.float32, 3)
        if not (parts.shape[0] == tokens and parts.shape[2] == hidden):
            raise ValueError(f"parts {tuple(parts.shape)} do not fit {tuple(residual.shape)}")
        n_parts = parts.shape[1]
    if part_weight is not None:
        _gpu("part_weight", part_weight, torch.float32)
        if parts is None or part_weight.numel() != tokens * n_parts:
            raise ValueError("part weights come with parts, one per part and row")
    normed = None
    if next_weight is not None:
        _gpu("next_weight", next_weight, torch.float32, 1)
        if next_weight.shape[0] != hidden:
            raise ValueError(f"next_weight must be [{hidden}]")
        normed = torch.empty((tokens, hidden), dtype=out_dtype, device=residual.device)
    rows = torch.empty((tokens, hidden), dtype=out_dtype, device=residual.device) if want_rows else None
    kind = kinds.pop() if kinds else torch.float32
    _run("cie_branch_norm_add", load_library().cie_branch_norm_add(
        _stream(), _i(_code(kind)), _i(_code(out_dtype)), _ptr(residual), _ptr(branch), _ptr(branch_gate),
        _i(gate_stride), _ptr(branch2), _f(scales[0]), _f(scales[1]), _ptr(parts), _ptr(part_weight), _i(n_parts),
        _ptr(weight), _ptr(rows), _i(tokens), _i(hidden), _f(eps), _ptr(next_weight), _ptr(normed)))
    return rows if next_weight is None else (rows, normed)


def group_norm_add(residual: torch.Tensor, branch: Optional[torch.Tensor], weight: torch.Tensor, groups: int, eps: float,
                   out_dtype: torch.dtype, rows: Optional[torch.Tensor] = None, branch_gate: Optional[torch.Tensor] = None,
                   parts: Optional[torch.Tensor] = None, part_weight: Optional[torch.Tensor] = None,
                   plus: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``residual += branch * sigmoid(branch_gate) + sum_p part_weight[:, p] * parts[:, p] + plus`` (whatever of it
    is given; float32, in place unless ``rows``), then the RMS norm of every row in ``groups`` equal consecutive
    parts, each over its own root mean square, the whole times ``weight`` (float32 [H]).  ``branch`` [T, H] float32
    or ``out_dtype``; ``branch_gate`` float32 [T] (logits; any stride); ``parts`` float32 [T, P, H]; ``part_weight`` float32
    [T, P]; ``plus`` float32 [T, H].  With ``rows`` (int32 [n]) only those rows come back, in that order."""
    _gpu("residual", residual, torch.float32, 2)
    tokens, hidden = residual.shape
    _gpu("weight", weight, torch.float32, 1)
    if not (weight.shape[0] == hidden and hidden + groups <= MAX_NORM_WIDTH and eps > 0):
        raise ValueError(f"weight {tuple(weight.shape)}, hidden {hidden}, eps {eps} do not fit the norm kernel")
    if groups < 1 or hidden % groups:
        raise ValueError(f"{groups} groups do not divide a row of {hidden}")
    if branch is not None:
        _gpu("branch", branch, dims=2)
        if not (branch.shape == residual.shape and branch.dtype in (torch.float32, out_dtype)):
            raise ValueError(f"branch {tuple(branch.shape)} {branch.dtype} does not fit {tuple(residual.shape)} {out_dtype}")
    gate_stride = 1
    if branch_gate is not None:
        # (one logit per row; the rows may lie apart, as the first column of a wider product's result does)
        if not (branch_gate.is_cuda and branch_gate.dtype == torch.float32 and branch_gate.dim() == 1):
            raise ValueError("branch_gate must be a float32 GPU vector")
        if branch is None or branch_gate.shape[0] != tokens:
            raise ValueError("a gate comes with a branch, one logit per row")
        gate_stride = max(branch_gate.stride(0), 1)
    n_parts = 0
    if parts is not None:
        _gpu("parts", parts, torch.float32, 3)
        if not (parts.shape[0] == tokens and parts.shape[2] == hidden):
            raise ValueError(f"parts {tuple(parts.shape)} do not fit {tuple(residual.shape)}")
        n_parts = parts.shape[1]
    if part_weight is not None:
        _gpu("part_weight", part_weight, torch.float32)
        if parts is None or part_weight.numel() != tokens * n_parts:
            raise ValueError("part weights come with parts, one per part and row")
    if plus is not None:
        _gpu("plus", plus, torch.float32, 2)
        if plus.shape != residual.shape:
            raise ValueError(f"plus {tuple(plus.shape)} vs residual {tuple(residual.shape)}")
    n_out = tokens
    if rows is not None:
        _gpu("rows", rows, torch.int32, 1)
        n_out = rows.shape[0]
    out = torch.empty((n_out, hidden), dtype=out_dtype, device=residual.device)
    _run("cie_group_norm_add", load_library().cie_group_norm_add(
        _stream(), _i(_code(branch.dtype if branch is not None else out_dtype)), _i(_code(out_dtype)), _ptr(residual),
        _ptr(branch), _ptr(branch_gate), _i(gate_stride), _ptr(parts), _ptr(part_weight), _i(n_parts), _ptr(plus), _ptr(weight),
        _ptr(out), _ptr(rows), _i(n_out), _i(hidden), _i(groups), _f(eps)))
    return out


# ---------------------------------------------------------------------------
DELTA_ROWS = (4, 8, 16, 32)       # rows of a column that one of its 16 lanes keeps in registers
DELTA_COLUMNS = (1, 2, 4, 8)      # columns a thread takes
DELTA_STATE_NUMBERS = 128         # numbers of the memory a thread keeps at most (64 with 32 rows)
DELTA_LDS_BYTES = 40 * 1024
DELTA_MAX_TAPS = 64
DELTA_BLOCKS_FROM = 16            # tokens a sequence (on average) from which the memory is walked in blocks of 32 tokens
DELTA_BLOCKS_MAX_DIM = 256        # ... for keys of up to this many numbers
DELTA_BLOCKS_MAX_BYTES = 2 << 30  # ... while the blocks' scratch memory is no larger


def plan_delta_walk(dim: int, vdim: int) -> tuple[int, int, int, int, int]:
    """(rows a thread, columns a thread, threads, columns a workgroup, tokens staged at once) of the token-by-token form
    for memories of ``dim`` x ``vdim``: all columns of a head in one workgroup where its registers hold them (the read-out's
    norm and gate then ride along), else slices."""
    if not (1 <= dim <= 512 and vdim >= 1):
        raise ValueError(f"a memory of {dim} x {vdim}: keys of up to 512 numbers")
    rows = next(r for r in DELTA_ROWS if 16 * r >= dim)
    most = 2 if rows == 32 else 8
    columns = next((c for c in DELTA_COLUMNS if c <= most and 32 * c >= vdim), most)
    slice_cols = min(vdim, 32 * columns)
    threads = -(-16 * -(-slice_cols // columns) // 64) * 64
    chunk = max(1, min(16, DELTA_LDS_BYTES // (4 * (32 * rows + 2 * slice_cols + 3))))
    return rows, columns, threads, slice_cols, chunk


def delta_rule(proj: torch.Tensor, offsets: tuple[int, int, int, int, int, int], taps_w: torch.Tensor, a_log: torch.Tensor,
               dt_bias: torch.Tensor, q_scale: float, norm_weight: torch.Tensor, eps: float, state: torch.Tensor,
               past: torch.Tensor, seq_of_token: torch.Tensor, seq_slot: torch.Tensor, q_start_loc: torch.Tensor,
               sequences: int, heads: int, kv_heads: int, dim: int, vdim: int, blocks: Optional[bool] = None) -> torch.Tensor:
    """The gated delta rule over a step's tokens (``csrc/delta_rule.hip``).  ``proj`` [T, ...] holds each token's queries
    and keys (kv_heads x dim), values and gates (heads x vdim), step-size and decay logits (heads) from the columns
    ``offsets`` on; ``taps_w`` [2 kv_heads dim + heads vdim, taps] in proj's type; ``a_log``, ``dt_bias`` float32 [heads];
    ``norm_weight`` float32 [vdim].  ``state`` float32 [slots, heads, vdim, dim] and ``past`` float32 [slots, heads,
    max(taps - 1, 1), 2 dim + vdim] are read and moved on at the sequences' slots.  Steps of ``DELTA_BLOCKS_FROM`` tokens a
    sequence and more go in blocks of 32 tokens on the matrix cores (``blocks``: force it or forbid it): the same sums in
    another order.  Returns the normed, gated read-out [T, heads * vdim] in proj's type."""
    if not (proj.is_cuda and proj.dim() == 2 and proj.stride(1) == 1 and proj.dtype in _CODES):
        raise ValueError("proj must be a float32 or bfloat16 GPU matrix with unit inner stride")
    tokens = proj.shape[0]
    if heads < 1 or kv_heads < 1 or heads % kv_heads:
        raise ValueError(f"{heads} heads are no multiple of {kv_heads} key heads")
    sizes = (kv_heads * dim, kv_heads * dim, heads * vdim, heads * vdim, heads, heads)
    if min(offsets) < 0 or max(o + n for o, n in zip(offsets, sizes)) > proj.shape[1]:
        raise ValueError(f"proj {tuple(proj.shape)} does not hold the parts at {offsets}")
    _gpu("taps_w", taps_w, proj.dtype, 2)
    channels, taps = taps_w.shape
    if channels != 2 * kv_heads * dim + heads * vdim or not 1 <= taps <= DELTA_MAX_TAPS:
        raise ValueError(f"taps {tuple(taps_w.shape)} for {2 * kv_heads * dim + heads * vdim} channels (up to {DELTA_MAX_TAPS} taps)")
    for name, t, size in (("a_log", a_log, heads), ("dt_bias", dt_bias, heads), ("norm_weight", norm_weight, vdim)):
        _gpu(name, t, torch.float32, 1)
        if t.shape[0] != size:
            raise ValueError(f"{name} must be [{size}], is {tuple(t.shape)}")
    _gpu("state", state, torch.float32, 4)
    _gpu("past", past, torch.float32, 4)
    if (tuple(state.shape[1:]) != (heads, vdim, dim) or tuple(past.shape[1:]) != (heads, max(taps - 1, 1), 2 * dim + vdim)
            or not eps > 0):
        raise ValueError(f"state {tuple(state.shape)} / past {tuple(past.shape)} do not fit {heads} heads of {dim} x {vdim}")
    for name, meta, least in (("seq_slot", seq_slot, sequences), ("seq_of_token", seq_of_token, tokens),
                              ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries, {least} are needed")
    f32 = dict(dtype=torch.float32, device=proj.device)
    common = (_stream(), _i(_code(proj.dtype)), _ptr(proj), _ld(proj), *(_i(o) for o in offsets), _ptr(taps_w), _i(taps),
              _ptr(a_log), _ptr(dt_bias), _f(q_scale))
    lib = load_library()
    padded, cols16 = -(-dim // 16) * 16, -(-vdim // 16) * 16
    wide = -(-dim // 64) * 64
    places = tokens // 32 + sequences + 1
    per_block = heads * 32 * (wide + cols16 + 34) + kv_heads * 64 * wide
    if blocks is None:
        blocks = tokens >= DELTA_BLOCKS_FROM * max(sequences, 1)
    if blocks and dim <= DELTA_BLOCKS_MAX_DIM and 4 * places * per_block <= DELTA_BLOCKS_MAX_BYTES:
        y = torch.empty((tokens, heads * vdim), **f32)
        rows = torch.empty((tokens, 2 * kv_heads * padded), **f32)
        values = torch.empty((tokens, heads * vdim), **f32)
        steps = torch.empty((2, tokens, heads), **f32)
        scratch = torch.empty(places * per_block, **f32)
        _run("cie_delta_blocks", lib.cie_delta_blocks(
            *common, _ptr(state), _ptr(past), _ptr(seq_of_token), _ptr(seq_slot), _ptr(q_start_loc), _ptr(y), _ptr(rows),
            _ptr(values), _ptr(steps), _ptr(scratch), _i(tokens), _i(sequences), _i(heads), _i(kv_heads), _i(dim), _i(vdim)))
    else:
        per_thread, columns, threads, slice_cols, chunk = plan_delta_walk(dim, vdim)
        whole = slice_cols >= vdim
        out = torch.empty((tokens, heads * vdim), dtype=proj.dtype, device=proj.device) if whole else None
        y = None if whole else torch.empty((tokens, heads * vdim), **f32)
        _run("cie_delta_walk", lib.cie_delta_walk(
            *common, _ptr(norm_weight), _f(eps), _ptr(state), _ptr(past), _ptr(seq_slot), _ptr(q_start_loc), _ptr(out), _ptr(y),
            _i(sequences), _i(heads), _i(kv_heads), _i(dim), _i(vdim), _i(per_thread), _i(columns), _i(threads), _i(slice_cols),
            _i(chunk)))
        if whole:
            return out
    gate = proj[:, offsets[3]: offsets[3] + heads * vdim]
    return gated_group_norm(y, gate, norm_weight, heads, eps, proj.dtype, gate_first=False)


# ---------------------------------------------------------------------------
def layer_norm_add(residual: torch.Tensor, branch: Optional[torch.Tensor], weight: torch.Tensor, bias: torch.Tensor, eps: float,
                   out_dtype: torch.dtype, rows: Optional[torch.Tensor] = None,
                   plus: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``residual += branch + plus`` (whatever of it is given; float32, in place unless ``rows``), then the layer norm of
    every row under ``weight`` and ``bias`` (float32 [H]).  ``branch`` [T, H] float32 or ``out_dtype``; ``plus`` float32
    [T, H], or [H] for every row alike.  With ``rows`` (int32 [n]) only those rows come back, in that order."""
    _gpu("residual", residual, torch.float32, 2)
    tokens, hidden = residual.shape
    for name, t in (("weight", weight), ("bias", bias)):
        _gpu(name, t, torch.float32, 1)
        if t.shape[0] != hidden:
            raise ValueError(f"{name} must be [{hidden}], is {tuple(t.shape)}")
    if not (hidden <= MAX_NORM_WIDTH and eps > 0):
        raise ValueError(f"rows of {hidden} numbers with eps {eps} do not fit the norm kernel")
    if branch is not None:
        _gpu("branch", branch, dims=2)
        if not (branch.shape == residual.shape and branch.dtype in (torch.float32, out_dtype)):
            raise ValueError(f"branch {tuple(branch.shape)} {branch.dtype} does not fit {tuple(residual.shape)} {out_dtype}")
    plus_stride = 0
    if plus is not None:
        _gpu("plus", plus, torch.float32)
        if plus.shape != residual.shape and tuple(plus.shape) != (hidden,):
            raise ValueError(f"plus {tuple(plus.shape)} vs residual {tuple(residual.shape)}")
        plus_stride = hidden if plus.dim() == 2 else 0
    n_out = tokens
    if rows is not None:
        _gpu("rows", rows, torch.int32, 1)
        n_out = rows.shape[0]
    out = torch.empty((n_out, hidden), dtype=out_dtype, device=residual.device)
    _run("cie_layer_norm_add", load_library().cie_layer_norm_add(
        _stream(), _i(_code(branch.dtype if branch is not None else out_dtype)), _i(_code(out_dtype)), _ptr(residual),
        _ptr(branch), _ptr(plus), plus_stride, _ptr(weight), _ptr(bias), _ptr(out), _ptr(rows), _i(n_out), _i(hidden), _f(eps)))
    return out


def branch_layer_norm_add(residual: torch.Tensor, branch: Optional[torch.Tensor], weight: torch.Tensor, bias: torch.Tensor,
                          eps: float, out_dtype: torch.dtype, parts: Optional[torch.Tensor] = None,
                          branch_gate: Optional[torch.Tensor] = None, part_weight: Optional[torch.Tensor] = None,
                          branch2: Optional[torch.Tensor] = None, scales: tuple[float, float] = (1.0, 1.0),
                          next_norm: Optional[tuple] = None, rows_out: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``residual += layer norm of y`` under ``weight`` and ``bias``, with ``y`` as in :func:`branch_norm_add`, row by row,
    in float32 and in place.  ``next_norm = (weight, bias)``: the layer norm of the new stream under those comes back in
    ``out_dtype``.  ``rows_out`` ([T, H] in ``out_dtype``; its rows may lie apart) takes the new stream itself."""
    _gpu("residual", residual, torch.float32, 2)
    tokens, hidden = residual.shape
    vectors = [("weight", weight), ("bias", bias)]
    if next_norm is not None:
        vectors += [("the next norm's weight", next_norm[0]), ("the next norm's bias", next_norm[1])]
    for name, t in vectors:
        _gpu(name, t, torch.float32, 1)
        if t.shape[0] != hidden:
            raise ValueError(f"{name} must be [{hidden}], is {tuple(t.shape)}")
    if not (hidden <= MAX_NORM_WIDTH and eps > 0):
        raise ValueError(f"rows of {hidden} numbers with eps {eps} do not fit the norm kernel")
    if branch is None and parts is None and branch2 is None:
        raise ValueError("nothing to add")
    kinds = set()
    for name, t in (("branch", branch), ("branch2", branch2)):
        if t is not None:
            _gpu(name, t, dims=2)
            if not (t.shape == residual.shape and t.dtype in (torch.float32, out_dtype)):
                raise ValueError(f"{name} {tuple(t.shape)} {t.dtype} does not fit {tuple(residual.shape)} {out_dtype}")
            kinds.add(t.dtype)
    if len(kinds) > 1:
        raise ValueError("the two branches must be of one type")
    gate_stride = 1
    if branch_gate is not None:
        if not (branch_gate.is_cuda and branch_gate.dtype == torch.float32 and branch_gate.dim() == 1):
            raise ValueError("branch_gate must be a float32 GPU vector")
        if branch is None or branch_gate.shape[0] != tokens:
            raise ValueError("a gate comes with a branch, one logit per row")
        gate_stride = max(branch_gate.stride(0), 1)
    n_parts = 0
    if parts is not None:
        _gpu("parts", parts, torch.float32, 3)
        if not (parts.shape[0] == tokens and parts.shape[2] == hidden):
            raise ValueError(f"parts {tuple(parts.shape)} do not fit {tuple(residual.shape)}")
        n_parts = parts.shape[1]
    if part_weight is not None:
        _gpu("part_weight", part_weight, torch.float32)
        if parts is None or part_weight.numel() != tokens * n_parts:
            raise ValueError("part weights come with parts, one per part and row")
    if rows_out is not None:
        _row_view("rows_out", rows_out, (tokens, hidden), (out_dtype,))
    normed = torch.empty((tokens, hidden), dtype=out_dtype, device=residual.device) if next_norm is not None else None
    kind = kinds.pop() if kinds else torch.float32
    _run("cie_branch_layer_norm_add", load_library().cie_branch_layer_norm_add(
        _stream(), _i(_code(kind)), _i(_code(out_dtype)), _ptr(residual), _ptr(branch), _ptr(branch_gate), _i(gate_stride),
        _ptr(branch2), _f(scales[0]), _f(scales[1]), _ptr(parts), _ptr(part_weight), _i(n_parts), _ptr(weight), _ptr(bias),
        _ptr(rows_out), _ld(rows_out) if rows_out is not None else 0, _i(tokens), _i(hidden), _f(eps),
        _ptr(next_norm[0] if next_norm is not None else None), _ptr(next_norm[1] if next_norm is not None else None),
        _ptr(normed)))
    return normed


def clamped_glu(gate_up: torch.Tensor, limit: float, alpha: float, offset: float, cubic: float = 0.0) -> torch.Tensor:
    """``g * sigmoid(alpha * (g + cubic * g^3)) * (u + offset)`` with ``g = min(gate, limit)``,
    ``u = clamp(up, -limit, limit)`` for gate_up [T, 2I] (gate half first).  ``cubic = 0`` is the plain sigmoid
    gate; ``alpha = 2 sqrt(2 / pi)`` with ``cubic = 0.044715`` is the tanh form of gelu."""
    _gpu("gate_up", gate_up, dims=2)
    tokens, twice = gate_up.shape
    if twice % 2 or not limit > 0:
        raise ValueError(f"gate_up rows must be even and the limit positive, got {twice}, {limit}")
    out = torch.empty((tokens, twice // 2), dtype=gate_up.dtype, device=gate_up.device)
    _run("cie_clamped_glu", load_library().cie_clamped_glu(_stream(), _i(_code(gate_up.dtype)), _ptr(gate_up), _ptr(out),
                                                           _i(tokens), _i(twice // 2), _f(limit), _f(alpha), _f(offset),
                                                           _f(cubic)))
    return out


def squared_relu(x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``max(x, 0)^2`` of a matrix [T, n] into ``out`` (the rows of either may lie apart; a new tensor if none is given)."""
    _row_view("x", x, tuple(x.shape), tuple(_CODES))
    if out is None:
        out = torch.empty(tuple(x.shape), dtype=x.dtype, device=x.device)
    _row_view("out", out, tuple(x.shape), (x.dtype,))
    tokens, columns = x.shape
    _run("cie_squared_relu", load_library().cie_squared_relu(_stream(), _i(_code(x.dtype)), _ptr(x), _ld(x), _ptr(out), _ld(out),
                                                             _i(tokens), _i(columns)))
    return out


def gated_token_rows(z: torch.Tensor, table: torch.Tensor, column: int, ids: torch.Tensor) -> torch.Tensor:
    """``gelu_tanh(z[t]) * table[ids[t], column : column + dim]`` for ``z`` float32 [T, dim], in the table's dtype."""
    _gpu("z", z, torch.float32, 2)
    _gpu("table", table, dims=2)
    _gpu("ids", ids, torch.int32, 1)
    tokens, dim = z.shape
    vocab, width = table.shape
    if column < 0 or column + dim > width or ids.shape[0] < tokens:
        raise ValueError(f"columns {column} .. {column + dim} of a table of {width}, {ids.shape[0]} ids for {tokens} rows")
    out = torch.empty((tokens, dim), dtype=table.dtype, device=z.device)
    _run("cie_gated_token_rows", load_library().cie_gated_token_rows(
        _stream(), _i(_code(table.dtype)), _ptr(z), _ptr(table), width, _i(column), _ptr(ids), _ptr(out), _i(tokens), _i(dim),
        _i(vocab)))
    return out


def _token_table(table: torch.Tensor, column: int, dim: int, ids: torch.Tensor, tokens: int, dtype: torch.dtype) -> None:
    _gpu("table", table, dtype, 2)
    _gpu("ids", ids, torch.int32, 1)
    if column < 0 or column + dim > table.shape[1] or ids.shape[0] < tokens:
        raise ValueError(f"columns {column} .. {column + dim} of a table of {table.shape[1]}, {ids.shape[0]} ids for {tokens} rows")


def weight_pieces(weight: torch.Tensor) -> torch.Tensor:
    """A weight [N, K] as the kernels of the token table's branch read it: pieces of 16 rows and 32 columns (zeros past either
    end), each as the 64 lanes of a matrix product hold it, [ceil(N / 16), ceil(K / 32), 64, 8]."""
    n, k = weight.shape
    wide = weight.new_zeros((-(-n // 16) * 16, -(-k // 32) * 32))
    wide[:n, :k] = weight
    return (wide.reshape(wide.shape[0] // 16, 16, wide.shape[1] // 32, 4, 8).permute(0, 2, 3, 1, 4)
            .reshape(wide.shape[0] // 16, wide.shape[1] // 32, 64, 8).contiguous())


def _check_pieces(name: str, pieces: torch.Tensor, n: int, k: int) -> None:
    _gpu(name, pieces, torch.bfloat16, 4)
    if tuple(pieces.shape) != (-(-n // 16), -(-k // 32), 64, 8) or pieces.data_ptr() % 16:
        raise ValueError(f"{name} {tuple(pieces.shape)} are not the pieces of a [{n}, {k}] weight")


def token_gate(stream: torch.Tensor, gate: torch.Tensor, dim: int, table: torch.Tensor, column: int,
               ids: torch.Tensor) -> torch.Tensor:
    """``gelu_tanh(stream @ W_gate.T) * table[ids, column : column + dim]`` in one kernel for few rows: ``stream`` float32
    [T, hidden] (rounded to bf16 on its way into the product), ``gate`` the pieces (:func:`weight_pieces`) of the bf16 weight
    [dim, hidden], hidden a multiple of 8."""
    _gpu("stream", stream, torch.float32, 2)
    tokens, hidden = stream.shape
    _check_pieces("gate", gate, dim, hidden)
    if hidden % 8 or stream.data_ptr() % 16:
        raise ValueError(f"rows of {hidden} numbers: a multiple of 8")
    _token_table(table, column, dim, ids, tokens, torch.bfloat16)
    out = torch.empty((tokens, dim), dtype=torch.bfloat16, device=stream.device)
    _run("cie_token_gate", load_library().cie_token_gate(
        _stream(), _ptr(stream), _ptr(gate), _ptr(table), table.shape[1], _i(column), _ptr(ids), _ptr(out), _i(tokens), _i(hidden),
        _i(dim), _i(table.shape[0])))
    return out


def plan_token_side(hidden: int, dim: int) -> int:
    """Shares of the width that :func:`token_side` cuts its first product into; 0: sizes that it does not take."""
    if hidden % 8 or not 8 <= hidden <= 4096 or dim < 1:
        return 0
    tiles, shares = -(-dim // 16), 1
    while tiles * shares * 2 <= 16:
        shares *= 2
    bytes_ = 16 * (-(-hidden // 32) * 32 + 8) * 2 + shares * 16 * tiles * 16 * 4 + 16 * (-(-dim // 32) * 32 + 8) * 2
    return shares if bytes_ <= 160 * 1024 else 0


def token_side(stream: torch.Tensor, branch: Optional[torch.Tensor], gate: torch.Tensor, proj: torch.Tensor, dim: int,
               table: torch.Tensor, column: int, ids: torch.Tensor, weight: torch.Tensor, eps: float,
               next_weight: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``x = stream + branch``; ``g = gelu_tanh(x @ W_gate.T) * table[ids, column : column + dim]``; ``y = g @ W_proj.T``;
    ``stream <- x + y / sqrt(mean(y^2) + eps) * weight``, in one kernel for many rows (sizes that :func:`plan_token_side`
    takes): ``stream`` float32 [T, hidden] in place, ``branch`` bf16 or ``None``, ``gate`` and ``proj`` the pieces
    (:func:`weight_pieces`) of the bf16 weights [dim, hidden] and [hidden, dim].  With ``next_weight`` (float32 [hidden]) the
    RMS norm of the new stream under it comes back in bf16."""
    _gpu("stream", stream, torch.float32, 2)
    tokens, hidden = stream.shape
    shares = plan_token_side(hidden, dim)
    if not shares or not eps > 0:
        raise ValueError(f"rows of {hidden} with {dim} columns of the table (eps {eps}) are not what this kernel takes")
    _check_pieces("gate", gate, dim, hidden)
    _check_pieces("proj", proj, hidden, dim)
    if stream.data_ptr() % 16:
        raise ValueError("operands must be 16-byte aligned")
    if branch is not None:
        _gpu("branch", branch, torch.bfloat16, 2)
        if branch.shape != stream.shape or branch.data_ptr() % 16:
            raise ValueError(f"branch {tuple(branch.shape)} vs stream {tuple(stream.shape)}")
    for name, w in (("weight", weight), ("next_weight", next_weight)):
        if w is not None:
            _gpu(name, w, torch.float32, 1)
            if w.shape[0] != hidden or w.data_ptr() % 16:
                raise ValueError(f"{name} must be [{hidden}], is {tuple(w.shape)}")
    _token_table(table, column, dim, ids, tokens, torch.bfloat16)
    normed = torch.empty((tokens, hidden), dtype=torch.bfloat16, device=stream.device) if next_weight is not None else None
    _run("cie_token_side", load_library().cie_token_side(
        _stream(), _ptr(stream), _ptr(branch), _ptr(gate), _ptr(proj), _ptr(table), table.shape[1], _i(column), _ptr(ids),
        _ptr(weight), _ptr(next_weight), _ptr(normed), _i(tokens), _i(hidden), _i(dim), _i(table.shape[0]), _f(eps), _i(shares)))
    return normed


def stream_rows(residual: torch.Tensor, branch: Optional[torch.Tensor], branch2: Optional[torch.Tensor],
                out_dtype: torch.dtype, want_rows: bool = True) -> Optional[torch.Tensor]:
    """``residual += branch + branch2`` (whichever are given; float32, in place), and the new stream in ``out_dtype``."""
    _gpu("residual", residual, torch.float32, 2)
    tokens, hidden = residual.shape
    if branch is None:
        branch, branch2 = branch2, None
    for name, t in (("branch", branch), ("branch2", branch2)):
        if t is not None:
            _gpu(name, t, dims=2)
            if not (t.shape == residual.shape and t.dtype in (torch.float32, out_dtype) and t.dtype == branch.dtype):
                raise ValueError(f"{name} {tuple(t.shape)} {t.dtype} does not fit {tuple(residual.shape)} {out_dtype}")
    rows = torch.empty((tokens, hidden), dtype=out_dtype, device=residual.device) if want_rows else None
    if branch is None and rows is None:
        return None
    _run("cie_stream_rows", load_library().cie_stream_rows(
        _stream(), _i(_code(branch.dtype if branch is not None else out_dtype)), _i(_code(out_dtype)), _ptr(residual),
        _ptr(branch), _ptr(branch2), _ptr(rows), _i(tokens), _i(hidden)))
    return rows


def soft_cap_(x: torch.Tensor, cap: float) -> torch.Tensor:
    """``x <- cap * tanh(x / cap)`` in place on a float32 tensor."""
    _gpu("x", x, torch.float32)
    if not cap > 0:
        raise ValueError(f"the cap must be positive, got {cap}")
    _run("cie_soft_cap", load_library().cie_soft_cap(_stream(), _ptr(x), _i(x.numel()), _f(cap)))
    return x


# ---------------------------------------------------------------------------
MAX_GENERIC_VALUE = 1024   # numbers of a value head in the generic attention
NORM_MODES = {None: 0, "unit": 1, "weight": 2, "whole": 3}
SCORED_MFMA_DIMS = ((64, 64), (128, 128), (64, 128), (128, 64))  # (key, value) head sizes of the matrix-core form
# ... those of heads with two maps: (a map's numbers, value numbers) -> the most tiles of 16 rows a workgroup takes ...
DIFFERENTIAL_MFMA_DIMS = {(32, 64): 4, (32, 128): 4, (64, 64): 4, (64, 128): 4, (64, 256): 2, (128, 128): 2, (128, 256): 2}
# ... and those of cache entries whose value is a part of the key: (entry, value) -> the most tiles of 16 rows
LATENT_MFMA_DIMS = {(64, 64): 4, (96, 64): 4, (128, 96): 4, (128, 128): 4, (160, 128): 2, (192, 160): 2, (256, 192): 2,
                    (320, 256): 2}


def _check_kv_pools(k_pool: torch.Tensor, v_pool: torch.Tensor, dtype: torch.dtype, kv_heads: int, dim: int,
                    vdim: int) -> int:
    _gpu("k_pool", k_pool, dtype, 4)
    _gpu("v_pool", v_pool, dtype, 4)
    pages, heads, page_size, width = k_pool.shape
    if not (heads == kv_heads and width == dim and tuple(v_pool.shape) == (pages, kv_heads, vdim, page_size)):
        raise ValueError(f"pools {tuple(k_pool.shape)}, {tuple(v_pool.shape)} do not fit {kv_heads} heads of {dim} and {vdim}")
    return page_size


def heads_prepare(proj: torch.Tensor, offsets: tuple[int, int, int], q_heads: int, kv_heads: int, dim: int, vdim: int,
                  kernel_dim: int, kernel_vdim: int, norm: Optional[str], q_weight: Optional[torch.Tensor],
                  k_weight: Optional[torch.Tensor], eps: float, temperature: Optional[tuple[float, int]],
                  positions: torch.Tensor, seq_of_token: torch.Tensor, seq_slot: torch.Tensor,
                  block_table: torch.Tensor, k_pool: torch.Tensor, v_pool: torch.Tensor, tokens: int,
                  write_kv: bool = True, rotary: Optional[tuple] = None, maps: int = 1) -> torch.Tensor:
    """From projected rows ``proj`` [T, >= ...] (queries at column ``offsets[0]``, keys at ``offsets[1]``, values at
    ``offsets[2]``, heads of ``dim`` / ``dim`` / ``vdim`` numbers) to queries ``[T, q_heads * kernel_dim]`` and the
    token's cache entries: per-head RMS norm of queries and keys (``norm``: ``None``, ``"unit"`` or ``"weight"`` with
    float32 weights [dim]; or ``"whole"``: over all query heads together and over all key heads together, weights
    [q_heads * dim] and [kv_heads * dim]), the queries times ``1 + coef * ln(floor((p + 1) / every) + 1)`` (``temperature = (coef,
    every)``), heads zero-padded up to the kernels' sizes.  ``rotary = (cos, sin, rot, neighbours)``: after the norm
    the first ``rot`` numbers of every query and key head turn by the token's position, in pairs of neighbours
    ``(2i, 2i + 1)`` or of the halves ``(i, i + rot / 2)``; cos and sin are float32 ``[positions, rot / 2]`` and must
    reach every position of the step (the caller sees to that).  ``maps=2``: every query and key head is a pair of maps
    of ``dim`` numbers each, projected one after the other; the queries come back and the keys go to the cache with a
    head's maps side by side, ``kernel_dim`` numbers each."""
    if maps not in (1, 2) or (maps > 1 and norm == "whole"):
        raise ValueError(f"one or two maps a head (two not under the norm over all heads), got {maps}")
    if not (proj.is_cuda and proj.dim() == 2 and proj.stride(1) == 1):
        raise ValueError("proj must be 2-d on the GPU with unit inner stride")
    dtype = proj.dtype
    q_off, k_off, v_off = offsets
    need = q_off + q_heads * maps * dim
    if write_kv:
        need = max(need, k_off + kv_heads * maps * dim, v_off + kv_heads * vdim)
    if not (proj.shape[0] >= tokens and proj.shape[1] >= need and min(offsets) >= 0):
        raise ValueError(f"proj {tuple(proj.shape)} too small for {tokens} tokens of {need} numbers")
    if norm not in NORM_MODES:
        raise ValueError(f"norm must be one of {list(NORM_MODES)}, got {norm!r}")
    if norm in ("weight", "whole"):
        # ("whole": one root mean square over all query heads of a token and one over all its key heads, a weight per
        # number of the projection; a call that writes no keys needs no key weight)
        for name, w, heads in (("q_weight", q_weight, q_heads), ("k_weight", k_weight, kv_heads)):
            if w is None and name == "k_weight" and not write_kv:
                continue
            if w is None:
                raise ValueError(f"{name} is missing")
            _gpu(name, w, torch.float32, 1)
            if w.shape[0] != (dim if norm == "weight" else heads * dim):
                raise ValueError(f"{name} {tuple(w.shape)} does not fit heads of {dim} under the {norm!r} norm")
    if kernel_dim < dim or kernel_vdim < vdim:
        raise ValueError("the kernels' head sizes must hold the projection's")
    page_size = _check_kv_pools(k_pool, v_pool, dtype, kv_heads, maps * kernel_dim, kernel_vdim)
    _gpu("block_table", block_table, torch.int32, 2)
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= tokens):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {tokens} tokens")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    coef, every = temperature if temperature else (0.0, 0)
    if temperature and every < 1:
        raise ValueError("the temperature's period must be positive")
    cos = sin = None
    rot, neighbours = 0, False
    if rotary is not None:
        cos, sin, rot, neighbours = rotary
        if rot < 2 or rot % 2 or rot > dim:
            raise ValueError(f"{rot} turning numbers in heads of {dim}: even, at least 2, at most the head")
        for name, table in (("cos", cos), ("sin", sin)):
            _gpu(name, table, torch.float32, 2)
            if table.shape[1] != rot // 2 or not table.is_contiguous():
                raise ValueError(f"{name} {tuple(table.shape)} does not hold {rot // 2} pairs per position")
    q_out = torch.empty((tokens, q_heads * maps * kernel_dim), dtype=dtype, device=proj.device)
    _run("cie_heads_prepare", load_library().cie_heads_prepare(
        _stream(), _i(_code(dtype)), _ptr(proj), _i(proj.stride(0)), _i(q_off), _i(k_off), _i(v_off), _ptr(q_weight),
        _ptr(k_weight), _i(NORM_MODES[norm]), _f(eps), _f(coef), _i(every), _ptr(positions), _ptr(seq_of_token),
        _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]), _ptr(q_out), _ptr(k_pool), _ptr(v_pool),
        _i(tokens), _i(q_heads), _i(kv_heads), _i(dim), _i(vdim), _i(kernel_dim), _i(kernel_vdim), _i(page_size),
        _i(1 if write_kv else 0), _ptr(cos), _ptr(sin), _i(rot), _i(1 if neighbours else 0), _i(maps)))
    return q_out


MAX_CONV_HEAD = 256        # numbers of a head that passes a convolution
CONV_HEADS_RUN = 8         # tokens that a wave of that kernel takes ...
CONV_HEADS_RUN_FROM = 768  # ... in steps of at least this many


def heads_conv_prepare(proj: torch.Tensor, offsets: tuple[int, int, int], q_heads: int, kv_heads: int, dim: int, vdim: int,
                       kernel_dim: int, kernel_vdim: int, taps_w: Optional[torch.Tensor], past: Optional[torch.Tensor],
                       q_start_loc: torch.Tensor, sequences: int, single: bool, norm: Optional[str],
                       q_weight: Optional[torch.Tensor], k_weight: Optional[torch.Tensor], eps: float,
                       temperature: Optional[tuple[float, int]], positions: torch.Tensor, seq_of_token: torch.Tensor,
                       seq_slot: torch.Tensor, block_table: torch.Tensor, k_pool: torch.Tensor, v_pool: torch.Tensor,
                       rotary: Optional[tuple] = None, first_out: Optional[torch.Tensor] = None,
                       first_in: Optional[torch.Tensor] = None, mix: float = 0.0, run: Optional[int] = None) -> torch.Tensor:
    """What :func:`heads_prepare` does (``norm``: ``None``, ``"unit"`` or ``"weight"``; one map a head; keys and values are
    always written), for projections that first pass a causal convolution over each sequence's tokens, channel by
    channel: ``taps_w`` [n, (q_heads + kv_heads) * dim + kv_heads * vdim] in ``proj``'s dtype, its last tap meeting the
    token itself (``None``: no convolution).  ``past`` (float32 [slots, max(n - 1, 1), channels], oldest first) holds each
    request's last inputs; they are moved on by the step's inputs.  ``single``: every sequence of the step brings one token.
    The values may be mixed: ``first_out`` ([T, kv_heads * vdim]) takes them as convolved; with ``first_in`` (another
    layer's) they become ``(1 - mix) * v + mix * first_in`` before they are cached.  ``run``: tokens that a wave of the kernel
    takes, 1 or 8."""
    if not (proj.is_cuda and proj.dim() == 2 and proj.stride(1) == 1 and proj.dtype in _CODES):
        raise ValueError("proj must be a float32 or bfloat16 GPU matrix with unit inner stride")
    dtype, tokens = proj.dtype, proj.shape[0]
    q_off, k_off, v_off = offsets
    channels = (q_heads + kv_heads) * dim + kv_heads * vdim
    if min(offsets) < 0 or proj.shape[1] < max(q_off + q_heads * dim, k_off + kv_heads * dim, v_off + kv_heads * vdim):
        raise ValueError(f"proj {tuple(proj.shape)} does not hold heads at {offsets}")
    if norm not in (None, "unit", "weight"):
        raise ValueError(f"the norm over the heads must be None, 'unit' or 'weight', got {norm!r}")
    if norm == "weight":
        for name, w in (("q_weight", q_weight), ("k_weight", k_weight)):
            if w is None:
                raise ValueError(f"{name} is missing")
            _gpu(name, w, torch.float32, 1)
            if w.shape[0] != dim:
                raise ValueError(f"{name} {tuple(w.shape)} does not fit heads of {dim}")
    if not (dim <= kernel_dim <= MAX_CONV_HEAD and vdim <= kernel_vdim <= MAX_CONV_HEAD):
        raise ValueError(f"heads of {dim} and {vdim} numbers in {kernel_dim} and {kernel_vdim}, at most {MAX_CONV_HEAD}")
    page_size = _check_kv_pools(k_pool, v_pool, dtype, kv_heads, kernel_dim, kernel_vdim)
    taps = 1
    if taps_w is not None:
        _gpu("taps_w", taps_w, dtype, 2)
        taps = taps_w.shape[0]
        if taps_w.shape[1] != channels or not 1 <= taps <= MAX_CONV_TAPS:
            raise ValueError(f"taps {tuple(taps_w.shape)} for {channels} channels (up to {MAX_CONV_TAPS} taps)")
    if taps > 1:
        if past is None:
            raise ValueError("a convolution of more than one tap needs the inputs of the tokens before the step")
        _gpu("past", past, torch.float32, 3)
        if tuple(past.shape[1:]) != (taps - 1, channels):
            raise ValueError(f"past {tuple(past.shape)} must be [slots, {taps - 1}, {channels}]")
        if offsets != (q_off, q_off + q_heads * dim, q_off + (q_heads + kv_heads) * dim):
            raise ValueError("queries, keys and values of a convolution lie side by side")
    _gpu("block_table", block_table, torch.int32, 2)
    for name, meta, least in (("positions", positions, tokens), ("seq_of_token", seq_of_token, tokens),
                              ("seq_slot", seq_slot, sequences), ("q_start_loc", q_start_loc, sequences + 1)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries, the step asks for {least}")
    if single and sequences != tokens:
        raise ValueError(f"{tokens} tokens of {sequences} sequences are not one each")
    for name, t in (("first_out", first_out), ("first_in", first_in)):
        if t is not None:
            _gpu(name, t, dtype, 2)
            if tuple(t.shape) != (tokens, kv_heads * vdim):
                raise ValueError(f"{name} must be {(tokens, kv_heads * vdim)}, is {tuple(t.shape)}")
    coef, every = temperature if temperature else (0.0, 0)
    cos, sin, rot, neighbours = _check_rotary(rotary, dim)
    if run is None:
        run = CONV_HEADS_RUN if not single and 2 <= taps <= 4 and tokens >= CONV_HEADS_RUN_FROM else 1
    q_out = torch.empty((tokens, q_heads * kernel_dim), dtype=dtype, device=proj.device)
    _run("cie_heads_conv_prepare", load_library().cie_heads_conv_prepare(
        _stream(), _i(_code(dtype)), _ptr(proj), _i(_ld(proj)), _i(q_off), _i(k_off), _i(v_off), _ptr(taps_w), _i(taps),
        _ptr(past if taps > 1 else None), _ptr(q_start_loc), _i(1 if single else 0), _ptr(first_out), _ptr(first_in), _f(mix),
        _ptr(q_weight), _ptr(k_weight), _i(NORM_MODES[norm]), _f(eps), _f(coef), _i(every), _ptr(positions), _ptr(seq_of_token),
        _ptr(seq_slot), _ptr(block_table), _i(block_table.shape[1]), _ptr(q_out), _ptr(k_pool), _ptr(v_pool), _i(tokens),
        _i(q_heads), _i(kv_heads), _i(dim), _i(vdim), _i(kernel_dim), _i(kernel_vdim), _i(page_size), _ptr(cos), _ptr(sin),
        _i(rot), _i(1 if neighbours else 0), _i(run)))
    if taps > 1 and not single:
        conv_keep(proj[:, q_off: q_off + channels], past, seq_slot, q_start_loc, sequences, taps)
    return q_out


def _attention_out(out: Optional[torch.Tensor], tokens: int, numbers: int, dtype: torch.dtype, device) -> torch.Tensor:
    """Where attention writes its rows: a new matrix, or one of the caller's whose rows may lie apart."""
    if out is None:
        return torch.empty((tokens, numbers), dtype=dtype, device=device)
    _row_view("out", out, (tokens, numbers), (dtype,))
    return out


def _check_score_shape(q_heads: int, slopes, sinks, softcap, window=None, chunk=None, keep_first=0) -> None:
    if chunk is not None and (chunk < 1 or window):
        raise ValueError(f"chunks hold at least one token and stand in a window's place, got chunk {chunk}, window {window}")
    if keep_first < 0 or (keep_first and not window):
        raise ValueError(f"kept first keys ({keep_first}) are a count and come with a window")
    for name, t in (("slopes", slopes), ("sinks", sinks)):
        if t is not None:
            _gpu(name, t, torch.float32, 1)
            if t.shape[0] != q_heads:
                raise ValueError(f"{name} must be [{q_heads}], is {tuple(t.shape)}")
    if softcap is not None and not softcap > 0:
        raise ValueError(f"the cap on the scores must be positive, got {softcap}")


def _check_gate(gate, tokens: int, numbers: int, dtype: torch.dtype) -> int:
    if gate is None:
        return 0
    if not (gate.is_cuda and gate.dim() == 2 and gate.stride(1) == 1 and gate.dtype == dtype
            and gate.shape[0] >= tokens and gate.shape[1] >= numbers):
        raise ValueError(f"gate {tuple(gate.shape)} {gate.dtype} does not hold {tokens} rows of {numbers} gates")
    return _ld(gate)


def _check_maps(differential, vdim: int, real_vdim: Optional[int], sinks) -> tuple[int, int, float, float, float]:
    """(maps, numbers of a value head that are not padding, lambda, factor, eps)."""
    real = vdim if real_vdim is None else int(real_vdim)
    if not 1 <= real <= vdim:
        raise ValueError(f"{real_vdim} numbers of a value head of {vdim}")
    if differential is None:
        return 1, real, 0.0, 1.0, 1.0
    lam, factor, eps = (float(x) for x in differential)
    if sinks is not None or not eps > 0:
        raise ValueError("two maps come without a sink and with a positive eps")
    return 2, real, lam, factor, eps


def scored_attention_generic(q: torch.Tensor, k_pool: torch.Tensor, v_pool: torch.Tensor, block_table: torch.Tensor,
                             positions: torch.Tensor, seq_of_token: torch.Tensor, seq_slot: torch.Tensor, tokens: int,
                             q_heads: int, kv_heads: int, dim: int, vdim: int, window: Optional[int], scale: float,
                             softcap: Optional[float] = None, slopes: Optional[torch.Tensor] = None,
                             sinks: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None,
                             chunk: Optional[int] = None, keep_first: int = 0, gate_wide: bool = False,
                             real_vdim: Optional[int] = None, differential: Optional[tuple] = None,
                             out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Attention of each token over its request's cached keys with shaped scores (see ``csrc/attention_scored.hip``;
    ``chunk``: a token sees the keys of its own chunk of that many positions, counted from position 0, up to itself;
    ``keep_first``: beside its window a token sees the first that many keys of its sequence):
    ``q`` [T, q_heads * dim]; returns [T, q_heads * vdim].  ``gate`` [T, >= q_heads] (a view is fine): head h's output
    is multiplied by ``sigmoid(gate[t, h])``; with ``gate_wide`` the gate has a number for each of a head's
    ``real_vdim`` numbers (``vdim`` less its padding).  ``differential = (lambda, factor, eps)``: query and key heads are
    pairs of maps (``q`` [T, q_heads * 2 * dim]), each a softmax of its own over the same values; head h's output is
    ``factor * (a1 - lambda a2) / rms(a1 - lambda a2)``.  float32 or bfloat16."""
    _gpu("q", q, dims=2)
    maps, real, lam, factor, eps = _check_maps(differential, vdim, real_vdim, sinks)
    if not (q.shape == (tokens, q_heads * maps * dim) and q_heads % kv_heads == 0 and dim % 8 == 0 and vdim % 8 == 0
            and vdim <= MAX_GENERIC_VALUE and 4 * (dim + (4 + maps) * vdim) <= 60 * 1024):
        raise ValueError(f"q {tuple(q.shape)} does not fit {tokens} tokens of {q_heads} heads of {dim} and {vdim} (multiples of "
                         f"8, values up to {MAX_GENERIC_VALUE})")
    page_size = _check_kv_pools(k_pool, v_pool, q.dtype, kv_heads, maps * dim, vdim)
    _gpu("block_table", block_table, torch.int32, 2)
    for name, meta in (("positions", positions), ("seq_of_token", seq_of_token)):
        _gpu(name, meta, torch.int32, 1)
        if not (meta.shape[0] >= tokens):
            raise ValueError(f"{name} has {meta.shape[0]} entries for {tokens} tokens")
    _gpu("seq_slot", seq_slot, torch.int32, 1)
    _check_score_shape(q_heads, slopes, sinks, softcap, window, chunk, keep_first)
    gate_stride = _check_gate(gate, tokens, q_heads * real if gate_wide else q_heads, q.dtype)
    out = _attention_out(out, tokens, q_heads * vdim, q.dtype, q.device)
    _run("cie_scored_attention_generic", load_library().cie_scored_attention_generic(
        _stream(), _i(_code(q.dtype)), _ptr(q), _ptr(k_pool), _ptr(v_pool), _ptr(block_table), _i(block_table.shape[1]),
        _ptr(positions), _ptr(seq_of_token), _ptr(seq_slot), _ptr(gate), _i(gate_stride), _ptr(out), _i(tokens),
        _i(q_heads), _i(kv_heads), _i(dim), _i(vdim), _i(page_size), _i(window or 0), _f(scale), _f(softcap or 0.0),
        _ptr(slopes), _ptr(sinks), _i(chunk or 0), _i(keep_first), _i(1 if gate_wide else 0), _i(real), _i(maps), _f(lam),
        _f(factor), _f(eps), _ld(out)))
    return out


def scored_attention_mfma(q: torch.Tensor, k_pool: torch.Tensor, v_pool: torch.Tensor, block_table: torch.Tensor,
                          tile_seq: Optional[torch.Tensor], tile_q0: Optional[torch.Tensor], n_tiles: int,
                          seq_slot: torch.Tensor, seq_start: torch.Tensor, seq_q_len: torch.Tensor,
                          q_start_loc: torch.Tensor, tokens: int, q_heads: int, kv_heads: int, dim: int, vdim: int,
                          tokens_per_tile: int, row_tiles: int, window: Optional[int], scale: float,
                          softcap: Optional[float] = None, slopes: Optional[torch.Tensor] = None,
                          sinks: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None,
                          n_splits: int = 1, keys_per_split: int = 0, chunk: Optional[int] = None,
                          keep_first: int = 0, gate_wide: bool = False, real_vdim: Optional[int] = None,
                          differential: Optional[tuple] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The same on the matrix cores (bfloat16, (dim, vdim) in ``SCORED_MFMA_DIMS`` or ``LATENT_MFMA_DIMS``, with two maps in
    ``DIFFERENTIAL_MFMA_DIMS``; pages of a power of two >= 4; two maps' rows fill ``row_tiles`` tiles together):
    tiles of ``tokens_per_tile`` consecutive tokens of one sequence (``tile_seq``, ``tile_q0`` int32 [n_tiles]; both
    ``None``: tile i is sequence i's first), whose rows times the heads per key head fill ``row_tiles`` tiles of 16.
    ``n_splits > 1``: every tile's keys in that many shares of ``keys_per_split`` (a multiple of 128; the shares must
    cover the longest range of keys a tile sees), a workgroup each, joined by a second kernel."""
    _gpu("q", q, torch.bfloat16, 2)
    maps, real, lam, factor, eps = _check_maps(differential, vdim, real_vdim, sinks)
    most = (DIFFERENTIAL_MFMA_DIMS.get((dim, vdim)) if maps == 2
            else 4 if (dim, vdim) in SCORED_MFMA_DIMS else LATENT_MFMA_DIMS.get((dim, vdim)))
    if most is None or not (q.shape == (tokens, q_heads * maps * dim) and q_heads % kv_heads == 0):
        raise ValueError(f"q {tuple(q.shape)} / heads of {dim}, {vdim} are not what the matrix-core form takes")
    page_size = _check_kv_pools(k_pool, v_pool, q.dtype, kv_heads, maps * dim, vdim)
    if page_size < 4 or page_size & (page_size - 1):
        raise ValueError(f"pages must hold a power of two >= 4 keys, hold {page_size}")
    group = q_heads // kv_heads
    if (row_tiles not in (1, 2, 4) or not maps <= row_tiles <= most or tokens_per_tile < 1
            or tokens_per_tile * group * maps > 16 * row_tiles):
        raise ValueError(f"{tokens_per_tile} tokens of {group} heads do not fit {row_tiles} tiles of 16 rows (at most {most})")
    _gpu("block_table", block_table, torch.int32, 2)
    if (tile_seq is None) != (tile_q0 is None):
        raise ValueError("tile_seq and tile_q0 come together")
    if tile_seq is not None:
        for name, t in (("tile_seq", tile_seq), ("tile_q0", tile_q0)):
            _gpu(name, t, torch.int32, 1)
            if t.shape[0] < n_tiles:
                raise ValueError(f"{name} has {t.shape[0]} entries for {n_tiles} tiles")
    sequences = seq_slot.shape[0]
    for name, meta, least in (("seq_slot", seq_slot, 1), ("seq_start", seq_start, sequences),
                              ("seq_q_len", seq_q_len, sequences), ("q_start_loc", q_start_loc, sequences)):
        _gpu(name, meta, torch.int32, 1)
        if meta.shape[0] < least:
            raise ValueError(f"{name} has {meta.shape[0]} entries for {sequences} sequences")
    if tile_seq is None and n_tiles > sequences:
        raise ValueError(f"{n_tiles} tiles for {sequences} sequences")
    _check_score_shape(q_heads, slopes, sinks, softcap, window, chunk, keep_first)
    gate_stride = _check_gate(gate, tokens, q_heads * real if gate_wide else q_heads, q.dtype)
    out = _attention_out(out, tokens, q_heads * vdim, q.dtype, q.device)
    part_o = part_ml = None
    if n_splits > 1:
        if keys_per_split < 128 or keys_per_split % 128:
            raise ValueError(f"shares of the keys are multiples of 128, got {keys_per_split}")
        units = n_tiles * kv_heads * n_splits * 16 * row_tiles
        part_o = torch.empty(units * vdim, dtype=torch.float32, device=q.device)
        part_ml = torch.empty(units * 2, dtype=torch.float32, device=q.device)
    elif n_splits != 1:
        raise ValueError("n_splits must be positive")
    _run("cie_scored_attention_mfma", load_library().cie_scored_attention_mfma(
        _stream(), _ptr(q), _ptr(k_pool), _ptr(v_pool), _ptr(block_table), _i(block_table.shape[1]), _ptr(tile_seq),
        _ptr(tile_q0), _i(n_tiles), _ptr(seq_slot), _ptr(seq_start), _ptr(seq_q_len), _ptr(q_start_loc), _ptr(gate),
        _i(gate_stride), _ptr(out), _i(q_heads), _i(kv_heads), _i(maps * dim), _i(vdim), _i(page_size), _i(tokens_per_tile),
        _i(row_tiles), _i(window or 0), _f(scale), _f(softcap or 0.0), _ptr(slopes), _ptr(sinks), _i(n_splits),
        _i(keys_per_split), _ptr(part_o), _ptr(part_ml), _i(chunk or 0), _i(keep_first), _i(1 if gate_wide else 0), _i(real),
        _i(maps), _f(lam), _f(factor), _f(eps), _ld(out)))
    return out


# ---------------------------------------------------------------------------
MAX_EXPERTS = 1024
EXPERT_TILE_ROWS = (16, 32, 64, 128)  # rows of one expert that a workgroup of the matrix-core forms takes (128: through LDS)


class ExpertRoute:
    """What ``experts_route`` leaves on the device for the expert products of one step."""

    __slots__ = ("pair_expert", "pair_weight", "sorted", "tile_expert", "tile_begin", "tile_count", "n_tiles",
                 "max_tiles", "tile_rows", "top", "pairs", "real", "pair_expert_outputs")


MAX_EXPERT_GROUPS = 64


def experts_route(logits: torch.Tensor, top: int, tile_rows: int = 16, real: Optional[int] = None,
                  scoring: str = "sigmoid", correction: Optional[torch.Tensor] = None,
                  groups: Optional[tuple[int, int]] = None, normalize: bool = False, scale: float = 1.0) -> ExpertRoute:
    """Scores ``sigmoid(logits)`` (float32 [T, E]), the ``top`` largest per token (ranked by the logits, which order
    the scores and do not saturate; lowest index first among equals),
    and the (token, choice) pairs sorted by expert in tiles of at most ``tile_rows`` rows.  Nothing comes back to
    the host: grids are sized for ``max_tiles`` and the kernels read the true count.

    What else a router may ask for: ``scoring="softmax"`` (scores are the softmax over all E outputs);
    ``correction`` (float32 [E], added to the scores for the choice only); ``groups=(count, keep)`` (the outputs form
    ``count`` equal runs of neighbours, a run counts by its largest choice score, and only outputs of the ``keep``
    best runs can be chosen); ``normalize`` (the chosen scores divided by their sum + 1e-20, times ``scale``);
    ``real`` (only the first ``real`` outputs are experts with weights: pairs of the others get no tiles, and
    ``experts_forward`` hands their token's row on as it is)."""
    _gpu("logits", logits, torch.float32, 2)
    tokens, experts = logits.shape
    if not (1 <= top <= experts <= MAX_EXPERTS and tile_rows >= 1):
        raise ValueError(f"{top} of {experts} experts (at most {MAX_EXPERTS}) in tiles of {tile_rows}")
    real = experts if real is None else real
    if not 0 <= real <= experts or scoring not in ("sigmoid", "softmax"):
        raise ValueError(f"{real} experts of {experts} outputs with {scoring!r} scores")
    if correction is not None:
        _gpu("correction", correction, torch.float32, 1)
        if correction.shape[0] != experts:
            raise ValueError(f"correction must be [{experts}], is {tuple(correction.shape)}")
    count, keep = groups if groups else (1, 1)
    if count > 1 and not (count <= MAX_EXPERT_GROUPS and experts % count == 0 and 1 <= keep <= count
                          and top <= keep * (experts // count)):
        raise ValueError(f"{count} groups of which {keep} are kept do not fit {top} of {experts} outputs")
    route = ExpertRoute()
    pairs = tokens * top
    route.pairs, route.top, route.tile_rows, route.real = pairs, top, tile_rows, real
    route.pair_expert_outputs = experts  # how many outputs the router has; those from ``real`` on have no weights
    route.max_tiles = min(pairs, pairs // tile_rows + real)
    ints = torch.empty(2 * pairs + 3 * max(route.max_tiles, 1) + 1, dtype=torch.int32, device=logits.device)
    route.pair_expert, route.sorted = ints[:pairs], ints[pairs: 2 * pairs]
    base = 2 * pairs
    width = max(route.max_tiles, 1)
    route.tile_expert, route.tile_begin, route.tile_count = (ints[base + i * width: base + (i + 1) * width] for i in range(3))
    route.n_tiles = ints[base + 3 * width:]
    route.pair_weight = torch.empty(pairs, dtype=torch.float32, device=logits.device)
    _run("cie_experts_route", load_library().cie_experts_route(
        _stream(), _ptr(logits), _i(tokens), _i(experts), _i(top), _i(tile_rows), _ptr(route.pair_expert),
        _ptr(route.pair_weight), _ptr(route.sorted), _ptr(route.tile_expert), _ptr(route.tile_begin),
        _ptr(route.tile_count), _ptr(route.n_tiles), _i(real), _i(1 if scoring == "softmax" else 0), _ptr(correction),
        _i(count), _i(keep), _i(1 if normalize else 0), _f(scale)))
    return route


def experts_forward(x: torch.Tensor, route: ExpertRoute, w_gate_up: torch.Tensor, w_down: torch.Tensor, limit: float,
                    alpha: float, offset: float, mfma: bool, weight_input: bool = True) -> torch.Tensor:
    """The chosen experts' outputs, float32 ``[T, top, hidden]``: row (t, k) is expert ``k`` of token t run on
    ``weight * x[t]``, or, with ``weight_input=False``, on ``x[t]`` itself (whoever sums the rows then applies
    ``route.pair_weight``).  ``w_gate_up`` [E, 2 * ff, hidden] (gate rows first), ``w_down`` [E, hidden, ff].  A pair
    whose choice lies behind the experts that have weights (``route.real``) gets ``x[t]`` as its row."""
    _gpu("x", x, dims=2)
    tokens, hidden = x.shape
    _gpu("w_gate_up", w_gate_up, x.dtype, 3)
    _gpu("w_down", w_down, x.dtype, 3)
    experts, twice, _ = w_gate_up.shape
    ff = twice // 2
    if not (w_gate_up.shape == (experts, 2 * ff, hidden) and w_down.shape == (experts, hidden, ff)
            and tokens * route.top == route.pairs and experts == route.real):
        raise ValueError(f"expert weights {tuple(w_gate_up.shape)}, {tuple(w_down.shape)} do not fit rows {tuple(x.shape)}")
    if mfma and not (x.dtype == torch.bfloat16 and hidden % 8 == 0 and ff % 8 == 0 and route.tile_rows in EXPERT_TILE_ROWS):
        raise ValueError("the matrix-core form takes bfloat16, widths that are multiples of 8 and tiles of 16, 32, 64 or 128 rows")
    if not mfma and route.tile_rows > 16:
        raise ValueError("the plain form takes tiles of up to 16 rows")
    act = torch.empty((route.pairs, ff), dtype=x.dtype, device=x.device)
    parts = torch.empty((tokens, route.top, hidden), dtype=torch.float32, device=x.device)
    lib = load_library()
    rows_in = x
    pair_weight = route.pair_weight if weight_input else None
    if mfma and route.tile_rows == 128:
        # many rows an expert: the rows in sorted order, weights applied, for the form that stages tiles through LDS
        gathered = torch.empty((route.pairs, hidden), dtype=x.dtype, device=x.device)
        _run("cie_experts_gather", lib.cie_experts_gather(_stream(), _ptr(x), _ptr(gathered), _ptr(route.sorted),
                                                          _ptr(pair_weight), _i(route.pairs), _i(route.top), _i(hidden)))
        x = gathered
    _run("cie_experts_gate_up", lib.cie_experts_gate_up(
        _stream(), _i(_code(x.dtype)), _i(1 if mfma else 0), _ptr(x), _ptr(w_gate_up), _ptr(act), _ptr(route.sorted),
        _ptr(pair_weight), _ptr(route.tile_expert), _ptr(route.tile_begin), _ptr(route.tile_count),
        _ptr(route.n_tiles), _i(route.max_tiles), _i(route.tile_rows), _i(route.top), _i(hidden), _i(ff), _f(limit),
        _f(alpha), _f(offset)))
    _run("cie_experts_down", lib.cie_experts_down(
        _stream(), _i(_code(x.dtype)), _i(1 if mfma else 0), _ptr(act), _ptr(w_down), _ptr(parts), _ptr(route.sorted),
        _ptr(route.tile_expert), _ptr(route.tile_begin), _ptr(route.tile_count), _ptr(route.n_tiles),
        _i(route.max_tiles), _i(route.tile_rows), _i(route.top), _i(hidden), _i(ff)))
    if route.real < route.pair_expert_outputs:
        _run("cie_experts_identity", lib.cie_experts_identity(
            _stream(), _i(_code(rows_in.dtype)), _ptr(rows_in), _ptr(route.pair_expert), _i(route.real), _ptr(parts),
            _i(route.pairs), _i(route.top), _i(hidden)))
    return parts
