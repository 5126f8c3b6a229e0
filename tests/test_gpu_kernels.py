"""GPU: each HIP kernel alone against a plain float32 torch reference of the same
operation, at sizes other than the tiny models' (odd widths, many heads and
groups, head sizes in steps of 16)."""

from __future__ import annotations

import math
import random

import pytest
import torch

import plain_qwen2

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


def tol(dtype):
    return dict(rtol=1e-5, atol=1e-5) if dtype == torch.float32 else dict(rtol=1.6e-2, atol=1e-2)


def rand(shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype).cuda()


@pytest.fixture(scope="module")
def ops():
    from cie_amd.kernels import ops as module

    return module


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed(ops, dtype):
    table = rand((1000, 72), dtype, 1)
    ids = torch.tensor([0, 999, 5, 5, 321], dtype=torch.int32).cuda()
    out = ops.embed(table, ids)
    assert out.dtype == torch.float32
    torch.testing.assert_close(out, table.float()[ids.long()], rtol=0, atol=0)
    # rows 1 and 3 take their tokens from a pool on the device instead
    feed = torch.tensor([-1, 2, -1, 0, -1], dtype=torch.int32).cuda()
    pool = torch.tensor([77, 500, 901], dtype=torch.int32).cuda()
    fed = ops.embed(table, ids, feed=feed, pool=pool)
    expect = torch.tensor([0, 901, 5, 77, 321]).cuda()
    torch.testing.assert_close(fed, table.float()[expect], rtol=0, atol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hidden", [72, 1000, 4104])
def test_add_rmsnorm(ops, dtype, hidden):
    residual = rand((7, hidden), torch.float32, 2, 3.0)
    branch = rand((7, hidden), dtype, 3)
    weight = rand((hidden,), dtype, 4) + 1
    eps = 1e-5
    expect_res = residual + branch.float()
    expect = plain_qwen2.rms_norm(expect_res, weight.float(), eps)
    out = ops.add_rmsnorm(residual, branch, weight, eps, dtype)
    torch.testing.assert_close(residual, expect_res, rtol=0, atol=0)  # the float32 sum is written back
    torch.testing.assert_close(out.float(), expect, **tol(dtype))
    # no branch, selected rows only, float32 weight beside bf16 activations
    rows = torch.tensor([6, 0, 3], dtype=torch.int32).cuda()
    before = residual.clone()
    out = ops.add_rmsnorm(residual, None, weight.float(), eps, dtype, rows=rows)
    torch.testing.assert_close(residual, before, rtol=0, atol=0)
    torch.testing.assert_close(out.float(), expect[rows.long()], **tol(dtype))


def test_rmsnorm_invariants(ops):
    """weight 1, tiny eps: every output row has RMS 1; scaling the input changes nothing."""
    x = rand((4, 200), torch.float32, 5, 2.0)
    ones = torch.ones(200, device="cuda")
    out = ops.add_rmsnorm(x.clone(), None, ones, 1e-12, torch.float32)
    torch.testing.assert_close(out.pow(2).mean(-1), torch.ones(4, device="cuda"), rtol=1e-5, atol=1e-5)
    out2 = ops.add_rmsnorm(x * 7.5, None, ones, 1e-12, torch.float32)
    torch.testing.assert_close(out, out2, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
def test_silu_mul(ops, dtype):
    gate_up = rand((5, 2 * 333), dtype, 6, 2.0)
    g, u = gate_up.float()[:, :333], gate_up.float()[:, 333:]
    out = ops.silu_mul(gate_up)
    torch.testing.assert_close(out.float(), torch.nn.functional.silu(g) * u, **tol(dtype))
    zero_gate = torch.cat([torch.zeros(5, 333), torch.randn(5, 333)], dim=1).to(dtype).cuda()
    assert ops.silu_mul(zero_gate).abs().max().item() == 0.0


@pytest.mark.parametrize("shape", [(1, 40, 24), (5, 515, 96), (70, 130, 200), (130, 64, 17)])
def test_gemm_f32(ops, shape):
    m, n, k = shape
    a, w, b = rand((m, k), torch.float32, 7), rand((n, k), torch.float32, 8), rand((n,), torch.float32, 9)
    expect = (a.double() @ w.double().t() + b.double()).float()
    torch.testing.assert_close(ops.gemm_f32(a, w, b), expect, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(ops.gemm_f32(a, w), (a.double() @ w.double().t()).float(), rtol=1e-5, atol=1e-5)
    # a row's result does not depend on the other rows of the batch (bitwise)
    assert torch.equal(ops.gemm_f32(a[:1].contiguous(), w, b), ops.gemm_f32(a, w, b)[:1])


# (rows, columns, K): single and half empty tiles, an odd K (no 16-byte loads), K at the edges of pieces, blocks and
# stretches, columns for the narrow, the middle and the wide workgroups of the few-row form
@pytest.mark.parametrize("shape", [(1, 8, 4), (9, 7, 33), (64, 66, 256), (65, 64, 1024), (17, 258, 1028), (33, 70, 2047),
                                   (8, 2048, 2052), (5, 16384, 64), (20, 16386, 40), (130, 130, 4100)])
def test_gemm_f32_forms(ops, shape):
    """Every form of the float32 product gives the same bits, also for rows that lie apart, and its gated unit the bits
    of the unit's own kernel behind the product.  The bound is what K + 8 roundings of half a unit in the last place
    (6e-8) can add up to."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.float32, 13), rand((n, k), torch.float32, 14), rand((n,), torch.float32, 15)
    wide = torch.zeros((m, k + 12)).cuda()
    wide[:, :k] = a
    exact = a.double() @ w.double().t() + b.double()
    bound = 6e-8 * (k + 8) * (a.double().abs() @ w.double().abs().t() + b.double().abs())
    outs = [ops.gemm_f32(a, w, b, form=form) for form in (0, 1, 2)] + [ops.gemm_f32(wide[:, :k], w, b), ops.gemm_f32(a, w, b)]
    assert ((outs[0].double() - exact).abs() <= bound).all()
    assert all(torch.equal(out, outs[0]) for out in outs[1:])
    if n % 2 == 0:
        unit = ops.silu_mul(ops.gemm_f32(a, w))
        assert all(torch.equal(ops.gemm_f32(a, w, gate=True, form=form), unit) for form in (0, 1, 2))


# (rows, columns, K): a part of a piece, segments of 512 numbers that are full and not, four and eight waves, one and several
# rounds of blocks, narrow, middle and wide workgroups (with the gate columns of either half past the last), the widest rows
@pytest.mark.parametrize("shape", [(1, 64, 8), (3, 384, 64), (8, 2560, 896), (7, 130, 1032), (4, 16384, 520), (6, 16386, 1104),
                                   (2, 48, 8192), (8, 48, 2048), (3, 100, 4104), (8, 16448, 2048),
                                   (8, 16386, 1000), (2, 22, 512), (5, 64, 4096)])
def test_gemm_f32_with_its_neighbours(ops, shape):
    """The gated float32 product of few rows that makes the norm in front of it, and the one that adds into the stream, give the bits
    of the kernels that they take the place of."""
    m, n, k = shape
    x, w, b = rand((m, k), torch.float32, 71, 3.0), rand((n, k), torch.float32, 72), rand((n,), torch.float32, 73)
    x *= torch.linspace(0.01, 5.0, m, device="cuda")[:, None]
    gain, eps = (1.0 + rand((k,), torch.float32, 74, 0.3)).contiguous(), 1e-5
    before = x.clone()
    if m * -(-k // 512) > 32:
        assert not ops.folds_norm_f32(x)
    else:
        normed = ops.add_rmsnorm(x.clone(), None, gain, eps, torch.float32)
        assert torch.equal(ops.gemm_f32_normed(x, gain, eps, w), ops.gemm_f32(normed, w, gate=True, form=0))
    assert torch.equal(x, before)
    wide = torch.zeros((m, k + 3)).cuda()
    wide[:, :k] = x
    stream = rand((m, n), torch.float32, 75)
    for a, bias in ((x, b), (x, None), (wide[:, :k], b)):
        sums = stream.clone()
        ops.gemm_f32_into(a, w, bias, sums)
        assert torch.equal(sums, stream + ops.gemm_f32(a, w, bias, form=0))


def test_gemm_f32_with_its_neighbours_refuses(ops):
    w, gain = torch.zeros((16, 64), device="cuda"), torch.ones(64, device="cuda")
    for stream in (torch.zeros((9, 64), device="cuda"), torch.zeros((0, 64), device="cuda"), torch.zeros((4, 128), device="cuda")[:, ::2],
                   torch.zeros(4 * 64 + 1, device="cuda")[1:].view(4, 64)):
        assert not ops.folds_norm_f32(stream)
        with pytest.raises(ValueError, match="makes the norm"):
            ops.gemm_f32_normed(stream, gain, 1e-6, w)
    with pytest.raises(ValueError, match="up to 8 rows"):
        ops.gemm_f32_into(torch.zeros((9, 64), device="cuda"), w, None, torch.zeros((9, 16), device="cuda"))


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16, 2048), (4, 2, 16, 8, 64), (3, 1, 64, 4, 328), (5, 5, 96, 32, 200), (2, 1, 48, 1, 1040)])
@pytest.mark.parametrize("rows", [1, 3, 7, 8])
@pytest.mark.parametrize("rotate,write,biased", [(True, True, True), (False, True, False), (True, False, True)])
@pytest.mark.parametrize("part", [False, True])
def test_gemm_f32_qkv_rope(ops, geometry, rows, rotate, write, biased, part):
    """... and with the rotation and the cache write, those of the norm's, the product's and the rotation's kernels."""
    q_heads, kv_heads, head_dim, page_size, hidden = geometry
    if rows * -(-hidden // 512) > 32:
        rows = 32 // -(-hidden // 512)
    n = (q_heads + 2 * kv_heads) * head_dim
    lengths = [40, 35, 100, 33, 64, 1, 17, 90][:rows]
    k_pool, v_pool, table, slots, _ = build_cache(torch.float32, lengths, kv_heads, head_dim, page_size, seed=81)
    k_two, v_two = k_pool.clone(), v_pool.clone()
    x = rand((rows, hidden), torch.float32, 82, 2.0)
    gain, eps = (1.0 + rand((hidden,), torch.float32, 83, 0.3)).contiguous(), 1e-6
    w, b = rand((n, hidden), torch.float32, 84, 0.05), rand((n,), torch.float32, 85) if biased else None
    cos, sin = plain_qwen2.rope_tables(head_dim, 512, 1e6)
    turning = 16 if part else head_dim  # (how much of a head rotates)
    cos, sin = (t[:, : turning // 2].contiguous().cuda() for t in (cos, sin))
    meta = (torch.tensor([length - 1 for length in lengths], dtype=torch.int32).cuda(), torch.arange(rows, dtype=torch.int32).cuda(),
            torch.tensor(slots, dtype=torch.int32).cuda(), table)
    got = ops.gemm_f32_qkv_rope(x, gain, eps, w, b, cos, sin, *meta, k_pool, v_pool, q_heads, kv_heads, head_dim, rotate=rotate, write_kv=write, rotary_dim=turning)
    expect = ops.gemm_f32(ops.add_rmsnorm(x.clone(), None, gain, eps, torch.float32), w, b, form=0)
    ops.rope_kv_write(expect, cos, sin, *meta, k_two, v_two, q_heads, kv_heads, head_dim, rotate=rotate, write_kv=write, rotary_dim=turning)
    assert torch.equal(got[:, : q_heads * head_dim], expect[:, : q_heads * head_dim])
    assert torch.equal(k_pool, k_two) and torch.equal(v_pool, v_two)


# five and more tiles of 64 x 64 to each of 256 units: whole row blocks, rows of which one and more than 48 are left, a
# number of slices that is no multiple of a chain's four, blocks of K behind one another, two stretches and a part of a third
@pytest.mark.parametrize("shape", [(640, 8192, 96), (641, 8194, 160), (700, 8130, 32), (1281, 4098, 2080)])
def test_gemm_f32_many_tiles(ops, shape):
    """The tiles that load straight into LDS give the bits of the form for few rows, and of its gated unit, also for rows
    that lie apart."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.float32, 13), rand((n, k), torch.float32, 14), rand((n,), torch.float32, 15)
    assert -(-m // 64) * -(-(n // 2) // 32) >= 5 * ops.compute_units()  # (with the gate a tile takes 32 of either half)
    wide = torch.zeros((m, k + 12)).cuda()
    wide[:, :k] = a
    expect, unit = ops.gemm_f32(a, w, b, form=0), ops.gemm_f32(a, w, gate=True, form=0)
    for rows in (a, wide[:, :k]):
        assert torch.equal(ops.gemm_f32(rows, w, b, form=1), expect) and torch.equal(ops.gemm_f32(rows, w, gate=True, form=1), unit)
    assert torch.equal(ops.gemm_f32(a, w, form=1), ops.gemm_f32(a, w, form=0))
    assert torch.equal(ops.gemm_f32(a, w, b, form=2), expect) and torch.equal(ops.gemm_f32(a, w, gate=True, form=2), unit)


@pytest.mark.parametrize("shape", [(600, 4098, 4128), (449, 4160, 6144)])
def test_gemm_f32_many_stretches(ops, shape):
    """Twelve and more tiles to a unit with K in stretches (the last one short, or all of them whole): loaded straight into
    LDS, the same bits, the gated unit's too, and for rows that lie apart."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.float32, 16), rand((n, k), torch.float32, 17), rand((n,), torch.float32, 18)
    assert -(-m // 64) * -(-n // 64) * -(-k // 1024) >= 12 * ops.compute_units() and ops.f32_bands(m, n, k)[0] == 1
    wide = torch.zeros((m, k + 4)).cuda()
    wide[:, :k] = a
    expect, unit = ops.gemm_f32(a, w, b, form=0), ops.gemm_f32(a, w, gate=True, form=0)
    for rows in (a, wide[:, :k]):
        assert torch.equal(ops.gemm_f32(rows, w, b, form=2), expect) and torch.equal(ops.gemm_f32(rows, w, gate=True, form=2), unit)


@pytest.mark.parametrize("shape", [(200, 66, 1028), (129, 130, 4100)])
def test_gemm_f32_in_bands_of_rows(ops, monkeypatch, shape):
    """Stretches of K whose sums do not fit the workspace: the rows go in bands, with the bits of the other forms."""
    m, n, k = shape
    wide = rand((m, k + 12), torch.float32, 13)
    a, w, b = wide[:, :k], rand((n, k), torch.float32, 14), rand((n,), torch.float32, 15)
    expect, unit = ops.gemm_f32(a, w, b, form=1), ops.gemm_f32(a, w, gate=True, form=1)
    monkeypatch.setattr(ops, "F32_WORKSPACE_BYTES", 1)
    assert ops.f32_bands(m, n, k) == (-(-m // 64), 64)
    assert torch.equal(ops.gemm_f32(a, w, b, form=2), expect) and torch.equal(ops.gemm_f32(a, w, gate=True, form=2), unit)


@pytest.mark.parametrize("shape", [(1, 40, 24), (5, 515, 96), (16, 64, 128), (17, 130, 200), (33, 70, 1032),
                                   (64, 256, 264), (150, 99, 72)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_gemm_fused_plain_any_size(ops, shape, out_dtype):
    """Plain product with bias: rows from 1 to more than a workgroup takes, column counts
    that are no multiple of 16, inner sizes that are no multiple of 128."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.bfloat16, 10), rand((n, k), torch.bfloat16, 11), rand((n,), torch.bfloat16, 12)
    expect = a.double() @ w.double().t()
    epilogue = ops.EPI_F32 if out_dtype == torch.float32 else ops.EPI_BF16
    out = ops.gemm_fused(w, epilogue, a)
    assert out.dtype == out_dtype and out.shape == (m, n)
    if out_dtype == torch.float32:
        torch.testing.assert_close(out.double(), expect, rtol=1e-4, atol=1e-4 * math.sqrt(k))
    else:
        torch.testing.assert_close(out.double(), expect, rtol=1e-2, atol=1e-2 * math.sqrt(k))
    out = ops.gemm_fused(w, ops.EPI_F32, a, bias=b)
    torch.testing.assert_close(out.double(), expect + b.double(), rtol=1e-4, atol=1e-4 * math.sqrt(k))
    # rows given as a strided view (a slice of a wider buffer)
    wide = torch.zeros((m, k + 64), dtype=torch.bfloat16).cuda()
    wide[:, :k] = a
    torch.testing.assert_close(ops.gemm_fused(w, ops.EPI_F32, wide[:, :k]), ops.gemm_fused(w, ops.EPI_F32, a), rtol=0, atol=0)


# (rows, columns, K): less than a tile, edges of 16 and of the tiles, a K that ends inside a slice, odd columns
@pytest.mark.parametrize("shape", [(1, 32, 8), (63, 64, 64), (65, 130, 136), (129, 256, 200), (200, 99, 72), (257, 96, 1032)])
@pytest.mark.parametrize("tile", [(64, 64), (128, 64), (128, 128), (128, 256)])
def test_gemm_tiles(ops, shape, tile):
    """Products of some hundred rows in tiles: the plain result with bias, its gated unit, the add into the stream and the
    parts of K (which sum to the same), for rows that lie apart too."""
    m, n, k = shape
    wide = torch.zeros((m, k + 24), dtype=torch.bfloat16).cuda()
    wide[:, :k] = rand((m, k), torch.bfloat16, 16)
    a, w, b = wide[:, :k], rand((n, k), torch.bfloat16, 17), rand((n,), torch.bfloat16, 18)
    product = a.double() @ w.double().t()
    sums = dict(rtol=1e-4, atol=1e-4 * math.sqrt(k))       # float32 sums of k products of numbers about 1
    rounded = dict(rtol=1e-2, atol=1e-2 * math.sqrt(k))    # ... rounded to bfloat16
    torch.testing.assert_close(ops.gemm_tiles(w, ops.TILE_BF16, a, *tile, bias=b).double(), product + b.double(), **rounded)
    if n % 2 == 0:
        gate, up = product[:, : n // 2], product[:, n // 2:]
        torch.testing.assert_close(ops.gemm_tiles(w, ops.TILE_SILU, a, *tile).double(), torch.nn.functional.silu(gate) * up,
                                   rtol=1e-2, atol=1e-2 * k)
    stream = rand((m, n), torch.float32, 19)
    expect = stream.double() + product + b.double()
    ops.gemm_tiles(w, ops.TILE_RESID, a, *tile, bias=b, into=stream)
    torch.testing.assert_close(stream.double(), expect, **sums)
    for parts in (1, 2, 3):
        if (parts - 1) * (-(-(-(-k // parts)) // 64) * 64) < k:  # (every part has some of K)
            got = ops.gemm_tiles(w, ops.TILE_PARTS, a, *tile, bias=b, parts=parts)
            assert got.shape == (parts, m, n)
            torch.testing.assert_close(got.double().sum(0), product + b.double(), **sums)


# (rows, columns, K): a stage or fewer of k, fewer slices than stages, edges of 16 and of the tiles, columns that are no
# multiple of 8, of 4 or of 2.  The loop over whole turns of the stages is entered from twice as many slices as a tile has
# stages (two to five): never, once and several times, with and without slices that are left behind it
@pytest.mark.parametrize("shape", [(1, 32, 64), (63, 64, 128), (65, 130, 192), (129, 256, 320), (200, 99, 448), (257, 100, 512),
                                   (530, 776, 576), (150, 274, 960), (257, 516, 1024), (300, 200, 1088), (131, 72, 2112)])
@pytest.mark.parametrize("tile", [(64, 64), (96, 64), (96, 128), (128, 64), (128, 128), (128, 192), (128, 256), (192, 128),
                                  (192, 192), (192, 256), (256, 128), (256, 160), (256, 256)])
def test_gemm_direct(ops, shape, tile):
    """The products of :func:`test_gemm_tiles` by the kernel whose operands go straight into LDS."""
    m, n, k = shape
    assert tile in ops.DIRECT_SHAPES
    wide = torch.zeros((m, k + 24), dtype=torch.bfloat16).cuda()
    wide[:, :k] = rand((m, k), torch.bfloat16, 16)
    a, w, b = wide[:, :k], rand((n, k), torch.bfloat16, 17), rand((n,), torch.bfloat16, 18)
    product = a.double() @ w.double().t()
    sums = dict(rtol=1e-4, atol=1e-4 * math.sqrt(k))       # float32 sums of k products of numbers about 1
    rounded = dict(rtol=1e-2, atol=1e-2 * math.sqrt(k))    # ... rounded to bfloat16
    run = lambda epilogue, **more: ops.gemm_tiles(w, epilogue, a, *tile, direct=True, **more)  # noqa: E731
    torch.testing.assert_close(run(ops.TILE_BF16, bias=b).double(), product + b.double(), **rounded)
    torch.testing.assert_close(run(ops.TILE_BF16).double(), product, **rounded)
    if n % 2 == 0:
        gate, up = product[:, : n // 2], product[:, n // 2:]
        torch.testing.assert_close(run(ops.TILE_SILU).double(), torch.nn.functional.silu(gate) * up, rtol=1e-2, atol=1e-2 * k)
    stream = rand((m, n), torch.float32, 19)
    expect = stream.double() + product + b.double()
    run(ops.TILE_RESID, bias=b, into=stream)
    torch.testing.assert_close(stream.double(), expect, **sums)
    for parts in (1, 2, 3):
        if (parts - 1) * (-(-(-(-k // parts)) // 64) * 64) < k:  # (every part has some of K)
            got = run(ops.TILE_PARTS, bias=b, parts=parts)
            assert got.shape == (parts, m, n)
            torch.testing.assert_close(got.double().sum(0), product + b.double(), **sums)


def close_to_gated_unit(got, a, w, scale, sums):
    """bf16(silu(g) * u) for g, u = scale x halves of a @ w.T: each row by its own numbers.  A float32 sum of k products is off by at
    most k 2^-24 of its terms' sizes, its scale (of `sums` partial sums, a root, a quotient) by (sums + 8) 2^-24; silu's slope is
    at most 1.1; the exponential and the last rounding to bf16 stay below 2^-8 of the result."""
    n, k = w.shape
    product, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    g, u = (scale * half for half in (product[:, : n // 2], product[:, n // 2:]))
    g_off, u_off = (scale * half * (k + sums + 8) * 2.0 ** -24 for half in (size[:, : n // 2], size[:, n // 2:]))
    expect = torch.nn.functional.silu(g) * u
    bound = 1.1 * g_off * (u.abs() + u_off) + torch.nn.functional.silu(g).abs() * u_off + 2.0 ** -8 * expect.abs() + 1e-30
    assert ((got.double() - expect).abs() <= bound).all()


@pytest.mark.parametrize("shape", [(41, 64, 512), (64, 130, 1088), (65, 100, 2112), (96, 520, 960), (128, 96, 1024), (1, 66, 128)])
@pytest.mark.parametrize("tile", [(64, 64), (96, 64), (128, 64), (96, 128), (128, 128)])
def test_gemm_direct_of_few_rows(ops, shape, tile):
    """Parts that add themselves into a stream (in no fixed order: the bound is that of float32 sums of k products of numbers
    about 1), and the gated unit of rows that lack their 1/rms, whose partial sums of squares come in any number."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.bfloat16, 26), rand((n, k), torch.bfloat16, 27), rand((n,), torch.bfloat16, 28)
    product = a.double() @ w.double().t()
    for parts in (1, 2, 8):
        if (parts - 1) * (-(-(-(-k // parts)) // 64) * 64) >= k:
            continue
        for bias in (None, b):
            stream = rand((m, n), torch.float32, 29)
            expect = stream.double() + product + (0.0 if bias is None else bias.double())
            ops.gemm_tiles(w, ops.TILE_ATOMIC, a, *tile, bias=bias, into=stream, parts=parts, direct=True)
            torch.testing.assert_close(stream.double(), expect, rtol=1e-4, atol=1e-4 * math.sqrt(k))
    for sums in (1, 3, 8, 56, 260):
        sumsq = rand((m, sums), torch.float32, 30).abs() * k
        scale = torch.rsqrt(sumsq.double().sum(1, keepdim=True) / k + 1e-5)
        close_to_gated_unit(ops.gemm_tiles_silu_scaled(w, a, *tile, sumsq, 1e-5), a, w, scale, sums)
    with pytest.raises(ValueError, match="straight into LDS"):
        ops.gemm_tiles(w, ops.TILE_ATOMIC, a, 64, 64, into=stream, parts=1)
    with pytest.raises(ValueError, match="tiles are one of"):
        ops.gemm_tiles(w, ops.TILE_ATOMIC, a, 256, 128, into=stream, parts=1, direct=True)


@pytest.mark.parametrize("rows", [17, 47, 48, 64, 65, 96, 128])
def test_linear_of_some_dozens_of_rows(ops, rows, monkeypatch):
    """What linear() makes of products that may go to the tiles that load straight into LDS, by rows: the form, what comes back, and
    its numbers against 64 bits (a float32 sum of k products is off by at most k 2^-24 of its terms' sizes)."""
    from cie_amd.parts import linear as L
    from cie_amd.parts.norm import RMSNorm

    forms = []
    for name in ("gemm_tiles", "gemm_tiles_silu_scaled"):
        real = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, real=real, scaled="scaled" in name, **k: (forms.append("scaled" if scaled else a[1]), real(*a, **k))[1])
    tiles = rows >= L.FEW_TILE_ROWS

    def product(n, k):
        x, w, b = rand((rows, k), torch.bfloat16, 61), rand((n, k), torch.bfloat16, 62, 0.1), rand((n,), torch.bfloat16, 63)
        return x, w, b, x.double() @ w.double().t(), (x.double().abs() @ w.double().abs().t()) * (k + 8) * 2.0 ** -24

    x, w, b, expect, bound = product(896, 4864)  # a narrow one of a long K: its parts add themselves into the stream
    for bias in (None, b):
        stream = rand((rows, 896), torch.float32, 64)
        whole = stream.double() + expect + (0.0 if bias is None else bias.double())
        assert type(L.linear(x, w, bias, into=stream, sums_parts=True)) is L.Added
        assert ((stream.double() - whole).abs() <= bound + 16 * 2.0 ** -24 * (whole.abs() + expect.abs() + 4)).all()
        # ... or come back
        branch = L.linear(x, w, bias, sums_parts=True)
        assert type(branch) is L.KParts
        assert ((branch.parts.double().sum(0) - expect - (0.0 if bias is None else bias.double())).abs() <= bound + 2.0 ** -22 * (expect.abs() + 4)).all()
    assert forms == [ops.TILE_ATOMIC, ops.TILE_PARTS] * 2 if tiles else not forms
    forms.clear()
    x, w, b, expect, bound = product(2112, 3200)  # one of more than FUSED_SMALL_WEIGHT numbers whose K is too short for that
    for bias in (None, b):
        stream = rand((rows, 2112), torch.float32, 65)
        before = stream.clone()
        branch = L.linear(x, w, bias, into=stream, sums_parts=True)
        assert type(branch) is L.KParts and torch.equal(stream, before)
        assert ((branch.parts.double().sum(0) - expect - (0.0 if bias is None else bias.double())).abs() <= bound + 2.0 ** -22 * (expect.abs() + 4)).all()
    assert forms == [ops.TILE_PARTS] * 2
    forms.clear()
    x, w, _b, _expect, _bound = product(9728, 896)  # a gate, and one of rows without their 1/rms
    one = torch.ones((rows, 1), dtype=torch.float64, device="cuda")
    close_to_gated_unit(L.linear(x, w, epilogue="silu"), x, w, one, 0)
    norm = RMSNorm(896, 1e-6)
    norm.bind({"weight": torch.ones(896, dtype=torch.bfloat16, device="cuda")}, "", torch.bfloat16, "cuda")
    sumsq = torch.rand((rows, 14), generator=torch.Generator().manual_seed(66)).cuda() * torch.arange(1, rows + 1, device="cuda")[:, None]
    scale = torch.rsqrt(sumsq.double().sum(1, keepdim=True) / 896 + 1e-6)
    close_to_gated_unit(L.linear(L.ScaledRows(x, sumsq, 1e-6, x.float(), norm), w, epilogue="silu"), x, w, scale, 14)
    assert forms == [ops.TILE_SILU, "scaled"] if tiles else not forms


@pytest.mark.parametrize("gates", ["of one", "of many sizes", "where 1 + e^-x passes 2^126", "tiny", "at the ends"])
def test_gemm_direct_gate_is_the_division(ops, gates):
    """The gate's quotient in the bits of the tiles that divide: a gate is three bf16 numbers (24 bits) times the column's scale,
    in one group of 8 k, so that either kernel has the same float32 sums."""
    g = torch.Generator().manual_seed(31)
    x = torch.rand(4096, generator=g) * 2 - 1
    if gates == "of many sizes":
        x *= 2.0 ** torch.linspace(-20, 6.4, 4096)
    elif gates == "where 1 + e^-x passes 2^126":
        x = torch.linspace(-88.8, -87.2, 4096)
    elif gates == "tiny":
        x *= 2.0 ** torch.linspace(-132, -100, 4096)
    elif gates == "at the ends":
        x = torch.tensor([3e38, -3e38, 1e38, -1e38, 89.0, -89.0, -104.0, 0.0, -0.0, 2.0 ** 126, -(2.0 ** 126)]).repeat(373)[:4096]
    hi = x.bfloat16()
    mid = torch.where(hi.isinf(), 0.0, x - hi.float()).bfloat16()
    lo = torch.where(hi.isinf(), 0.0, x - hi.float() - mid.float()).bfloat16()
    a = torch.zeros((4096, 64), dtype=torch.bfloat16)
    a[:, 0], a[:, 1], a[:, 2], a[:, 3] = hi, mid, lo, 1.0
    w = torch.zeros((128, 64), dtype=torch.bfloat16)
    w[:64, :3] = (torch.ones(64) if gates != "of many sizes" else 1.0 + torch.arange(64) / 64).bfloat16()[:, None]
    w[64:, 3] = (0.5 + torch.arange(64) / 64).bfloat16()  # (the up halves)
    a, w = a.cuda(), w.cuda()
    got, divided = (ops.gemm_tiles(w, ops.TILE_SILU, a, 128, 64, direct=direct) for direct in (True, False))
    assert torch.equal(got.isnan(), divided.isnan()) and torch.equal(got.nan_to_num(nan=7.0).view(torch.int16), divided.nan_to_num(nan=7.0).view(torch.int16))


@pytest.mark.parametrize("gate", [0.0, 0.5, -0.5, 9.0, -9.0, 40.0, -40.0, -80.0, -87.5, -88.5, 1e30, -1e30, math.inf])
def test_gemm_direct_gate_over_its_range(ops, gate):
    """Each row's one number k = 0 is its gate, k = 1 its up; the result is rounded once to bf16 (half of 2^-7), behind float32
    steps of a few 2^-24; what lies below float32's normal numbers is nothing."""
    a = torch.zeros((130, 64), dtype=torch.bfloat16, device="cuda")
    a[:, 0], a[:, 1] = gate, 1.5
    w = torch.zeros((64, 64), dtype=torch.bfloat16, device="cuda")
    w[:32, 0], w[32:, 1] = 1.0, 1.0
    if math.isinf(gate):
        w[32:, 0], a[:, 1] = 1.0, 0.0  # (no 0 x inf in the up columns)
    got = ops.gemm_tiles(w, ops.TILE_SILU, a, 64, 64, direct=True).double()
    x = a[0, 0].double().cpu()
    expect = x * torch.sigmoid(x) * (x if math.isinf(gate) else 1.5)
    if math.isinf(gate):
        assert torch.isinf(got).all() and (got > 0).all()
    else:
        assert (got.cpu() - expect).abs().max() <= expect.abs() * 2.0 ** -7.99 + 2.0 ** -126


@pytest.mark.parametrize("heads", [(4, 2, 128), (3, 1, 96), (14, 2, 64), (2, 2, 32)])
@pytest.mark.parametrize("tile", [(64, 64), (96, 64), (96, 128), (128, 64), (128, 128), (128, 192), (128, 256), (192, 128),
                                  (192, 192), (192, 256), (256, 128), (256, 160), (256, 256)])
@pytest.mark.parametrize("k,rotate,write,biased", [(192, True, True, True), (1088, True, True, False), (1024, False, True, True),
                                                   (576, True, False, True)])
def test_gemm_direct_rope(ops, heads, tile, k, rotate, write, biased):
    """... and its q/k/v epilogue, whose rows' places are asked for between the last slices, behind none, one and several
    turns of the stages: the bits of the plain one and the rotation's kernel behind it."""
    q_heads, kv_heads, dim = heads
    m, page, n = 300, 8, (heads[0] + 2 * heads[1]) * heads[2]
    a, w = rand((m, k), torch.bfloat16, 20), rand((n, k), torch.bfloat16, 21)
    b = rand((n,), torch.bfloat16, 22) if biased else None
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    positions, seqs, slots = as_dev(list(range(3, 203)) + list(range(100))), as_dev([0] * 200 + [1] * 100), as_dev([2, 0])
    table = torch.randperm(96, generator=torch.Generator().manual_seed(23)).to(torch.int32).reshape(3, 32).cuda()
    cos, sin = rand((256, dim // 2), torch.float32, 24), rand((256, dim // 2), torch.float32, 25)
    pools = [torch.zeros((96, kv_heads, page, dim), dtype=torch.bfloat16).cuda(), torch.zeros((96, kv_heads, dim, page), dtype=torch.bfloat16).cuda()]
    plain_pools = [p.clone() for p in pools]
    how = dict(rotate=rotate, write_kv=write)
    got = ops.gemm_tiles_rope(w, a, b, cos, sin, positions, seqs, slots, table, *pools, q_heads, kv_heads, dim, *tile, direct=True, **how)
    expect = ops.gemm_tiles(w, ops.TILE_BF16, a, *tile, bias=b, direct=True)
    ops.rope_kv_write(expect, cos, sin, positions, seqs, slots, table, *plain_pools, q_heads, kv_heads, dim, **how)
    assert torch.equal(got[:, : q_heads * dim], expect[:, : q_heads * dim])
    assert all(torch.equal(x, y) for x, y in zip(pools, plain_pools)) and bool(pools[0].any()) == write


@pytest.mark.parametrize("heads", [(4, 2, 128), (3, 1, 96), (14, 2, 64), (2, 2, 32)])
@pytest.mark.parametrize("tile", [(64, 64), (128, 64), (128, 128), (128, 256)])
@pytest.mark.parametrize("rotate,write", [(True, True), (False, True), (True, False)])
def test_gemm_tiles_rope(ops, heads, tile, rotate, write):
    """The q/k/v product whose epilogue rotates and writes the cache: the bits of the plain epilogue and the rotation's
    kernel behind it, with rows of two sequences in pages that are not in order."""
    q_heads, kv_heads, dim = heads
    m, k, page = 133, 200, 8
    n = (q_heads + 2 * kv_heads) * dim
    a, w, b = rand((m, k), torch.bfloat16, 20), rand((n, k), torch.bfloat16, 21), rand((n,), torch.bfloat16, 22)
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    first = 70
    positions = as_dev(list(range(5, 5 + first)) + list(range(m - first)))
    seqs, slots = as_dev([0] * first + [1] * (m - first)), as_dev([2, 0])
    table = torch.randperm(48, generator=torch.Generator().manual_seed(23)).to(torch.int32).reshape(3, 16).cuda()
    cos, sin = rand((128, dim // 2), torch.float32, 24), rand((128, dim // 2), torch.float32, 25)
    pools = [torch.zeros((48, kv_heads, page, dim), dtype=torch.bfloat16).cuda(), torch.zeros((48, kv_heads, dim, page), dtype=torch.bfloat16).cuda()]
    plain_pools = [p.clone() for p in pools]
    got = ops.gemm_tiles_rope(w, a, b, cos, sin, positions, seqs, slots, table, *pools, q_heads, kv_heads, dim, *tile,
                              rotate=rotate, write_kv=write)
    expect = ops.gemm_tiles(w, ops.TILE_BF16, a, *tile, bias=b)
    ops.rope_kv_write(expect, cos, sin, positions, seqs, slots, table, *plain_pools, q_heads, kv_heads, dim, rotate=rotate, write_kv=write)
    assert torch.equal(got[:, : q_heads * dim], expect[:, : q_heads * dim])
    assert all(torch.equal(x, y) for x, y in zip(pools, plain_pools))


@pytest.mark.parametrize("dtype,hidden", [(torch.bfloat16, 64), (torch.bfloat16, 100), (torch.float32, 96)])
@pytest.mark.parametrize("parts", [1, 3, 6])
def test_add_rmsnorm_sums_parts(ops, dtype, hidden, parts):
    """Parts of a branch join the stream in order, in the whole step's form and for chosen rows."""
    stream, weight = rand((37, hidden), torch.float32, 26), rand((hidden,), dtype, 27)
    pieces = rand((parts, 37, hidden), torch.float32, 28)
    whole = stream.clone()
    for piece in pieces:
        whole += piece
    expect = ops.add_rmsnorm(whole.clone(), None, weight, 1e-6, dtype)
    rows = torch.tensor([36, 0, 5], dtype=torch.int32).cuda()
    chosen = ops.add_rmsnorm(stream, None, weight, 1e-6, dtype, rows=rows, parts=pieces)
    assert torch.equal(chosen, ops.add_rmsnorm(whole.clone(), None, weight, 1e-6, dtype, rows=rows))
    assert torch.equal(ops.add_rmsnorm(stream, None, weight, 1e-6, dtype, parts=pieces), expect)
    assert torch.equal(stream, whole)


@pytest.mark.parametrize("hidden", [8192, 8200, 16384])
@pytest.mark.parametrize("dtype", DTYPES)
def test_add_rmsnorm_of_wide_rows(ops, dtype, hidden):
    """Rows of which a thread has one piece of eight, and two (the second waits in LDS): a branch, parts, chosen rows."""
    stream, weight, branch = rand((5, hidden), torch.float32, 29), rand((hidden,), dtype, 30), rand((5, hidden), dtype, 31)
    pieces = rand((3, 5, hidden), torch.float32, 32)
    added = stream + branch.float()
    whole = added + pieces[0] + pieces[1] + pieces[2]
    rows = torch.tensor([4, 0], dtype=torch.int32).cuda()
    for extra, total in ((None, added), (pieces, whole)):
        expect = plain_qwen2.rms_norm(total, weight.float(), 1e-6)
        chosen = ops.add_rmsnorm(stream, branch, weight, 1e-6, dtype, rows=rows, parts=extra)
        torch.testing.assert_close(chosen.float(), expect[[4, 0]], **tol(dtype))
        left = stream.clone()
        torch.testing.assert_close(ops.add_rmsnorm(left, branch, weight, 1e-6, dtype, parts=extra).float(), expect, **tol(dtype))
        assert torch.equal(left, total)


def build_cache(dtype, lengths, kv_heads, head_dim, page_size, seed, shuffle=True):
    """Random keys/values for sequences of the given lengths, scattered over the
    pages of a pool in a shuffled order.  Returns pools, block table and the
    dense per-sequence tensors."""
    g = torch.Generator().manual_seed(seed)
    pages_per = [-(-n // page_size) for n in lengths]
    total = sum(pages_per) + 3
    order = torch.randperm(total, generator=g).tolist() if shuffle else list(range(total))
    width = max(pages_per) + 2
    table = torch.zeros((len(lengths) + 2, width), dtype=torch.int32)
    slots = list(range(len(lengths), 0, -1))  # slot != sequence index, on purpose
    k_pool = torch.zeros((total, kv_heads, page_size, head_dim))
    v_pool = torch.zeros_like(k_pool)
    dense = []
    cursor = 0
    for s, n in enumerate(lengths):
        k = torch.randn((n, kv_heads, head_dim), generator=g)
        v = torch.randn((n, kv_heads, head_dim), generator=g)
        k, v = k.to(dtype).float(), v.to(dtype).float()
        dense.append((k, v))
        for p in range(pages_per[s]):
            page = order[cursor]
            cursor += 1
            table[slots[s], p] = page
            rows = slice(p * page_size, min((p + 1) * page_size, n))
            count = rows.stop - rows.start
            k_pool[page, :, :count] = k[rows].transpose(0, 1)
            v_pool[page, :, :count] = v[rows].transpose(0, 1)
    # values are cached transposed: [page, head, head_dim, page_size]
    v_pool = v_pool.transpose(2, 3).contiguous()
    return k_pool.to(dtype).cuda(), v_pool.to(dtype).cuda(), table.cuda(), slots, dense


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geometry", [(4, 2, 16, 16), (16, 2, 128, 16), (6, 6, 48, 8), (8, 1, 64, 32), (5, 5, 80, 4)])
def test_paged_attention_generic(ops, dtype, geometry):
    """Ragged batch: a long prompt portion with context, a fresh prompt, single
    decode tokens at page edges.  Context/query sizes follow the reference's
    matrix (tests/remote_ragged_gpu_tests.py:118-121) scaled down."""
    q_heads, kv_heads, head_dim, page_size = geometry
    contexts = [0, 15, 16, 17, 127, 300, 1]
    q_lens = [7, 1, 1, 2, 16, 1, 33]
    lengths = [c + q for c, q in zip(contexts, q_lens)]
    k_pool, v_pool, table, slots, dense = build_cache(dtype, lengths, kv_heads, head_dim, page_size, seed=20)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(21)
    positions, seq_of_token, expected, qs = [], [], [], []
    for s, (c, n) in enumerate(zip(contexts, q_lens)):
        q = (torch.randn((n, q_heads, head_dim), generator=g) * 2).to(dtype).float()
        qs.append(q)
        positions += list(range(c, c + n))
        seq_of_token += [s] * n
        k, v = dense[s]
        expected.append(plain_qwen2.causal_attention(q, k, v, scale, past_len=c))
    q_all = torch.cat(qs).reshape(len(positions), q_heads * head_dim)
    stride = (q_heads + 2 * kv_heads) * head_dim  # as if q sat inside a fused qkv buffer
    buffer = torch.zeros((len(positions), stride))
    buffer[:, : q_heads * head_dim] = q_all
    buffer = buffer.to(dtype).cuda()
    out = ops.paged_attention_generic(
        buffer, stride, k_pool, v_pool, table, torch.tensor(positions, dtype=torch.int32).cuda(),
        torch.tensor(seq_of_token, dtype=torch.int32).cuda(), torch.tensor(slots, dtype=torch.int32).cuda(),
        len(positions), q_heads, kv_heads, head_dim, None, scale)
    torch.testing.assert_close(out.float().cpu(), torch.cat(expected), **tol(dtype))


def run_f32(ops, q_all, contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads, head_dim, window, scale, per_tile,
            turns):
    """Drive the float32 attention of the matrix cores: tiles of ``per_tile`` tokens, whole or in blocks of keys."""
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    loc = [sum(q_lens[:i]) for i in range(len(q_lens) + 1)]
    tiles = [(s, first) for s, n in enumerate(q_lens) for first in range(0, n, per_tile)]
    stride = (q_heads + 2 * kv_heads) * head_dim
    buffer = torch.zeros((sum(q_lens), stride)).cuda()
    buffer[:, : q_heads * head_dim] = q_all.cuda()
    out = torch.full((sum(q_lens), q_heads * head_dim), float("nan")).cuda()
    spaces = {}
    if turns:
        blocks, rows = max(-(-(c + n) // 64) for c, n in zip(contexts, q_lens)), per_tile * (q_heads // kv_heads)
        units = len(tiles) * kv_heads * blocks * rows
        spaces = dict(turns=turns, blocks=blocks, part_o=torch.full((units * head_dim,), float("nan")).cuda(),
                      part_ml=torch.full((units * 2,), float("nan")).cuda())
    ops.paged_attention_f32(buffer, stride, k_pool, v_pool, table, as_dev([s for s, _ in tiles]), as_dev([q for _, q in tiles]),
                            len(tiles), as_dev(slots), as_dev(contexts), as_dev(q_lens), as_dev(loc), out, q_heads, kv_heads,
                            head_dim, window, scale, per_tile, **spaces)
    return out.cpu()


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (3, 1, 32, 4), (14, 2, 64, 8), (16, 1, 96, 32), (64, 1, 32, 128),
                                      (40, 8, 128, 64)])
@pytest.mark.parametrize("window", [None, 1, 50, 300])
def test_paged_attention_f32(ops, geometry, window):
    """The float32 attention of the matrix cores on the ragged batch of the bfloat16 forms: near the plain
    implementation, and the same bits whole or in blocks, in large tiles or token by token."""
    q_heads, kv_heads, head_dim, page_size = geometry
    contexts = [0, 15, 16, 17, 127, 511, 1, 40, 100]
    q_lens = [7, 1, 2, 16, 1, 33, 64, 5, 200]
    lengths = [c + q for c, q in zip(contexts, q_lens)]
    k_pool, v_pool, table, slots, dense = build_cache(torch.float32, lengths, kv_heads, head_dim, page_size, seed=70)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(71)
    qs, expected = [], []
    for s, (c, n) in enumerate(zip(contexts, q_lens)):
        q = torch.randn((n, q_heads, head_dim), generator=g) * 2
        qs.append(q.reshape(n, -1))
        expected.append(plain_qwen2.causal_attention(q, *dense[s], scale, past_len=c, window=window))
    most = 64 // (q_heads // kv_heads)
    outs = [run_f32(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads, head_dim, window,
                    scale, per_tile, turns) for per_tile, turns in ((most, 0), (1, 0), (most, 1), (most, 3), (1, 16))]
    torch.testing.assert_close(outs[0], torch.cat(expected), **tol(torch.float32))
    assert all(torch.equal(out, outs[0]) for out in outs[1:])


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (3, 1, 96, 8), (64, 1, 32, 4)])
@pytest.mark.parametrize("window", [None, 1, 65, 500])
@pytest.mark.parametrize("captured", [False, True])
def test_attend_float32_in_rounds(ops, monkeypatch, geometry, window, captured):
    """Single tokens (and two prompt portions behind them) whose blocks exceed the workspace: an eager step runs as many
    rounds as its lengths need, a step with a captured step's plan one round and whole tiles behind it, and with room for
    every tile's bound none of both: all the bits of the whole form."""
    from cie_amd.engine.batch import PagedView, StepBatch
    from cie_amd.engine.graphs import StaticPlan
    from cie_amd.parts import attention

    q_heads, kv_heads, head_dim, page_size = geometry
    contexts = [0, 62, 63, 1000, 1500, 130, 2000, 700, 64, 100]
    q_lens = [1] * 8 + [40, 7]
    k_pool, v_pool, table, slots, _ = build_cache(torch.float32, [c + n for c, n in zip(contexts, q_lens)], kv_heads, head_dim,
                                                  page_size, seed=76)
    view = PagedView(k_pool, v_pool, table, page_size)
    qkv = rand((sum(q_lens), (q_heads + 2 * kv_heads) * head_dim), torch.float32, 77)
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    loc = [sum(q_lens[:i]) for i in range(len(q_lens) + 1)]
    tokens = [(s, t) for s, n in enumerate(q_lens) for t in range(n)]
    plan = StaticPlan(None, None, as_dev([2001]), 4096, decode_rows=8) if captured else None

    def attend():
        batch = StepBatch(tokens=len(tokens), sequences=len(q_lens), token_ids=as_dev([0] * len(tokens)),
                          positions=as_dev([contexts[s] + t for s, t in tokens]), seq_of_token=as_dev([s for s, _ in tokens]),
                          seq_slot=as_dev(slots), seq_start=as_dev(contexts), seq_q_len=as_dev(q_lens), q_start_loc=as_dev(loc),
                          logit_rows=as_dev([0]), host_slots=slots, host_starts=[0] * 10 if captured else contexts,
                          host_q_lens=q_lens, static_plan=plan)
        return attention.attend(qkv, batch, view, q_heads, kv_heads, head_dim, window, 0.1)

    calls, launch = [], ops.paged_attention_f32
    monkeypatch.setattr(ops, "paged_attention_f32", lambda *a, **k: (calls.append((k.get("capacity", 0), k.get("round", 0), k.get("turns", 0))), launch(*a, **k)))
    roomy = attend()
    assert not any(capacity for capacity, _, _ in calls)
    calls.clear()
    monkeypatch.setattr(ops, "F32_WORKSPACE_BYTES", 1)  # (the least there is: places for one tile's bound a round)
    tight = attend()
    rounds = [(turn, turns > 0) for capacity, turn, turns in calls if capacity]
    if captured:
        assert rounds in ([(0, True), (1, False)], [(0, True), (1, False)] * 2)  # (the portions may be cut too)
    else:
        assert rounds[0] == (0, True) and all(turn in (0, last + 1) and cut for (last, _), (turn, cut) in zip(rounds, rounds[1:]))
        assert len(rounds) > 2 or window is not None
    monkeypatch.setattr(attention, "F32_WHOLE_KEYS", 1 << 20)
    whole = attend()
    assert torch.equal(roomy, whole) and torch.equal(tight, whole)


@pytest.mark.parametrize("turns", [0, 2])
def test_paged_attention_f32_odd_values_reach_the_rows_that_see_them(ops, turns):
    """An infinity and a NaN among the cached values: the rows before them in the same tile stay as they are, the rows
    that see them have the generic kernel's infinities and NaN."""
    q_heads, kv_heads, head_dim, page_size, n = 16, 2, 128, 16, 100
    k_pool, v_pool, table, slots, _ = build_cache(torch.float32, [n], kv_heads, head_dim, page_size, seed=74)
    odd = v_pool.clone()
    page = int(table[slots[0], 3])
    odd[page, :, 5, 2] = float("inf")
    odd[page, 0, 7, 3] = float("nan")
    q = rand((n, q_heads * head_dim), torch.float32, 75)
    run = lambda values: run_f32(ops, q, [0], [n], k_pool, values, table, slots, q_heads, kv_heads, head_dim, None, 0.1, 8, turns)  # noqa: E731
    plain, got = run(v_pool), run(odd)
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    buffer = torch.zeros((n, (q_heads + 2 * kv_heads) * head_dim)).cuda()
    buffer[:, : q_heads * head_dim] = q
    generic = ops.paged_attention_generic(buffer, buffer.shape[1], k_pool, odd, table, as_dev(list(range(n))), as_dev([0] * n),
                                          as_dev(slots), n, q_heads, kv_heads, head_dim, None, 0.1).cpu()
    assert torch.equal(got[:50], plain[:50])
    assert torch.equal(torch.isnan(got), torch.isnan(generic)) and torch.equal(torch.isinf(got), torch.isinf(generic))
    finite = torch.isfinite(generic)
    assert not finite.all()
    torch.testing.assert_close(got[finite], generic[finite], **tol(torch.float32))


def run_mfma(ops, q_all, contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads, head_dim, window,
             scale, per_tile, row_tiles, n_splits=1, keys_per_split=0, decode_only=None, tile_waves=1,
             max_context_dev=None):
    """Drive the matrix-core kernel the way the attention part does: tiles of
    ``per_tile`` tokens for the chosen sequences; returns [tokens, Hq*D] (rows of
    sequences that were not chosen stay zero)."""
    tokens = sum(q_lens)
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    loc = [0]
    for n in q_lens:
        loc.append(loc[-1] + n)
    tile_seq, tile_q0 = [], []
    for s, n in enumerate(q_lens):
        if decode_only is not None and (n == 1) != decode_only:
            continue
        for first in range(0, n, per_tile):
            tile_seq.append(s)
            tile_q0.append(first)
    stride = (q_heads + 2 * kv_heads) * head_dim
    buffer = torch.zeros((tokens, stride))
    buffer[:, : q_heads * head_dim] = q_all
    buffer = buffer.to(torch.bfloat16).cuda()
    out = torch.zeros((tokens, q_heads * head_dim), dtype=torch.bfloat16).cuda()
    part_o = part_ml = None
    if n_splits > 1:
        units = len(tile_seq) * kv_heads * n_splits
        part_o = torch.full((units * 16 * row_tiles * head_dim,), float("nan")).cuda()
        part_ml = torch.full((units * 16 * row_tiles * 2,), float("nan")).cuda()
    ops.paged_attention_mfma(buffer, stride, k_pool, v_pool, table, as_dev(tile_seq), as_dev(tile_q0), len(tile_seq),
                             as_dev(slots), as_dev(contexts), as_dev(q_lens), as_dev(loc), out, q_heads, kv_heads,
                             head_dim, window, scale, per_tile, row_tiles, n_splits=n_splits,
                             keys_per_split=keys_per_split, part_o=part_o, part_ml=part_ml, tile_waves=tile_waves,
                             max_context_dev=max_context_dev)
    return out.float().cpu()


# (query heads, KV heads, head size, page size); 28/4 and 40/8 are the head counts of the 7B and 14B shapes
MFMA_GEOMETRY = [(16, 2, 128, 16), (4, 2, 32, 8), (3, 1, 32, 8), (6, 6, 64, 4), (16, 1, 96, 32), (12, 4, 256, 16),
                 (28, 4, 128, 16), (40, 8, 128, 64)]


@pytest.mark.parametrize("geometry", MFMA_GEOMETRY)
@pytest.mark.parametrize("row_tiles,tile_waves", [(1, 1), (2, 1), (4, 1), (1, 4), (2, 4), (4, 4), (8, 8), (4, 8)])
def test_paged_attention_mfma_ragged(ops, geometry, row_tiles, tile_waves):
    """The tiled forms (one wave per tile; four waves that share a tile's keys; eight waves per tile of
    128 rows with keys and values in LDS) on
    a ragged batch (reference matrix of contexts and query lengths,
    tests/remote_ragged_gpu_tests.py:118-121): portions with and without context,
    lengths that do not fill a tile, single tokens at page edges."""
    q_heads, kv_heads, head_dim, page_size = geometry
    group = q_heads // kv_heads
    if (group > 16 * row_tiles or (head_dim == 256 and row_tiles > (2 if tile_waves == 1 else 1))):
        pytest.skip("more heads per group than rows, or a variant the kernel refuses")
    if tile_waves >= 4:
        page_size = max(page_size, 16)  # these forms keep the 16 keys of a product in one page
    contexts = [0, 15, 16, 17, 127, 511, 1, 40, 100]
    q_lens = [7, 1, 2, 16, 1, 33, 64, 5, 200]
    lengths = [c + q for c, q in zip(contexts, q_lens)]
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=70)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(71)
    qs, expected = [], []
    for s, (c, n) in enumerate(zip(contexts, q_lens)):
        q = (torch.randn((n, q_heads, head_dim), generator=g) * 2).to(torch.bfloat16).float()
        qs.append(q.reshape(n, -1))
        expected.append(plain_qwen2.causal_attention(q, *dense[s], scale, past_len=c))
    per_tile = (16 * row_tiles) // group
    out = run_mfma(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads, head_dim,
                   None, scale, per_tile, row_tiles, tile_waves=tile_waves)
    torch.testing.assert_close(out, torch.cat(expected), **tol(torch.bfloat16))


@pytest.mark.parametrize("geometry", MFMA_GEOMETRY)
@pytest.mark.parametrize("splits", [(1, 0), (3, 704), (16, 128), (64, 32)])
@pytest.mark.parametrize("tile_waves", [1, 4])
def test_paged_attention_mfma_decode_splits(ops, geometry, splits, tile_waves):
    """Single tokens over contexts up to 2047 (boundary lengths of
    tests/remote_gpu_tests.py:204), the keys cut into parts that are merged;
    parts beyond a short context are empty.  With one wave per part and with four
    (a part of 32 keys then leaves three of them without a key)."""
    q_heads, kv_heads, head_dim, page_size = geometry
    if tile_waves == 4:
        page_size = max(page_size, 16)
    n_splits, per_split = splits
    contexts = [0, 1, 15, 16, 17, 127, 128, 129, 1000, 2047]
    q_lens = [1] * len(contexts)
    lengths = [c + 1 for c in contexts]
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=72)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(73)
    qs, expected = [], []
    for s, c in enumerate(contexts):
        q = (torch.randn((1, q_heads, head_dim), generator=g) * 2).to(torch.bfloat16).float()
        qs.append(q.reshape(1, -1))
        expected.append(plain_qwen2.causal_attention(q, *dense[s], scale, past_len=c))
    out = run_mfma(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads, head_dim,
                   None, scale, 1, 1, n_splits=n_splits, keys_per_split=per_split, tile_waves=tile_waves)
    torch.testing.assert_close(out, torch.cat(expected), **tol(torch.bfloat16))
    if n_splits > 1:
        # as in a captured step: the size of a part is derived on the device from the longest context,
        # here once the true one and once a loose bound
        for longest in (max(lengths), 3000):
            out = run_mfma(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads,
                           head_dim, None, scale, 1, 1, n_splits=n_splits, tile_waves=tile_waves,
                           max_context_dev=torch.tensor([longest], dtype=torch.int32).cuda())
            torch.testing.assert_close(out, torch.cat(expected), **tol(torch.bfloat16))


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (6, 2, 32, 16), (5, 5, 64, 32)])
@pytest.mark.parametrize("row_tiles", [1, 2, 4, 8, -4])
@pytest.mark.parametrize("splits", [(3, 512), (5, 256), (9, 128)])
def test_paged_attention_mfma_prompt_portions_with_their_keys_cut(ops, geometry, row_tiles, splits):
    """Portions of prompts behind long contexts, tiles of 16 to 128 rows whose keys are cut into
    parts (some of them empty for the shorter sequences, some ending inside the portion); tiles of 128
    rows, and of 64 where ``row_tiles`` is given as -4, in the form that shares keys and values through LDS."""
    q_heads, kv_heads, head_dim, page_size = geometry
    through_lds = row_tiles in (8, -4)
    row_tiles = abs(row_tiles)
    group = q_heads // kv_heads
    if group > 16 * row_tiles:
        pytest.skip("the group does not fit the tile")
    n_splits, per_split = splits
    contexts, q_lens = [1000, 0, 300, 37], [40, 70, 9, 33]
    lengths = [c + n for c, n in zip(contexts, q_lens)]
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=82)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(83)
    qs, expected = [], []
    for s, (c, n) in enumerate(zip(contexts, q_lens)):
        q = (torch.randn((n, q_heads, head_dim), generator=g) * 2).to(torch.bfloat16).float()
        qs.append(q.reshape(n, -1))
        expected.append(plain_qwen2.causal_attention(q, *dense[s], scale, past_len=c))
    per_tile = (16 * row_tiles) // group
    out = run_mfma(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads, head_dim,
                   None, scale, per_tile, row_tiles, n_splits=n_splits, keys_per_split=per_split,
                   tile_waves=8 if through_lds else 4)
    torch.testing.assert_close(out, torch.cat(expected), **tol(torch.bfloat16))


@pytest.mark.parametrize("window", [5, 32, 100])
def test_paged_attention_mfma_window(ops, window):
    q_heads, kv_heads, head_dim = 4, 2, 64
    contexts = [0, 90, 300, 33]
    q_lens = [40, 1, 17, 1]
    lengths = [c + q for c, q in zip(contexts, q_lens)]
    scale = 1.0 / math.sqrt(head_dim)
    for page_size, variants in ((8, ((1, 1),)), (16, ((4, 1), (4, 2), (8, 8), (8, 4))), (64, ((4, 4), (8, 8), (8, 4)))):
        k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=74)
        g = torch.Generator().manual_seed(75)
        qs, expected = [], []
        for s, (c, n) in enumerate(zip(contexts, q_lens)):
            q = (torch.randn((n, q_heads, head_dim), generator=g) * 2).to(torch.bfloat16).float()
            qs.append(q.reshape(n, -1))
            expected.append(plain_qwen2.causal_attention(q, *dense[s], scale, past_len=c, window=window))
        want = torch.cat(expected)
        for tile_waves, row_tiles in variants:
            tiled = run_mfma(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads,
                             head_dim, window, scale, 8 * row_tiles, row_tiles, tile_waves=tile_waves)  # (groups of two)
            torch.testing.assert_close(tiled, want, **tol(torch.bfloat16))
        rows = [40, 58]  # the two single-token sequences
        for tile_waves in ((1,) if page_size < 16 else (1, 4)):
            split = run_mfma(ops, torch.cat(qs), contexts, q_lens, k_pool, v_pool, table, slots, q_heads, kv_heads,
                             head_dim, window, scale, 1, 1, n_splits=4, keys_per_split=32, decode_only=True,
                             tile_waves=tile_waves)
            torch.testing.assert_close(split[rows], want[rows], **tol(torch.bfloat16))


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (16, 1, 96, 32), (12, 4, 256, 16), (6, 6, 64, 16)])
def test_paged_attention_mfma_decode_hundreds_of_parts(ops, geometry):
    """Two single tokens over 9,000 and 3,100 keys cut into parts of 32 and 64 keys: the merge sums
    up to 282 parts per row, most of them in its loop behind the parts it fetches early; one far key
    carries the weight of the first sequence, so a part lost or counted twice shows."""
    q_heads, kv_heads, head_dim, page_size = geometry
    group = q_heads // kv_heads
    lengths, far = [9000, 3100], 7777
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=91)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(92)
    qs = [torch.stack([dense[0][0][far, h // group] * 2.0 for h in range(q_heads)])[None].to(torch.bfloat16).float(),
          (torch.randn((1, q_heads, head_dim), generator=g) * 2).to(torch.bfloat16).float()]
    contexts = [n - 1 for n in lengths]
    expected = torch.cat([plain_qwen2.causal_attention(q, *dense[s], scale, past_len=contexts[s])
                          for s, q in enumerate(qs)])
    for n_splits, per_split, tile_waves in [(282, 32, 1), (141, 64, 1), (71, 128, 4)]:
        out = run_mfma(ops, torch.cat([q.reshape(1, -1) for q in qs]), contexts, [1, 1], k_pool, v_pool, table, slots,
                       q_heads, kv_heads, head_dim, None, scale, 1, 1, n_splits=n_splits, keys_per_split=per_split,
                       tile_waves=tile_waves)
        torch.testing.assert_close(out, expected, **tol(torch.bfloat16))


@pytest.mark.parametrize("joined_rows", [0, 32])
@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (28, 4, 128, 16), (6, 2, 64, 32)])
def test_attention_planning_of_steps_with_single_tokens_beside_portions(ops, geometry, joined_rows, monkeypatch):
    """The planner of the attention part on a step as a scheduler makes it: four sequences that bring one
    token over 1 to 3,001 keys beside two prompt portions (one behind 2,000 cached keys), once with two
    launches (decode form and prompt form) and once with the single tokens riding in the prompt form's
    launch, against plain attention per sequence."""
    from cie_amd.engine.batch import PagedView, StepBatch
    from cie_amd.parts import attention

    monkeypatch.setattr(attention, "JOINED_DECODE_ROWS", joined_rows)
    q_heads, kv_heads, head_dim, page_size = geometry
    contexts = [0, 31, 600, 3000, 100, 2000]
    q_lens = [1, 1, 1, 1, 40, 70]
    lengths = [c + n for c, n in zip(contexts, q_lens)]
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=95)
    scale = 1.0 / math.sqrt(head_dim)
    g = torch.Generator().manual_seed(96)
    total = sum(q_lens)
    width = (q_heads + 2 * kv_heads) * head_dim
    qkv = torch.zeros((total, width), dtype=torch.bfloat16)
    expected, row = [], 0
    for s, (c, n) in enumerate(zip(contexts, q_lens)):
        q = (torch.randn((n, q_heads, head_dim), generator=g) * 2).to(torch.bfloat16)
        qkv[row: row + n, : q_heads * head_dim] = q.reshape(n, -1)
        expected.append(plain_qwen2.causal_attention(q.float(), *dense[s], scale, past_len=c))
        row += n
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")  # noqa: E731
    loc = [0]
    for n in q_lens:
        loc.append(loc[-1] + n)
    positions = [c + i for c, n in zip(contexts, q_lens) for i in range(n)]
    seq_of_token = [s for s, n in enumerate(q_lens) for _ in range(n)]
    batch = StepBatch(tokens=total, sequences=len(q_lens), token_ids=as_dev([0] * total), positions=as_dev(positions),
                      seq_of_token=as_dev(seq_of_token), seq_slot=as_dev(slots), seq_start=as_dev(contexts),
                      seq_q_len=as_dev(q_lens), q_start_loc=as_dev(loc), logit_rows=as_dev([0]),
                      host_slots=list(slots), host_starts=contexts, host_q_lens=q_lens)
    view = PagedView(k_pool, v_pool, table, page_size)
    launches = []
    real = ops.paged_attention_mfma
    monkeypatch.setattr(ops, "paged_attention_mfma", lambda *a, **k: (launches.append(k["tokens_per_tile"]), real(*a, **k))[1])
    out = attention.attend(qkv.cuda(), batch, view, q_heads, kv_heads, head_dim, None, scale)
    assert len(launches) == (1 if joined_rows else 2), launches
    torch.testing.assert_close(out.float().cpu(), torch.cat(expected), **tol(torch.bfloat16))


@pytest.mark.parametrize("alone", [0.0, 99.0])
@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (6, 2, 64, 32), (7, 1, 128, 16)])
@pytest.mark.parametrize("portions", [((613, 0),), ((17, 1500), (130, 911), (2, 63)), ((64, 0), (65, 64), (1, 700)), ((33, 2100),)])
def test_attention_of_portions_with_little_beside_them(ops, geometry, portions, alone, monkeypatch):
    """Portions of few tiles in the form that shares keys and values through LDS (cut and whole) and in the other one: parts of
    a tile, of a page and of 64 keys, each against plain attention per sequence."""
    from cie_amd.engine.batch import PagedView, StepBatch
    from cie_amd.parts import attention

    monkeypatch.setattr(attention, "ALONE_TILES", alone)
    monkeypatch.setattr(attention, "ALONE_TILE_KEYS", 1 << 40)
    monkeypatch.setattr(attention, "JOINED_DECODE_ROWS", 0)
    q_heads, kv_heads, head_dim, page_size = geometry
    q_lens, contexts = [n for n, _c in portions], [c for _n, c in portions]
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, [c + n for n, c in portions], kv_heads, head_dim, page_size, seed=97)
    scale, total = 1.0 / math.sqrt(head_dim), sum(q_lens)
    qkv = torch.zeros((total, (q_heads + 2 * kv_heads) * head_dim), dtype=torch.bfloat16)
    q = (torch.randn((total, q_heads, head_dim), generator=torch.Generator().manual_seed(98)) * 2).to(torch.bfloat16)
    qkv[:, : q_heads * head_dim] = q.reshape(total, -1)
    loc = [sum(q_lens[:s]) for s in range(len(q_lens) + 1)]
    expected = torch.cat([plain_qwen2.causal_attention(q[loc[s]: loc[s + 1]].float(), *dense[s], scale, past_len=contexts[s])
                          for s in range(len(q_lens))])
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")  # noqa: E731
    batch = StepBatch(tokens=total, sequences=len(q_lens), token_ids=as_dev([0] * total),
                      positions=as_dev([c + i for n, c in portions for i in range(n)]),
                      seq_of_token=as_dev([s for s, n in enumerate(q_lens) for _ in range(n)]), seq_slot=as_dev(slots),
                      seq_start=as_dev(contexts), seq_q_len=as_dev(q_lens), q_start_loc=as_dev(loc), logit_rows=as_dev([0]),
                      host_slots=list(slots), host_starts=contexts, host_q_lens=q_lens)
    forms = []
    real = ops.paged_attention_mfma
    monkeypatch.setattr(ops, "paged_attention_mfma", lambda *a, **k: (forms.append(k["tile_waves"]), real(*a, **k))[1])
    out = attention.attend(qkv.cuda(), batch, PagedView(k_pool, v_pool, table, page_size), q_heads, kv_heads, head_dim, None, scale)
    tiles = -(-sum(n for n in q_lens if n > 1) * (q_heads // kv_heads) // 64) * kv_heads
    assert (ops.PROMPT_WAVES in forms) == (alone == 0.0 or tiles >= 0.75 * ops.compute_units())
    torch.testing.assert_close(out.float().cpu(), expected.reshape(total, -1), **tol(torch.bfloat16))


def test_paged_attention_mfma_far_key(ops):
    """One key among two thousand carries the weight: output = its value row, in
    the tiled form and in every split layout."""
    q_heads, kv_heads, head_dim, page_size = 16, 2, 128, 16
    length, far = 2000, 1234
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, [length], kv_heads, head_dim, page_size, seed=76)
    k, v = dense[0]
    q = torch.stack([k[far, h // 8] * 2.0 for h in range(q_heads)])[None].to(torch.bfloat16).float()
    scale = 1.0 / math.sqrt(head_dim)
    expect = plain_qwen2.causal_attention(q, k, v, scale, past_len=length - 1)
    for tile_waves in (1, 4):
        for n_splits, per_split in [(1, 0), (7, 288), (63, 32)]:
            out = run_mfma(ops, q.reshape(1, -1), [length - 1], [1], k_pool, v_pool, table, slots, q_heads, kv_heads,
                           head_dim, None, scale, 1, 1, n_splits=n_splits, keys_per_split=per_split,
                           tile_waves=tile_waves)
            torch.testing.assert_close(out, expect, **tol(torch.bfloat16))
            torch.testing.assert_close(out.view(q_heads, head_dim), v[far].repeat_interleave(8, dim=0), rtol=0.05, atol=0.05)
    # the prompt form: the last of 40 tokens asks for the far key; the four waves of its tile each see a
    # quarter of the keys and only one of them holds the key that counts
    q_many = torch.cat([torch.randn((39, q_heads, head_dim), generator=torch.Generator().manual_seed(77)), q])
    q_many = q_many.to(torch.bfloat16).float()
    expect = plain_qwen2.causal_attention(q_many, k, v, scale, past_len=length - 40)
    # (tiles of 128 rows, and of 64 a second time: the form through LDS, whose two halves each see every other block)
    for row_tiles, tile_waves in ((1, 4), (2, 4), (4, 4), (8, 8), (4, 8)):
        out = run_mfma(ops, q_many.reshape(40, -1), [length - 40], [40], k_pool, v_pool, table, slots, q_heads,
                       kv_heads, head_dim, None, scale, 2 * row_tiles, row_tiles, tile_waves=tile_waves)
        torch.testing.assert_close(out, expect, **tol(torch.bfloat16))
        torch.testing.assert_close(out[-1].view(q_heads, head_dim), v[far].repeat_interleave(8, dim=0), rtol=0.05, atol=0.05)


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_far_key_and_window(ops, dtype):
    """One far key is made to dominate: the output must be its value row.  With a
    window that excludes it, it must vanish; the window's edge is exact."""
    q_heads, kv_heads, head_dim, page_size = 4, 2, 32, 8
    length, far = 400, 37
    k_pool, v_pool, table, slots, dense = build_cache(dtype, [length], kv_heads, head_dim, page_size, seed=30)
    k, v = dense[0]
    q = torch.zeros((1, q_heads, head_dim))
    for h in range(q_heads):
        q[0, h] = k[far, h // 2] * 4.0  # aligned with the far key, far larger score than any other
    q = q.to(dtype).float()
    scale = 1.0 / math.sqrt(head_dim)
    args = (k_pool, v_pool, table, torch.tensor([length - 1], dtype=torch.int32).cuda(),
            torch.tensor([0], dtype=torch.int32).cuda(), torch.tensor(slots, dtype=torch.int32).cuda(),
            1, q_heads, kv_heads, head_dim)
    qd = q.reshape(1, -1).to(dtype).cuda()
    full = ops.paged_attention_generic(qd, q_heads * head_dim, *args, None, scale).float().cpu()
    expect_full = plain_qwen2.causal_attention(q, k, v, scale, past_len=length - 1)
    torch.testing.assert_close(full, expect_full, **tol(dtype))
    # the far key carries nearly all the weight
    torch.testing.assert_close(full.reshape(q_heads, head_dim), v[far].repeat_interleave(2, dim=0), rtol=0.1, atol=0.1)
    for window in (length - far, length - far - 1):  # far key just inside / just outside
        got = ops.paged_attention_generic(qd, q_heads * head_dim, *args, window, scale).float().cpu()
        expect = plain_qwen2.causal_attention(q, k, v, scale, past_len=length - 1, window=window)
        torch.testing.assert_close(got, expect, **tol(dtype))
    assert (got - full).abs().max() > 0.1  # outside the window the answer changes


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("geometry", [(4, 2, 16, 16), (3, 1, 48, 8), (16, 2, 128, 16)])
def test_rope_kv_write(ops, dtype, geometry):
    q_heads, kv_heads, head_dim, page_size = geometry
    theta, max_pos = 10000.0, 512
    lengths = [40, 3, 100]
    starts = [30, 0, 99]  # tokens of this step: positions start..length-1
    k_pool, v_pool, table, slots, _ = build_cache(dtype, lengths, kv_heads, head_dim, page_size, seed=40)
    k_before, v_before = k_pool.clone(), v_pool.clone()
    positions, seq_of_token = [], []
    for s, (start, n) in enumerate(zip(starts, lengths)):
        positions += list(range(start, n))
        seq_of_token += [s] * (n - start)
    t = len(positions)
    qkv = rand((t, (q_heads + 2 * kv_heads) * head_dim), dtype, 41)
    original = qkv.float().cpu()
    cos, sin = plain_qwen2.rope_tables(head_dim, max_pos, theta)
    half = head_dim // 2
    pos_t = torch.tensor(positions)
    ops.rope_kv_write(qkv, cos[:, :half].contiguous().cuda(), sin[:, :half].contiguous().cuda(),
                      torch.tensor(positions, dtype=torch.int32).cuda(),
                      torch.tensor(seq_of_token, dtype=torch.int32).cuda(),
                      torch.tensor(slots, dtype=torch.int32).cuda(), table, k_pool, v_pool,
                      q_heads, kv_heads, head_dim)
    q_in = original[:, : q_heads * head_dim].view(t, q_heads, head_dim)
    k_in = original[:, q_heads * head_dim: (q_heads + kv_heads) * head_dim].view(t, kv_heads, head_dim)
    v_in = original[:, (q_heads + kv_heads) * head_dim:].view(t, kv_heads, head_dim)
    q_expect = plain_qwen2.apply_rope(q_in, cos, sin, pos_t)
    k_expect = plain_qwen2.apply_rope(k_in, cos, sin, pos_t)
    torch.testing.assert_close(qkv.float().cpu()[:, : q_heads * head_dim].view(t, q_heads, head_dim), q_expect, **tol(dtype))
    table_h = table.cpu()
    touched = torch.zeros(k_pool.shape[:3], dtype=torch.bool)  # [page, head, row]
    for i, (pos, s) in enumerate(zip(positions, seq_of_token)):
        page = int(table_h[slots[s], pos // page_size])
        row = pos % page_size
        torch.testing.assert_close(k_pool[page, :, row].float().cpu(), k_expect[i], **tol(dtype))
        torch.testing.assert_close(v_pool[page, :, :, row].float().cpu(), v_in[i], rtol=0, atol=0)  # transposed
        touched[page, :, row] = True
    # nothing else in the pools moved
    untouched = ~touched.cuda()
    assert torch.equal(k_pool[untouched], k_before[untouched])
    assert torch.equal(v_pool.transpose(2, 3)[untouched], v_before.transpose(2, 3)[untouched])


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16, 2048), (4, 2, 32, 8, 96), (3, 1, 64, 4, 328), (5, 5, 96, 32, 200)])
@pytest.mark.parametrize("rows", [1, 7, 16, 24, 40, 64, 72, 100, 128])
@pytest.mark.parametrize("waves", [None, 1, 8])
def test_gemm_qkv_rope_equals_product_then_rotation(ops, geometry, rows, waves):
    """The q/k/v product whose epilogue rotates and writes the cache, against the plain
    product followed by the rotation kernel (themselves checked against the plain
    implementation above): rotated queries, touched cache rows and untouched ones."""
    q_heads, kv_heads, head_dim, page_size, hidden = geometry
    n = (q_heads + 2 * kv_heads) * head_dim
    row_tiles = 1 if rows <= 16 else 2 if rows <= 32 else 4
    if waves == 1 and row_tiles > 1:
        waves = 4  # the fewest with more than 16 rows
    lengths = [40, 35, 100, 33][: max(1, min(4, rows))]  # every sequence has at least rows / 4 tokens
    k_pool, v_pool, table, slots, _ = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=44)
    k_two, v_two = k_pool.clone(), v_pool.clone()
    # the rows: the last tokens of the sequences in turn (decode rows), several per sequence when rows > sequences
    positions, seq_of_token = [], []
    for i in range(rows):
        s = i % len(lengths)
        positions.append(lengths[s] - 1 - i // len(lengths))
        seq_of_token.append(s)
    assert min(positions) >= 0
    a = rand((rows, hidden), torch.bfloat16, 45)
    w, b = rand((n, hidden), torch.bfloat16, 46, 0.3), rand((n,), torch.bfloat16, 47)
    cos, sin = plain_qwen2.rope_tables(head_dim, 512, 1e6)
    half = head_dim // 2
    cos, sin = cos[:, :half].contiguous().cuda(), sin[:, :half].contiguous().cuda()
    meta = (torch.tensor(positions, dtype=torch.int32).cuda(), torch.tensor(seq_of_token, dtype=torch.int32).cuda(),
            torch.tensor(slots, dtype=torch.int32).cuda(), table)
    fused = ops.gemm_qkv_rope(w, a, b, cos, sin, *meta, k_pool, v_pool, q_heads, kv_heads, head_dim, waves=waves)
    plain_qkv = ops.gemm_fused(w, ops.EPI_BF16, a, bias=b, plan=None if waves is None else (row_tiles, waves, 1))
    ops.rope_kv_write(plain_qkv, cos, sin, *meta, k_two, v_two, q_heads, kv_heads, head_dim)
    q_cols = q_heads * head_dim
    # one bf16 step at most (the two kernels may round a fused multiply-add differently)
    step = dict(rtol=2 ** -7, atol=1e-6)
    torch.testing.assert_close(fused[:, :q_cols].float(), plain_qkv[:, :q_cols].float(), **step)
    torch.testing.assert_close(k_pool.float(), k_two.float(), **step)
    assert torch.equal(v_pool, v_two)
    # without rotation and without cache writes
    k_before, v_before = k_pool.clone(), v_pool.clone()
    bare = ops.gemm_qkv_rope(w, a, b, cos, sin, *meta, k_pool, v_pool, q_heads, kv_heads, head_dim, rotate=False,
                             write_kv=False, waves=waves)
    if waves is None:  # the two plans may cut K differently: sums in another order
        torch.testing.assert_close(bare[:, :q_cols].float(), ops.gemm_fused(w, ops.EPI_BF16, a, bias=b)[:, :q_cols].float(), **step)
    else:
        same_plan = ops.gemm_fused(w, ops.EPI_BF16, a, bias=b, plan=(row_tiles, waves, 1))
        if row_tiles == 1:
            assert torch.equal(bare[:, :q_cols], same_plan[:, :q_cols])
        else:  # a pair of column tiles per workgroup here, one there: the waves' sums meet in another order
            torch.testing.assert_close(bare[:, :q_cols].float(), same_plan[:, :q_cols].float(), **step)
    assert torch.equal(k_pool, k_before) and torch.equal(v_pool, v_before)
    with pytest.raises(ValueError, match="steps of 32"):
        ops.gemm_qkv_rope(w[: 3 * 16], a, None, cos[:, :8].contiguous(), sin[:, :8].contiguous(), *meta,
                          k_pool[..., :16].contiguous(), v_pool[:, :, :16].contiguous(), 1, 1, 16)


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16, 2048), (4, 2, 32, 8, 96), (3, 1, 64, 4, 328), (28, 4, 128, 16, 3584),
                                      (5, 5, 96, 32, 200), (64, 8, 128, 16, 8192)])
@pytest.mark.parametrize("rows", [1, 3, 8, 13, 16, 17])
@pytest.mark.parametrize("waves", [None, 1, 8])
def test_gemm_qkv_rope_that_makes_the_norm_itself(ops, geometry, rows, waves):
    """The q/k/v product of up to 16 rows that is given the float32 residual stream instead of normalised rows:
    the rotated queries and the cache against float64 arithmetic on the kernel's own operand rounding (rows are
    bf16(x * weight), their 1/rms multiplies the sums), and against the two kernels it replaces."""
    q_heads, kv_heads, head_dim, page_size, hidden = geometry
    if not ops.folds_norm(rows, hidden):
        with pytest.raises(ValueError, match="makes the norm of up to"):
            ops.gemm_qkv_rope(rand(((q_heads + 2 * kv_heads) * head_dim, hidden), torch.bfloat16, 1), None, None,
                              *([torch.zeros(1, device="cuda")] * 8), q_heads, kv_heads, head_dim,
                              folded=(torch.zeros((rows, hidden), device="cuda"), torch.ones(hidden, device="cuda"), 1e-6))
        return
    n = (q_heads + 2 * kv_heads) * head_dim
    eps = 1e-5
    lengths = [40, 35, 100, 33, 64, 1, 17, 90, 41, 36, 101, 34, 65, 2, 18, 91][:rows]
    k_pool, v_pool, table, slots, _ = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=61)
    k_two, v_two = k_pool.clone(), v_pool.clone()
    positions = [length - 1 for length in lengths]
    residual = rand((rows, hidden), torch.float32, 62, 2.0) * torch.linspace(0.2, 3.0, rows, device="cuda")[:, None]
    norm_weight = (1.0 + rand((hidden,), torch.float32, 64, 0.3)).contiguous()
    w, b = rand((n, hidden), torch.bfloat16, 65, 0.05), rand((n,), torch.bfloat16, 66)
    cos, sin = plain_qwen2.rope_tables(head_dim, 512, 1e6)
    half = head_dim // 2
    cos, sin = cos[:, :half].contiguous().cuda(), sin[:, :half].contiguous().cuda()
    meta = (torch.tensor(positions, dtype=torch.int32).cuda(), torch.arange(rows, dtype=torch.int32).cuda(),
            torch.tensor(slots, dtype=torch.int32).cuda(), table)
    before = residual.clone()
    fused = ops.gemm_qkv_rope(w, None, b, cos, sin, *meta, k_pool, v_pool, q_heads, kv_heads, head_dim,
                              waves=waves, folded=(residual, norm_weight, eps))
    assert torch.equal(residual, before)  # the stream is read only
    scale = torch.rsqrt(residual.double().pow(2).mean(-1, keepdim=True) + eps)
    operand = (residual * norm_weight).to(torch.bfloat16).double()  # the rows as the kernel rounds them
    unrotated = ((operand @ w.double().t()) * scale + b.double()).to(torch.bfloat16)
    ops.rope_kv_write(unrotated, cos, sin, *meta, k_two, v_two, q_heads, kv_heads, head_dim)
    q_cols = q_heads * head_dim
    # a bf16 step in a value before its rotation moves the rotated pair by that much of the larger of the two
    step = dict(rtol=2 ** -6, atol=2 ** -7 * float(unrotated.float().abs().max()))
    torch.testing.assert_close(fused[:, :q_cols].float(), unrotated[:, :q_cols].float(), **step)
    torch.testing.assert_close(k_pool.float(), k_two.float(), **step)
    torch.testing.assert_close(v_pool.float(), v_two.float(), **step)
    # ... and it agrees with the two kernels it replaces to the rounding of their different order
    normed = ops.add_rmsnorm(residual.clone(), None, norm_weight, eps, torch.bfloat16)
    two = ops.gemm_qkv_rope(w, normed, b, cos, sin, *meta, k_two, v_two, q_heads, kv_heads, head_dim)
    torch.testing.assert_close(fused[:, :q_cols].float(), two[:, :q_cols].float(), rtol=2 ** -5,
                               atol=2 ** -6 * float(unrotated.float().abs().max()))


def test_rope_shift_invariance():
    """Scores of rotated q and k depend on the distance of their positions only
    (pins sign and pairing of the rotation in the plain implementation)."""
    head_dim = 32
    cos, sin = plain_qwen2.rope_tables(head_dim, 600, 10000.0)
    g = torch.Generator().manual_seed(50)
    q = torch.randn((1, 1, head_dim), generator=g, dtype=torch.float64)
    k = torch.randn((1, 1, head_dim), generator=g, dtype=torch.float64)
    cos, sin = cos.double(), sin.double()

    def score(m, n):
        qm = plain_qwen2.apply_rope(q, cos, sin, torch.tensor([m]))
        kn = plain_qwen2.apply_rope(k, cos, sin, torch.tensor([n]))
        return (qm * kn).sum()

    assert abs(score(10, 3) - score(210, 203)) < 1e-3  # float32 tables limit the agreement
    assert abs(score(10, 3) - score(10, 4)) > 1e-3


def test_sample_greedy_and_temperature(ops):
    g = torch.Generator().manual_seed(60)
    logits = torch.randn((6, 1003), generator=g).cuda() * 3
    logits[2, 500] = logits[2, 17] = logits[2].max() + 1  # a tie: the lower index wins
    out = ops.sample(logits)
    assert out.tolist() == torch.argmax(logits, dim=-1).tolist()
    assert out[2].item() == 17
    temperature = torch.tensor([0.0, 0.7, 1.0, 1.3, 0.7, 2.0]).cuda()
    uniform = torch.tensor([0.3, 0.0, 0.999999, 0.5, 0.25, 0.75]).cuda()
    got = ops.sample(logits, temperature, uniform).tolist()
    assert got[0] == out[0].item()  # temperature 0 is greedy
    for r in range(1, 6):
        p = torch.softmax(logits[r].double() / temperature[r].double(), dim=-1).cpu()
        cdf = torch.cumsum(p, dim=0)
        u = float(uniform[r])
        lo = cdf[got[r] - 1].item() if got[r] > 0 else 0.0
        assert lo - 1e-5 <= u <= cdf[got[r]].item() + 1e-5, (r, got[r], lo, u, cdf[got[r]].item())


@pytest.mark.parametrize("vocab", [1024, 4099, 8192, 9001, 151936])
def test_sample_over_many_chunks(ops, vocab):
    """A vocabulary of many chunks of the kernel's walk (and one that ends inside a chunk, with rows that are
    not 16-byte aligned), and from 8,192 tokens on rows that many workgroups take in parts and a second kernel
    finishes: the token is the one whose share of [0, 1) holds the row's number, for numbers at the very start,
    inside and at the very end, and for a row whose weight sits in its last tokens."""
    g = torch.Generator().manual_seed(62)
    rows = 7
    logits = (torch.randn((rows, vocab), generator=g) * 2).cuda()
    logits[5, vocab - 3:] += 30.0       # nearly all weight in the last three tokens
    logits[6, : vocab - 1] -= 60.0      # all of it in the last one
    temperature = torch.tensor([0.7, 1.0, 1.5, 0.3, 1.0, 1.0, 1.0]).cuda()
    uniform = torch.tensor([0.0, 0.37, 0.999999, 0.5, 0.123456, 0.9, 0.4]).cuda()
    got = ops.sample(logits, temperature, uniform).tolist()
    for r in range(rows):
        p = torch.softmax(logits[r].double() / temperature[r].double(), dim=-1).cpu()
        cdf = torch.cumsum(p, dim=0)
        u = float(uniform[r])
        lo = cdf[got[r] - 1].item() if got[r] > 0 else 0.0
        assert 0 <= got[r] < vocab and lo - 2e-5 <= u <= cdf[got[r]].item() + 2e-5, (r, got[r], lo, u, cdf[got[r]].item())
    assert got[5] >= vocab - 3 and got[6] == vocab - 1
    # the same draw whatever else is in the batch: row 1 alone
    assert ops.sample(logits[1:2], temperature[1:2], uniform[1:2]).tolist() == [got[1]]
    # rows without a temperature among the others: the first index of the largest logit
    logits[3, vocab - 1] = logits[3, 5] = logits[3].max() + 1
    mixed = temperature.clone()
    mixed[3] = mixed[0] = 0.0
    again = ops.sample(logits, mixed, uniform).tolist()
    assert again[3] == 5 and again[0] == int(torch.argmax(logits[0])) and again[1] == got[1] and again[6] == got[6]


@pytest.mark.parametrize("vocab", [3000, 40000])
def test_sample_with_a_number_next_to_one_never_draws_a_token_without_probability(ops, vocab):
    """The row's number is the largest below 1 and the target may round past the running sums (they are made
    in another order than the total): the token then is the last one that has any probability, never the
    last of a chunk or part whose tail lies so far below the maximum that its terms are zero.  Many rows
    with their weight in the first tokens, spread over several chunks (and, in the large vocabulary, two parts)."""
    g = torch.Generator().manual_seed(64)
    rows = 256
    logits = torch.full((rows, vocab), -1.0e4)
    heads = torch.randint(1500, 2600, (rows,), generator=g)
    for r in range(rows):
        logits[r, : heads[r]] = torch.randn(int(heads[r]), generator=g) * 0.5
    temperature = torch.full((rows,), 1.0)
    uniform = torch.full((rows,), 1.0 - 2.0 ** -24)
    assert float(uniform[0]) < 1.0
    got = ops.sample(logits.cuda(), temperature.cuda(), uniform.cuda()).tolist()
    for r in range(rows):
        p = torch.softmax(logits[r].double(), dim=-1)
        assert p[got[r]] > 0, (r, got[r], int(heads[r]))
        assert got[r] >= int(heads[r]) - 3, (r, got[r], int(heads[r]))  # and it is (next to) the last such token


def test_sample_frequencies(ops):
    """Empirical frequencies on a four-token vocabulary follow softmax(l / T)."""
    logits = torch.tensor([[0.0, 1.0, 2.0, -1.0]]).repeat(4000, 1).cuda()
    g = torch.Generator().manual_seed(61)
    uniform = torch.rand(4000, generator=g).cuda()
    temperature = torch.full((4000,), 0.8).cuda()
    got = ops.sample(logits, temperature, uniform)
    freq = torch.bincount(got.long().cpu(), minlength=4).double() / 4000
    expect = torch.softmax(torch.tensor([0.0, 1.0, 2.0, -1.0]).double() / 0.8, dim=0)
    assert (freq - expect).abs().max() < 0.03


@pytest.mark.parametrize("shape", [(1, 64, 128), (8, 2560, 2048), (16, 96, 328), (17, 208, 1032), (40, 66, 264),
                                   (64, 2048, 1408), (70, 48, 96)])
@pytest.mark.parametrize("plan", [None, "few", "many", "paired"])
def test_gemm_fused_epilogues(ops, shape, plan):
    """The fused few-row product: SiLU-gate and residual-accumulate epilogues, for every plan the
    kernel has (the fewest and the most waves per workgroup, partial tiles summed through LDS;
    one or two column tiles per workgroup with more than 16 rows; more than 64 rows as several
    rows of workgroups), against float64 products."""
    m, n, k = shape
    row_tiles = 1 if m <= 16 else 2 if m <= 32 else 4
    if plan == "paired" and row_tiles == 1:
        pytest.skip("workgroups of 16 rows take one column tile")
    chosen = {None: None, "few": (row_tiles, 1 if row_tiles == 1 else 4, 1), "many": (row_tiles, 8, 1),
              "paired": (row_tiles, 8, 2)}[plan]
    a, w = rand((m, k), torch.bfloat16, 80), rand((n, k), torch.bfloat16, 81, 0.3)
    b = rand((n,), torch.bfloat16, 82)
    exact = a.double() @ w.double().t()
    gate, up = exact[:, : n // 2], exact[:, n // 2:]
    out = ops.gemm_fused(w, ops.EPI_SILU, a, plan=chosen)
    assert out.shape == (m, n // 2) and out.dtype == torch.bfloat16
    want = torch.nn.functional.silu(gate) * up
    torch.testing.assert_close(out.double(), want, rtol=1e-2, atol=1e-2 * float(want.abs().max()))
    plain_out = ops.gemm_fused(w, ops.EPI_F32, a, bias=b, plan=chosen)
    torch.testing.assert_close(plain_out.double(), exact + b.double(), rtol=1e-4, atol=2e-4 * math.sqrt(k))
    residual = rand((m, n), torch.float32, 83, 2.0)
    before = residual.clone()
    parts = -(-n // 16)
    sumsq = torch.full((m + 2, parts), float("nan")).cuda()
    assert ops.gemm_fused(w, ops.EPI_RESID, a, bias=b, residual_out=residual, sumsq_out=sumsq, plan=chosen) is sumsq
    want = before.double() + exact + b.double()
    torch.testing.assert_close(residual.double(), want, rtol=1e-4, atol=2e-4 * math.sqrt(k))
    padded = torch.zeros((m, parts * 16), dtype=torch.float64).cuda()
    padded[:, :n] = want
    torch.testing.assert_close(sumsq[:m].double(), padded.pow(2).view(m, parts, 16).sum(-1), rtol=1e-4, atol=1e-3)
    assert torch.isnan(sumsq[m:]).all()


def test_gemm_fused_random_shapes(ops):
    """Seeded random shapes (rows to 70, any column count, K any multiple of 8) through every
    epilogue, against float64 products: the edges of row tiles, column tiles and K slices in
    combinations the hand-picked shapes do not hold."""
    rng = random.Random(1234)
    for case in range(40):
        m, n, k = rng.randint(1, 70), 2 * rng.randint(1, 150), 8 * rng.randint(1, 180)
        k_parts = rng.choice([1, 1, 2, 3, 5])
        a, w = rand((m, k), torch.bfloat16, 300 + case), rand((n, k), torch.bfloat16, 400 + case, 0.3)
        b = rand((n,), torch.bfloat16, 500 + case)
        exact = a.double() @ w.double().t()
        tag = f"case {case}: m={m} n={n} k={k} parts={k_parts}"
        out = ops.gemm_fused(w, ops.EPI_F32, a, bias=b)
        torch.testing.assert_close(out.double(), exact + b.double(), rtol=1e-4, atol=2e-4 * math.sqrt(k), msg=lambda t: f"{tag}: {t}")
        parts = ops.gemm_shared_rows(w, ops.EPI_PARTIAL, a, bias=b, k_parts=k_parts, column_tiles=1 + case % 2, waves=2 + case % 3)
        torch.testing.assert_close(parts.double().sum(0), exact + b.double(), rtol=1e-4, atol=2e-4 * math.sqrt(k),
                                   msg=lambda t: f"{tag}: {t}")
        gated = ops.gemm_fused(w, ops.EPI_SILU, a)
        want = torch.nn.functional.silu(exact[:, : n // 2]) * exact[:, n // 2:]
        torch.testing.assert_close(gated.double(), want, rtol=1e-2, atol=1e-2 * float(want.abs().max()) + 1e-6,
                                   msg=lambda t: f"{tag}: {t}")
        residual = rand((m, n), torch.float32, 600 + case, 2.0)
        want = residual.double() + exact + b.double()
        sumsq = ops.gemm_fused(w, ops.EPI_RESID, a, bias=b, residual_out=residual)
        torch.testing.assert_close(residual.double(), want, rtol=1e-4, atol=2e-4 * math.sqrt(k), msg=lambda t: f"{tag}: {t}")
        torch.testing.assert_close(sumsq.double().sum(-1), want.pow(2).sum(-1), rtol=1e-3, atol=1e-3, msg=lambda t: f"{tag}: {t}")


@pytest.mark.parametrize("shape", [(1, 64, 256), (8, 2048, 11008), (13, 96, 328), (16, 48, 1032), (40, 200, 1032),
                                   (64, 2048, 2752), (5, 50, 264), (8, 3584, 1024), (72, 2048, 11008), (100, 200, 1032),
                                   (128, 96, 328)])
@pytest.mark.parametrize("k_parts", [1, 3, 4])
def test_gemm_fused_partial_products_and_their_norm(ops, shape, k_parts):
    """K cut into parts: the float32 partial products sum to the product (bias once); and the same parts added
    into a float32 stream with atomic adds leave the stream plus the product there, twice in a row."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.bfloat16, 94), rand((n, k), torch.bfloat16, 95, 0.3), rand((n,), torch.bfloat16, 96)
    parts = ops.gemm_shared_rows(w, ops.EPI_PARTIAL, a, bias=b, k_parts=k_parts)
    assert parts.shape == (k_parts, m, n) and parts.dtype == torch.float32
    exact = a.double() @ w.double().t() + b.double()
    torch.testing.assert_close(parts.double().sum(0), exact, rtol=1e-4, atol=2e-4 * math.sqrt(k))
    residual = rand((m, n), torch.float32, 97, 2.0)
    before = residual.double()
    for turn in (1, 2):
        out = ops.gemm_shared_rows(w, ops.EPI_ATOMIC, a, bias=b, k_parts=k_parts, add_into=residual)
        assert out is residual
        torch.testing.assert_close(residual.double(), before + turn * exact, rtol=1e-4, atol=turn * 2e-4 * math.sqrt(k))
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_ATOMIC, a, k_parts=k_parts)                       # nothing to add into
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_PARTIAL, a, k_parts=k_parts, add_into=residual)   # only the atomic form adds
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_ATOMIC, a, k_parts=k_parts, add_into=residual[:, : n - 8])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 8), (5, 200), (40, 4864), (3, 25)])
def test_silu_mul_with_the_rows_scale(ops, dtype, shape):
    """The SiLU-gate kernel applying the 1/rms that the rows of the product before it lacked."""
    tokens, inter = shape
    hidden, parts, eps = 96, 7, 1e-5
    gate_up = rand((tokens, 2 * inter), dtype, 710, 3.0)
    sumsq = rand((tokens, parts), torch.float32, 711).abs() * 40 + 1
    factor = torch.rsqrt(sumsq.double().sum(-1, keepdim=True) / hidden + eps)
    g, u = gate_up.double()[:, :inter] * factor, gate_up.double()[:, inter:] * factor
    want = torch.nn.functional.silu(g) * u
    got = ops.silu_mul(gate_up, row_sumsq=sumsq, hidden=hidden, eps=eps)
    torch.testing.assert_close(got.double(), want, **({"rtol": 1e-2, "atol": 1e-3} if dtype == torch.bfloat16 else {"rtol": 1e-5, "atol": 1e-6}))
    plain = torch.nn.functional.silu(gate_up.double()[:, :inter]) * gate_up.double()[:, inter:]
    torch.testing.assert_close(ops.silu_mul(gate_up).double(), plain,
                               **({"rtol": 1e-2, "atol": 1e-3} if dtype == torch.bfloat16 else {"rtol": 1e-5, "atol": 1e-6}))


@pytest.mark.parametrize("shape", [(1, 128, 64), (8, 2048, 2048), (13, 200, 328), (16, 96, 1032)])
def test_norm_folded_into_the_products_around_it(ops, shape):
    """o_proj adds into the residual and leaves residual * weight; the gate/up product
    applies each row's 1 / rms to its sums: together the same as the residual product,
    the norm kernel and the plain gate/up product."""
    m, hidden, k = shape
    inter = 2 * 88
    a = rand((m, k), torch.bfloat16, 700)
    w_o, b_o = rand((hidden, k), torch.bfloat16, 701, 0.3), rand((hidden,), torch.bfloat16, 702)
    w_gu = rand((inter, hidden), torch.bfloat16, 703, 0.3)
    norm_weight = (rand((hidden,), torch.float32, 704) + 1).to(torch.bfloat16)
    eps = 1e-5
    residual = rand((m, hidden), torch.float32, 705, 2.0)
    apart = residual.clone()
    sumsq = ops.gemm_fused(w_o, ops.EPI_RESID, a, bias=b_o, residual_out=apart)
    normed = ops.rmsnorm_from_sumsq(apart, sumsq, norm_weight, eps)
    want = ops.gemm_fused(w_gu, ops.EPI_SILU, normed)
    scaled = torch.empty((m, hidden), dtype=torch.bfloat16).cuda()
    folded_sumsq = ops.gemm_fused(w_o, ops.EPI_RESID, a, bias=b_o, residual_out=residual,
                                  norm_weight=norm_weight.float().contiguous(), scaled_out=scaled)
    assert torch.equal(residual, apart) and torch.equal(folded_sumsq, sumsq)
    got = ops.gemm_fused(w_gu, ops.EPI_SILU, scaled, row_sumsq=folded_sumsq, eps=eps)
    # the same values rounded to bf16 at another point (before instead of after the division by the rms)
    exact = torch.nn.functional.silu(
        plain_qwen2.rms_norm(residual.cpu(), norm_weight.float().cpu(), eps).double() @ w_gu.double().cpu().t()[:, : inter // 2]
    ) * (plain_qwen2.rms_norm(residual.cpu(), norm_weight.float().cpu(), eps).double() @ w_gu.double().cpu().t()[:, inter // 2:])
    bound = 1e-2 * float(exact.abs().max())
    torch.testing.assert_close(got.double().cpu(), exact, rtol=2e-2, atol=bound)
    torch.testing.assert_close(want.double().cpu(), exact, rtol=2e-2, atol=bound)
    with pytest.raises(ValueError, match="scale"):
        ops.gemm_fused(w_gu, ops.EPI_BF16, scaled, row_sumsq=folded_sumsq, eps=eps)


@pytest.mark.parametrize("norm_dtype", [torch.bfloat16, torch.float32])
def test_rmsnorm_from_sumsq(ops, norm_dtype):
    residual = rand((5, 1000), torch.float32, 90, 2.0)
    weight = (rand((1000,), torch.float32, 91) + 1).to(norm_dtype)
    full = residual.pow(2).sum(-1, keepdim=True)
    sumsq = (full * torch.softmax(rand((5, 13), torch.float32, 92), dim=-1)).contiguous()
    out = ops.rmsnorm_from_sumsq(residual, sumsq, weight, 1e-5)
    want = plain_qwen2.rms_norm(residual.cpu(), weight.float().cpu(), 1e-5)
    torch.testing.assert_close(out.float().cpu(), want, **tol(torch.bfloat16))


def test_argmax_over_a_large_vocabulary(ops):
    """Two-stage greedy: chunk edges, ties across chunks (the lower index wins), a vocabulary that is no multiple of the chunk."""
    vocab = 151936 + 5
    g = torch.Generator().manual_seed(93)
    logits = torch.randn((9, vocab), generator=g).cuda()
    logits[1, vocab - 1] = 50.0
    logits[2, 0] = 50.0
    logits[3, 2047] = logits[3, 2048] = 50.0
    logits[4, 100000] = logits[4, 4096] = 50.0
    out = ops.sample(logits).tolist()
    assert out == torch.argmax(logits, dim=-1).tolist()
    assert out[1:5] == [vocab - 1, 0, 2047, 4096]


@pytest.mark.parametrize("shape", [(17, 40, 24), (64, 2560, 2048), (150, 99, 72), (300, 515, 328), (2048, 256, 2048)])
def test_gemm_library_matches_float64(ops, shape):
    """The cached interface to the vendor library: with and without bias, rows given as a strided view,
    twice (the second call takes the kept plan)."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.bfloat16, 20), rand((n, k), torch.bfloat16, 21), rand((n,), torch.bfloat16, 22)
    expect = a.double() @ w.double().t()
    for _ in range(2):
        out = ops.gemm_library(a, w)
        if out is None:
            pytest.skip("the library has no algorithm for this shape")
        assert out.dtype == torch.bfloat16 and out.shape == (m, n)
        torch.testing.assert_close(out.double(), expect, rtol=1e-2, atol=1e-2 * math.sqrt(k))
        out = ops.gemm_library(a, w, b)
        torch.testing.assert_close(out.double(), expect + b.double(), rtol=1e-2, atol=1e-2 * math.sqrt(k))
        exact = ops.gemm_library(a, w, out_dtype=torch.float32)  # as for logits
        if exact is not None:
            assert exact.dtype == torch.float32
            torch.testing.assert_close(exact.double(), expect, rtol=1e-4, atol=1e-4 * math.sqrt(k))
    if k % 8 == 0:
        wide = torch.zeros((m, k + 64), dtype=torch.bfloat16).cuda()
        wide[:, :k] = a
        torch.testing.assert_close(ops.gemm_library(wide[:, :k], w, b).double(), expect + b.double(), rtol=1e-2,
                                   atol=1e-2 * math.sqrt(k))


@pytest.mark.parametrize("waves", [2, 3, 4])
@pytest.mark.parametrize("shape", [(5, 32, 128), (17, 656, 520), (37, 80, 264), (64, 2000, 2048), (70, 48, 88), (128, 130, 1160)])
def test_gemm_shared_rows_matches_float64(ops, shape, waves):
    """The form for 17 to 128 rows whose waves own columns and share the rows of A through LDS: plain with
    bias, SiLU-gate with and without rows that lack their 1/rms, and partial products of a cut K (parts that
    end inside a slice of 128, a part without any k, bias in the first part only); widths and row counts that
    fill no tile, one and two tiles a wave, rows given as a strided view."""
    m, n, k = shape
    a, w, b = rand((m, k), torch.bfloat16, 40), rand((n, k), torch.bfloat16, 41, scale=0.1), rand((n,), torch.bfloat16, 42)
    wide = torch.zeros((m, k + 24), dtype=torch.bfloat16).cuda()
    wide[:, :k] = a
    expect = a.double() @ w.double().t()
    tol = dict(rtol=1e-2, atol=1e-2 * math.sqrt(k) * 0.1)
    for tiles in (1, 2):
        out = ops.gemm_shared_rows(w, ops.EPI_BF16, a, bias=b, column_tiles=tiles, waves=waves)
        torch.testing.assert_close(out.double(), expect + b.double(), **tol)
        for parts in (1, 3, 7):
            rows = wide[:, :k] if parts == 3 else a
            out = ops.gemm_shared_rows(w, ops.EPI_PARTIAL, rows, bias=b, column_tiles=tiles, waves=waves, k_parts=parts)
            assert out.shape == (parts, m, n) and out.dtype == torch.float32
            torch.testing.assert_close(out.double().sum(0), expect + b.double(), rtol=1e-4, atol=1e-4 * math.sqrt(k))
    out = ops.gemm_shared_rows(w, ops.EPI_F32, a, bias=b, waves=waves)  # as for logits
    assert out.dtype == torch.float32
    torch.testing.assert_close(out.double(), expect + b.double(), rtol=1e-4, atol=1e-4 * math.sqrt(k))
    gate, up = expect[:, : n // 2], expect[:, n // 2:]
    out = ops.gemm_shared_rows(w, ops.EPI_SILU, a, waves=waves)
    assert out.shape == (m, n // 2) and out.dtype == torch.bfloat16
    torch.testing.assert_close(out.double(), torch.nn.functional.silu(gate) * up, rtol=2e-2, atol=2e-2)
    # rows that lack their 1/rms: partial sums of squares of some other row vector stand for the norm's (a count
    # that is no multiple of four, one that a lane holds at once, one that needs the loop behind it)
    for sumsq_parts in (5, 8, 264):
        sumsq = torch.rand((m + 3, sumsq_parts), generator=torch.Generator().manual_seed(43)).cuda() * k / sumsq_parts
        scale = torch.rsqrt(sumsq[:m].double().sum(1, keepdim=True) / k + 1e-5)
        out = ops.gemm_shared_rows(w, ops.EPI_SILU, a, waves=waves, row_sumsq=sumsq, eps=1e-5)
        torch.testing.assert_close(out.double(), torch.nn.functional.silu(gate * scale) * (up * scale), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("shape", [(1, 2048, 96), (8, 2048, 22016), (16, 4096, 200), (40, 2048, 328), (96, 6144, 72), (5, 2048, 33)])
def test_products_whose_rows_lie_4_kb_apart_match_float64(ops, shape):
    """Where K is a multiple of 2,048 the workgroups begin with different k: logits in both forms, the SiLU product, sums of K in
    parts.  The operands are exact in bf16; K float32 adds of partial sums that grow like sqrt(K) miss the float64 product by some
    K 2^-24 of a term in the root mean square, and four roundings of the sum of the terms' magnitudes are several times that."""
    m, k, n = shape
    a, w = rand((m, k), torch.bfloat16, 71), rand((n, k), torch.bfloat16, 72, 0.3)
    want = a.double() @ w.double().t()
    close = dict(rtol=0.0, atol=float(2.0 ** -22 * (a.double().abs() @ w.double().abs().t()).max()))
    # (the form whose waves share K begins at different k only with one wave over all of it, and one tile of rows)
    torch.testing.assert_close(ops.gemm_fused(w, ops.EPI_F32, a, plan=(1, 1, 1)).double(), want, **close)
    torch.testing.assert_close(ops.gemm_fused(w, ops.EPI_F32, a).double(), want, **close)
    torch.testing.assert_close(ops.gemm_shared_rows(w, ops.EPI_F32, a).double(), want, **close)
    for parts in (1, 3):
        out = ops.gemm_shared_rows(w, ops.EPI_PARTIAL, a, k_parts=parts, column_tiles=1)
        torch.testing.assert_close(out.double().sum(dim=0), want, **close)
    if n % 2 == 0:
        gate, up = want[:, : n // 2], want[:, n // 2:]
        torch.testing.assert_close(ops.gemm_shared_rows(w, ops.EPI_SILU, a).double(), gate * torch.sigmoid(gate) * up,
                                   rtol=2 ** -7, atol=2e-3)


@pytest.mark.parametrize("rows", [4, 16, 40, 90])
@pytest.mark.parametrize("k", [8, 136, 384, 896, 2048])
def test_an_infinite_weight_shows_as_infinity(ops, rows, k):
    """One infinite weight in a column, among the first, the middle or the last k: the column's float32 results are infinite
    in both forms, and no other result is; also where K ends inside a slice or the slices are odd in number."""
    n = 160
    a, w = rand((rows, k), torch.bfloat16, 73), rand((n, k), torch.bfloat16, 74)
    a[a == 0] = 1.0
    for column, at, value in ((3, 0, math.inf), (17, k - 1, math.inf), (40, k // 2, -math.inf), (159, k - 8, -math.inf)):
        w[column, at] = value
    for out in (ops.gemm_fused(w, ops.EPI_F32, a), ops.gemm_shared_rows(w, ops.EPI_F32, a)):
        assert not out.isnan().any()
        assert torch.equal(out.isinf().any(0).nonzero().flatten().cpu(), torch.tensor([3, 17, 40, 159]))
        assert torch.equal(out[:, 17], math.inf * a[:, k - 1].float().sign())


def test_gemm_shared_rows_refuses_what_it_does_not_take(ops):
    a, w = rand((129, 64), torch.bfloat16, 44), rand((32, 64), torch.bfloat16, 45)
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_BF16, a)            # more than 128 rows
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_RESID, a[:8])       # an epilogue of the other form
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_BF16, a[:8], k_parts=2)
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(w, ops.EPI_BF16, a[:8], waves=5)
    with pytest.raises(ValueError):
        ops.gemm_shared_rows(rand((32, 60), torch.bfloat16, 46), ops.EPI_BF16, rand((8, 60), torch.bfloat16, 47))


def test_gemm_library_with_every_algorithm_timed(ops):
    """A row count that an engine has named has every algorithm of the library timed at a shape's first
    call, and the one kept is still the product: shapes that no other test uses, so that their first call is here."""
    assert ops._tune_level(768) == 1  # (a multiple of 256 that nobody has named: the heuristic's candidates)
    with ops.library_search({768}):
        assert ops._tune_level(768) == 2 and ops._tune_level(1024) == 1 and ops._tune_level(700) == 0
        for n, k in ((1040, 520), (264, 1288)):
            a, w, b = rand((768, k), torch.bfloat16, 30), rand((n, k), torch.bfloat16, 31), rand((n,), torch.bfloat16, 32)
            expect = a.double() @ w.double().t()
            for _ in range(2):
                out = ops.gemm_library(a, w)
                if out is None:
                    pytest.skip("the library has no algorithm for this shape")
                torch.testing.assert_close(out.double(), expect, rtol=1e-2, atol=1e-2 * math.sqrt(k))
                torch.testing.assert_close(ops.gemm_library(a, w, b).double(), expect + b.double(), rtol=1e-2,
                                           atol=1e-2 * math.sqrt(k))
                exact = ops.gemm_library(a, w, out_dtype=torch.float32)
                if exact is not None:
                    torch.testing.assert_close(exact.double(), expect, rtol=1e-4, atol=1e-4 * math.sqrt(k))
    assert ops._tune_level(768) == 1  # outside the block nothing is searched


@pytest.mark.parametrize("rows", [1, 2, 3, 8, 9, 16])
@pytest.mark.parametrize("geometry", [(16, 2, 128, 2048, 16), (14, 2, 64, 896, 7), (2, 2, 64, 100, 1), (28, 4, 128, 3584, 33),
                                      (32, 1, 64, 130, 129), (4, 4, 96, 33, 2), (8, 2, 32, 640, 5), (2, 1, 256, 1040, 3)])
def test_merge_project(ops, geometry, rows):
    """The merge of a decode step's shares and the output product in one: against 64 bits; shares without keys hold what they held."""
    heads, kv, dim, n, splits = geometry
    group, tile_rows = heads // kv, 16 if heads // kv <= 16 else 32
    part_o = rand((rows, kv, splits, tile_rows, dim), torch.float32, 1)
    part_ml = torch.stack([rand((rows, kv, splits, tile_rows), torch.float32, 2, 8.0),
                           rand((rows, kv, splits, tile_rows), torch.float32, 3).abs() + 1], dim=-1).contiguous()
    empty = torch.rand((rows, kv, splits, 1), generator=torch.Generator().manual_seed(4)).cuda().expand(-1, -1, -1, tile_rows) < 0.3
    empty = empty & (torch.arange(splits).cuda() > 0)[None, None, :, None]  # (a row's first share has keys)
    part_ml[empty] = torch.tensor([-math.inf, 0.0]).cuda()
    part_o[empty] = math.nan
    part_o[:, :, :, group:] = math.inf  # (rows of the tiles that are no head's)
    w, b = rand((n, heads * dim), torch.bfloat16, 5, 0.05), rand((n,), torch.bfloat16, 6)
    start = rand((rows, n), torch.float32, 7, 3.0)

    m, l = part_ml[..., :group, 0].double(), part_ml[..., :group, 1].double()
    weight = torch.exp2(m - m.amax(dim=2, keepdim=True))
    sums = torch.where(empty[..., :group, None], 0.0, part_o[..., :group, :].double())
    merged = (sums * weight[..., None]).sum(dim=2) / (l * weight).sum(dim=2)[..., None]
    merged = merged.reshape(rows, heads * dim)
    for bias in (b, None):
        residual = start.clone()
        ops.merge_project(part_o, part_ml, w, bias, residual, heads, kv, dim, splits, tile_rows)
        want = start.double() + merged @ w.double().t() + (bias.double() if bias is not None else 0.0)
        # merged rows are rounded to bf16 (half of 2^-8 of each number); float32 sums over K, and the stream's own last bits
        bound = 2.0 ** -9 * (1 + 2.0 ** -7) * (merged.abs() @ w.double().abs().t()) + 1e-4
        assert ((residual.double() - want).abs() <= bound).all()
    with pytest.raises(ValueError):
        ops.merge_project(part_o, part_ml, w, b, start[:, : n - 1].contiguous(), heads, kv, dim, splits, tile_rows)
    with pytest.raises(ValueError):
        ops.merge_project(part_o, part_ml, w, b, start, heads, kv, dim, splits + 1, tile_rows)


@pytest.mark.parametrize("waves", [2, 3, 4])
@pytest.mark.parametrize("shape", [(1, 64, 128), (8, 2208, 2048), (9, 96, 136), (16, 48, 328), (5, 34, 1032), (12, 1000, 264), (8, 22016, 8)])
def test_gemm_shared_rows_that_makes_the_norm_itself(ops, shape, waves):
    m, n, k = shape
    stream, norm = rand((m, k), torch.float32, 1, 3.0), rand((k,), torch.float32, 2, 0.1) + 1
    w = rand((n, k), torch.bfloat16, 3, 0.1)
    rows = (stream * norm).bfloat16().double()  # (rounded short of the rows' scale)
    scale = torch.rsqrt((stream.double() ** 2).mean(dim=1, keepdim=True) + 1e-6)
    gate, up = ((rows @ w.double().t()) * scale).split(n // 2, dim=1)
    want = gate * torch.sigmoid(gate) * up
    out = ops.gemm_shared_rows_normed(stream, norm, 1e-6, w, waves=waves)
    # the result's own rounding, and float32 sums of K terms in front of it
    torch.testing.assert_close(out.double(), want, rtol=2.0 ** -8, atol=2e-5 * math.sqrt(k) * float(gate.abs().max() + up.abs().max()))
    with pytest.raises(ValueError):
        ops.gemm_shared_rows_normed(rand((17, k), torch.float32, 1), norm, 1e-6, w)


@pytest.mark.parametrize("counts", [(1, 300), (0, 1, 255, 256, 257, 700, 3)])
def test_table_rows(ops, counts):
    table = torch.arange(40 * 1000, dtype=torch.int32).reshape(40, 1000).cuda()
    want, heads, entries = table.clone(), [], []
    for index, count in enumerate(counts):
        slot, first = (index * 7 + 3) % 40, 1000 - count - (5 if index % 2 else 0)
        if count + first > 1000 or first < 0:
            first = 0
        heads += [slot, first, count, 4 * len(counts) + len(entries)]
        new = list(range(-count, 0))
        entries += new
        want[slot, first: first + count] = torch.tensor(new, dtype=torch.int32).cuda()
    ops.table_rows(torch.tensor(heads + entries, dtype=torch.int32).cuda(), len(counts), table)
    assert torch.equal(table, want)
    with pytest.raises(ValueError):
        ops.table_rows(torch.zeros(7, dtype=torch.int32).cuda(), 2, table)


@pytest.mark.parametrize("slots", [[0], [5, 2, 6]])
def test_clear_rows(ops, slots):
    shapes = [(8, 128, 256), (2048,), (3, 5), (1,), (7,)]
    types = [torch.float32, torch.float32, torch.float32, torch.int32, torch.bfloat16]
    states = [torch.ones((7, *shape), dtype=dtype).cuda() for shape, dtype in zip(shapes, types)]
    size = [s[0].numel() * s.element_size() for s in states]
    rows = torch.tensor([[s.data_ptr(), b] for s, b in zip(states, size)], dtype=torch.int64).cuda()
    ops.clear_rows(rows, torch.tensor(slots, dtype=torch.int32).cuda(), max(size))
    for state in states:
        for slot in range(7):
            assert (state[slot] == (0 if slot in slots else 1)).all()


@pytest.mark.parametrize("n,size,fed", [(1, 1, False), (3, 4, True), (5, 8, False), (64, 64, True), (70, 128, True), (128, 128, False)])
def test_step_rows(ops, n, size, fed):
    from array import array

    places = [torch.full((size + 1,), 99, dtype=torch.int32).cuda() for _ in range(5)] + [torch.full((2,), 99, dtype=torch.int32).cuda()]
    tokens, positions, slots = [7 * i for i in range(n)], [3 * i + 1 for i in range(n)], [n - i for i in range(n)]
    feed = [i % 3 - 1 for i in range(n)]
    ops.step_rows(array("i", tokens + positions + slots + (feed if fed else [])), n, size, fed, 4321, 200, *places)
    rest = size - n
    want = [tokens + [0] * rest, positions + [0] * rest, positions + [0] * rest, slots + [200] * rest,
            (feed if fed else [-1] * n) + [-1] * rest]
    for place, values in zip(places, want):
        assert place.tolist() == values + [99]
    assert places[5].tolist() == [4321, 99]
    with pytest.raises(ValueError):
        ops.step_rows(array("i", tokens), n, size, fed, 1, 200, *places)


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16), (3, 1, 96, 8), (14, 2, 64, 8), (8, 1, 32, 4)])
@pytest.mark.parametrize("window", [None, 70])
def test_attention_f32_blocks_shared_by_four_waves_keep_their_bits(ops, geometry, window):
    """The block form gives a row the same bits whether a wave takes a block (many places of 16 rows and a block) or four
    share one (few); one sequence has infinities and a NaN among its last block's values."""
    q_heads, kv_heads, dim, page = geometry
    g = torch.Generator().manual_seed(21)
    lengths = [1, 63, 64, 65, 200, 513] * 60  # (360 tiles of up to 9 blocks)
    n = len(lengths)
    width = -(-max(lengths) // page)
    table = torch.arange(n * width, dtype=torch.int32).reshape(n, width).cuda()
    k_pool = torch.randn((n * width, kv_heads, page, dim), generator=g).cuda()
    v_pool = torch.randn((n * width, kv_heads, dim, page), generator=g).cuda()
    v_pool[4 * width + 199 // page, 0, 3, 199 % page] = math.inf
    v_pool[4 * width + 199 // page, 0, dim - 1, 198 % page] = math.nan
    q = torch.randn((n, q_heads * dim), generator=g).cuda()
    meta = lambda values: torch.tensor(values, dtype=torch.int32).cuda()

    def run(count):
        group, blocks = q_heads // kv_heads, 9
        out = torch.zeros((count, q_heads * dim)).cuda()
        part_o, part_ml = torch.empty(count * kv_heads * blocks * group * dim).cuda(), torch.empty(count * kv_heads * blocks * group * 2).cuda()
        ops.paged_attention_f32(q[:count], q.stride(0), k_pool, v_pool, table, None, None, count, meta(range(count)),
                                meta([m - 1 for m in lengths[:count]]), meta([1] * count), meta(range(count + 1)), out, q_heads, kv_heads,
                                dim, window, dim ** -0.5, 1, turns=blocks, blocks=blocks, part_o=part_o, part_ml=part_ml)
        return out

    few, many = run(6), run(n)
    assert torch.equal(torch.nan_to_num(few, 3.0, 5.0, 7.0), torch.nan_to_num(many[:6], 3.0, 5.0, 7.0))


@pytest.mark.parametrize("shape", [(1, 64, 32, 128), (8, 22016, 6144, 2048), (8, 9728, 2304, 896), (3, 34, 40, 136), (16, 1000, 4736, 328), (9, 96, 17, 2048)])
@pytest.mark.parametrize("waves", [2, 3, 4])
def test_gemm_silu_beside(ops, shape, waves):
    """A SiLU-gate product and a plain one of other rows in one launch, against 64 bits."""
    m, n, n2, k = shape
    a, a2 = rand((m, k), torch.bfloat16, 1), rand((m, 2 * k), torch.bfloat16, 2)[:, :k]  # (rows that lie apart)
    w, w2, b2 = rand((n, k), torch.bfloat16, 3, 0.05), rand((n2, k), torch.bfloat16, 4, 0.05), rand((n2,), torch.bfloat16, 5)
    gate, up = (a.double() @ w.double().t()).split(n // 2, dim=1)
    for bias in (b2, None):
        out, out2 = ops.gemm_silu_beside(w, a, w2, a2, bias, waves=waves)
        # (a bf16 result's own rounding, float32 sums of k terms in front of it)
        torch.testing.assert_close(out.double(), gate * torch.sigmoid(gate) * up, rtol=2.0 ** -8, atol=1e-5 * math.sqrt(k))
        want = a2.double() @ w2.double().t() + (bias.double() if bias is not None else 0.0)
        torch.testing.assert_close(out2.double(), want, rtol=2.0 ** -8, atol=1e-5 * math.sqrt(k))
    with pytest.raises(ValueError):
        ops.gemm_silu_beside(w, rand((17, k), torch.bfloat16, 1), w2, rand((17, k), torch.bfloat16, 2), b2)


@pytest.mark.parametrize("shape", [(1, 64, 128, 128), (8, 2048, 11008, 2048), (16, 896, 4864, 768), (5, 40, 1032, 3000), (9, 130, 8, 136)])
def test_gemm_parts_beside(ops, shape):
    from cie_amd.parts.linear import plan_parts_beside

    m, n, k, k2 = shape
    a, a2 = rand((m, k), torch.bfloat16, 1), rand((m, k2), torch.bfloat16, 2)
    w, w2 = rand((n, k), torch.bfloat16, 3, 0.05), rand((n, k2), torch.bfloat16, 4, 0.05)
    want = a.double() @ w.double().t() + a2.double() @ w2.double().t()
    for parts, parts2 in ((1, 1), plan_parts_beside(-(-n // 16), k, k2, 256)):
        out = ops.gemm_parts_beside(w, a, parts, w2, a2, parts2)
        assert tuple(out.shape) == (parts + parts2, m, n)
        torch.testing.assert_close(out.double().sum(dim=0), want, rtol=0, atol=2e-6 * math.sqrt(k + k2))
    stream = rand((m, n), torch.float32, 6)
    got, _ = ops.depth_stream(stream, parts=out, mult=0.5, out_dtype=torch.bfloat16)  # (parts and no other branch)
    torch.testing.assert_close(got.double(), stream.double() + 0.5 * want, rtol=1e-6, atol=4e-6 * math.sqrt(k + k2))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 4099, 136), (3, 2050, 1024), (8, 40000, 256), (8, 513, 2056), (40, 300, 264), (80, 50304, 128)])
def test_logits_go_where_an_address_says(ops, dtype, shape):
    """A result whose address lies on the device has the bits of one that comes back, and nothing around it is touched; replays
    of a captured launch follow the address."""
    from cie_amd.parts import linear as L

    m, n, k = shape
    a, w = rand((m, k), dtype, 1), rand((n, k), dtype, 2)
    want = L.linear(a, w, out_dtype=torch.float32)
    outs = [torch.full((m + 2, n), 7.0).cuda() for _ in range(3)]
    at = torch.tensor([outs[0].data_ptr() + 4 * n], dtype=torch.int64).cuda()
    wrote = L.logits_at(a, w, at)
    assert wrote == (dtype == torch.bfloat16 or m <= ops.F32_FEW_ROWS)
    if not wrote:
        assert (outs[0] == 7.0).all()
        return
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert L.logits_at(a, w, at)
    for out in outs[1:]:
        at.copy_(torch.tensor([out.data_ptr() + 4 * n]))
        graph.replay()
    for out in outs:
        assert torch.equal(out[1: m + 1], want) and (out[0] == 7.0).all() and (out[m + 1] == 7.0).all()
    with pytest.raises(ValueError):
        ops.gemm_fused(w.bfloat16(), ops.EPI_BF16, a.bfloat16()[:1], out_at=at)


@pytest.mark.parametrize("shape", [(896, 896), (2048, 2048), (1024, 4096), (48, 136), (2304, 1032)])
@pytest.mark.parametrize("rows", [17, 31, 33, 49, 64, 65, 97, 128])
def test_products_of_more_rows_in_blocks_of_rows(ops, shape, rows):
    """The product added into the stream in blocks of 16, 32 and 64 rows and as planned, against float64: the stream, the next
    norm's rows and their sums of squares; the same bits where as many waves share K."""
    n, k = shape
    a, w, b = rand((rows, k), torch.bfloat16, 1), rand((n, k), torch.bfloat16, 2, 0.05), rand((n,), torch.bfloat16, 3)
    stream, gain = rand((rows, n), torch.float32, 4), rand((n,), torch.float32, 5, 0.1) + 1
    want = stream.double() + a.double() @ w.double().t() + b.double()
    # float32 sums of k products and two more numbers: k + 2 roundings of at most the sum of the magnitudes
    bound = (k + 2) * 2.0 ** -24 * (stream.double().abs() + a.double().abs() @ w.double().abs().t() + b.double().abs())
    first = {}
    for plan in (None, (1, 4, 1), (1, 8, 1), (2, 4, 1), (2, 8, 1), (4, 4, 1), (4, 8, 1)):
        out, scaled = stream.clone(), torch.empty((rows, n), dtype=torch.bfloat16, device="cuda")
        sumsq = ops.gemm_fused(w, ops.EPI_RESID, a, bias=b, residual_out=out, norm_weight=gain, scaled_out=scaled, plan=plan)
        assert ((out.double() - want).abs() <= bound).all()
        assert torch.equal(out, first.setdefault((plan or ops.plan_fused(rows, n // 16, k))[1], out))
        assert torch.equal(scaled, (out * gain).to(torch.bfloat16))
        torch.testing.assert_close(sumsq.sum(dim=1), out.double().pow(2).sum(dim=1).float(), rtol=1e-5, atol=0)


@pytest.mark.parametrize("geometry", [(16, 2, 128, 16, 2048), (14, 2, 64, 16, 896), (3, 1, 32, 4, 328), (24, 8, 96, 16, 1024)])
@pytest.mark.parametrize("rows", [17, 33, 48, 64, 65, 96, 128])
def test_gemm_qkv_rope_in_blocks_of_rows(ops, geometry, rows):
    """Every block of rows and columns that the q/k/v product may be planned in, against the plain product and the rotation's
    kernel: the same values, and what two kernels make of one rotation (a bf16 step)."""
    q_heads, kv_heads, head_dim, page_size, hidden = geometry
    n, q_cols = (q_heads + 2 * kv_heads) * head_dim, q_heads * head_dim
    lengths = [rows + 3, rows + 40]
    k_pool, v_pool, table, slots, _ = build_cache(torch.bfloat16, lengths, kv_heads, head_dim, page_size, seed=9)
    positions = torch.tensor([lengths[i % 2] - 1 - i // 2 for i in range(rows)], dtype=torch.int32).cuda()
    meta = (positions, torch.tensor([i % 2 for i in range(rows)], dtype=torch.int32).cuda(),
            torch.tensor(slots, dtype=torch.int32).cuda(), table)
    a, w, b = rand((rows, hidden), torch.bfloat16, 1), rand((n, hidden), torch.bfloat16, 2, 0.3), rand((n,), torch.bfloat16, 3)
    cos, sin = (t[:, : head_dim // 2].contiguous().cuda() for t in plain_qwen2.rope_tables(head_dim, 512, 1e6))
    for waves in (4, 8):
        plain = ops.gemm_fused(w, ops.EPI_BF16, a, bias=b, plan=(4, waves, 1))
        k_want, v_want = k_pool.clone(), v_pool.clone()
        ops.rope_kv_write(plain, cos, sin, *meta, k_want, v_want, q_heads, kv_heads, head_dim)
        planned = ops.plan_qkv_rope(rows, n // 32, hidden)[1] == waves
        for blocks in ((1, False), (1, True), (2, False), (2, True), (4, False), (4, True)) + ((None,) if planned else ()):
            k_got, v_got = k_pool.clone(), v_pool.clone()
            got = ops.gemm_qkv_rope(w, a, b, cos, sin, *meta, k_got, v_got, q_heads, kv_heads, head_dim,
                                    waves=None if blocks is None else waves, blocks=blocks)
            torch.testing.assert_close(got[:, :q_cols].float(), plain[:, :q_cols].float(), rtol=2 ** -7, atol=1e-6)
            torch.testing.assert_close(k_got.float(), k_want.float(), rtol=2 ** -7, atol=1e-6)
            assert torch.equal(v_got, v_want)
    with pytest.raises(ValueError):
        ops.gemm_qkv_rope(w, a, b, cos, sin, *meta, k_got, v_got, q_heads, kv_heads, head_dim, waves=2, blocks=(2, True))


# (query heads, key heads, head size, rows, longest context): both sides of every line between the forms of a decode step's keys, and
# the (waves a part, parts, whether the output product merges them) of each step launch by launch, captured for that bound, for one
# 900 keys longer and for 32,768
DECODE_LINES = {
    (16, 2, 128, 8, 1023): [(1, 16, True), (1, 16, True), (4, 16, True), (4, 16, True)],
    (16, 2, 128, 8, 1024): [(4, 16, True), (4, 16, True), (4, 16, True), (4, 16, True)],
    (14, 2, 64, 16, 511): [(1, 8, True), (1, 8, True), (4, 8, True), (4, 8, True)],
    (14, 2, 64, 16, 512): [(4, 8, True), (4, 8, True), (4, 8, True), (4, 8, True)],
    (16, 2, 128, 3, 2500): [(1, 40, True), (1, 40, True), (1, 36, True), (4, 32, True)],
    (16, 2, 128, 4, 2048): [(4, 32, True), (4, 32, True), (4, 32, True), (4, 32, True)],
    (28, 4, 128, 9, 600): [(4, 7, True), (4, 7, True), (4, 7, True), (4, 7, True)],
    (32, 8, 64, 12, 700): [(4, 1, False), (4, 1, False), (4, 1, False), (4, 2, True)],
    (8, 1, 128, 3, 700): [(1, 11, True), (1, 11, True), (1, 50, True), (4, 64, True)],
    (14, 2, 64, 17, 704): [(4, 1, False), (4, 1, False), (1, 26, False), (4, 7, False)],
    (14, 2, 64, 17, 705): [(1, 12, False), (1, 12, False), (1, 26, False), (4, 7, False)],
    (16, 2, 128, 30, 352): [(4, 1, False), (4, 1, False), (1, 14, False), (4, 4, False)],
    (16, 2, 128, 30, 353): [(1, 6, False), (1, 6, False), (1, 14, False), (4, 4, False)],
    (16, 2, 128, 25, 983): [(1, 16, False), (1, 16, False), (1, 20, False), (4, 5, False)],
    (16, 2, 128, 25, 984): [(4, 5, False), (1, 16, False), (1, 20, False), (4, 5, False)],
    (14, 2, 64, 32, 1700): [(4, 4, False), (1, 14, False), (4, 4, False), (4, 4, False)],
    (4, 2, 32, 20, 90): [(1, 1, False), (1, 1, False), (4, 1, False), (4, 6, False)],
    (8, 1, 128, 40, 1300): [(4, 6, False), (1, 21, False), (4, 6, False), (4, 6, False)],
}


def decode_line(ops, monkeypatch, line, window=None):
    """The (waves, parts, unmerged) of a step of single tokens launch by launch and as captured.  The step's context, or, where the
    output product merges the parts, what that makes of them with an identity for its weight, is checked against the oracle, and
    against what the merge kernel makes of the same parts; a part or a head that is lost would show."""
    from cie_amd.engine.batch import PagedView, StepBatch
    from cie_amd.engine.graphs import StaticPlan
    from cie_amd.parts import attention as A

    q_heads, kv_heads, dim, rows, longest = line
    width, page = q_heads * dim, 16
    contexts = [longest - 1 if i == rows // 2 else (i * 977) % longest for i in range(rows)]
    lengths = [c + 1 for c in contexts]
    k_pool, v_pool, table, slots, dense = build_cache(torch.bfloat16, lengths, kv_heads, dim, page, seed=5)
    as_dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()  # noqa: E731
    qkv = rand((rows, width + 2 * kv_heads * dim), torch.bfloat16, 1, 2.0)
    one = torch.eye(width, dtype=torch.bfloat16, device="cuda")
    query = lambda i: qkv[i: i + 1, :width].float().cpu().view(1, q_heads, dim)  # noqa: E731
    want = torch.cat([plain_qwen2.causal_attention(query(i), *dense[i], dim ** -0.5, past_len=contexts[i], window=window)
                      for i in range(rows)])
    near = lambda got, expect: bool(torch.isclose(got.float().cpu(), expect, **tol(torch.bfloat16)).all())  # noqa: E731
    # (what the bound sees: the oracle without 32 of the longest row's last keys, and without one head)
    i = rows // 2
    last = slice(contexts[i] - 40, contexts[i] - 8)
    fewer = [torch.cat([t[: last.start], t[last.stop:]]) for t in dense[i]]
    assert not near(plain_qwen2.causal_attention(query(i), *fewer, dim ** -0.5, past_len=contexts[i] - 32,
                                                 window=None if window is None else window - 32), want[i: i + 1])
    no_head = want.clone()
    no_head[:, :dim] = 0
    assert not near(no_head, want)

    batch = dict(tokens=rows, sequences=rows, token_ids=as_dev([0] * rows), positions=as_dev(contexts), seq_of_token=as_dev(range(rows)),
                 seq_slot=as_dev(slots), seq_start=as_dev(contexts), seq_q_len=as_dev([1] * rows), q_start_loc=as_dev(range(rows + 1)),
                 logit_rows=as_dev([0]), host_slots=slots, host_starts=contexts, host_q_lens=[1] * rows)
    forms, merged, real = [], [], ops.paged_attention_mfma

    def attention(*args, **kwargs):
        forms.append((kwargs["tile_waves"], kwargs["n_splits"], not kwargs["merge"]))
        if not kwargs["merge"]:
            real(*args, **{**kwargs, "merge": True})
            merged.append(args[12].clone())
        real(*args, **kwargs)

    monkeypatch.setattr(ops, "paged_attention_mfma", attention)
    plans = [None] + [StaticPlan(as_dev(range(rows)), as_dev([0] * rows), as_dev([longest]), bound) for bound in (longest, longest + 900, 32768)]
    for plan in plans:
        view = PagedView(k_pool, v_pool, table, page)
        stream = torch.zeros((rows, width), device="cuda")
        joins = A.joins_merge(rows, one, stream)
        assert joins == (rows <= 16 and width % 128 == 0)
        out = A.attend(qkv, StepBatch(**batch, static_plan=plan), view, q_heads, kv_heads, dim, window, dim ** -0.5, unmerged=joins)
        if isinstance(out, A.Shares):
            ops.merge_project(out.part_o, out.part_ml, one, None, stream, q_heads, kv_heads, dim, out.splits, out.tile_rows)
            # (a row's numbers, rounded to bf16 and times 1; both roundings are of float32 sums of the same parts: one step apart at most)
            assert ((stream - merged[-1].float()).abs() <= 2.0 ** -7 * merged[-1].float().abs()).all()
            out = stream
        torch.testing.assert_close(out.float().cpu(), want, **tol(torch.bfloat16))
    return forms


@pytest.mark.parametrize("line", DECODE_LINES)
def test_decode_forms_on_both_sides_of_their_lines(ops, line, monkeypatch):
    """A step of single tokens through the attention and, where that takes the keys' shares as they are, the output product."""
    assert decode_line(ops, monkeypatch, line) == DECODE_LINES[line]


@pytest.mark.parametrize("line,window", [((16, 2, 128, 8, 3000), 1000), ((14, 2, 64, 16, 1500), 300), ((16, 2, 128, 3, 900), 640),
                                         ((28, 4, 128, 9, 600), 333)])
def test_shares_under_a_window_left_to_the_output_product(ops, line, window, monkeypatch):
    """... where a row's first shares begin behind its first key, and a short row's last ones have none."""
    forms = decode_line(ops, monkeypatch, line, window)
    assert all(parts > 1 and unmerged for _waves, parts, unmerged in forms)
