"""What a layer's parts hand to one another, without a GPU: the forms of a pending branch, the arguments that a part is
given, and the rules that pick a kernel by sizes alone."""

from __future__ import annotations

import pytest
import torch


class Norm:
    """A norm of the plain interface: a tensor or nothing to add, rows that join the stream."""

    takes_plus = True

    def forward(self, residual, branch, out_dtype, rows=None, plus=None):
        assert branch is None or isinstance(branch, torch.Tensor)
        residual += (0 if branch is None else branch) + (0 if plus is None else plus)
        return residual.to(out_dtype)


def parts_of(*values):
    from cie_amd.parts.linear import KParts

    return KParts(torch.stack([torch.full((3, 4), float(v)) for v in values]))


def test_parts_of_a_product_join_the_stream_for_a_norm_that_cannot_sum_them():
    from cie_amd.parts.block import normalise, whole_stream
    from cie_amd.parts.norm import GroupedRMSNorm, LayerNorm, OnePlusRMSNorm, RMSNorm, ScalarRMSNorm
    from cie_amd.parts.base import declares

    assert all(declares(kind(8, 1e-5), "takes_parts") for kind in (RMSNorm, OnePlusRMSNorm))
    assert not any(declares(kind(8, 1e-5), "takes_parts") for kind in (GroupedRMSNorm, LayerNorm, ScalarRMSNorm))
    for plus in (None, torch.full((3, 4), 0.5)):
        residual = torch.ones(3, 4)
        rows = normalise(Norm(), residual, parts_of(2, 3), torch.float32, plus=plus)
        assert torch.equal(rows, torch.full((3, 4), 6.0 if plus is None else 6.5)) and torch.equal(residual, rows)
    assert torch.equal(whole_stream(torch.ones(3, 4), parts_of(2, 3)), torch.full((3, 4), 6.0))


@pytest.mark.parametrize("arrangement", ["pre_norm", "sandwich_norm", "parallel"])
def test_a_layer_that_adds_rows_takes_a_branch_in_parts(arrangement):
    """The layer in front leaves the parts of its last product; this one's first norm adds rows in its own kernel and
    knows no parts."""
    from cie_amd.parts.block import BranchNormBlock, ParallelBlock, PreNormBlock, SandwichNormBlock  # noqa: F401

    class Mixer:
        def forward(self, x, batch, view, writes=True):
            return x

    kind = {"pre_norm": PreNormBlock, "sandwich_norm": SandwichNormBlock, "parallel": ParallelBlock}[arrangement]
    block = kind.__new__(kind)
    block.norm1, block.mixer, block.has_feed_forward, block.dtype = Norm(), Mixer(), False, torch.float32
    block.joined, block.side = False, None
    residual, seen = torch.ones(3, 4), []
    if arrangement == "sandwich_norm":
        class Out:
            def joins_into(self, then):
                return False

            def add_normed(self, residual, branch, dtype, **_):
                seen.append(branch)

        block.norm1_out, block.scale1 = Out(), None
    _, pending = block.forward(residual, parts_of(2, 3), None, None, plus=torch.full((3, 4), 0.5))
    assert torch.equal(residual, torch.full((3, 4), 6.5))
    assert torch.equal(seen[0] if seen else pending, residual)


def test_a_variant_with_a_forward_of_its_own_is_not_given_what_its_base_declares():
    from cie_amd.parts.attention import Attention
    from cie_amd.parts.base import declares
    from cie_amd.parts.feed_forward import GatedMLP

    class Reuses(GatedMLP):
        pass

    class Plain(GatedMLP):
        def forward(self, x, residual=None):
            return x

    class Own(GatedMLP):
        sums_parts = True

        def forward(self, x, residual=None, sums_parts=False):
            return x

    class Shaped(Attention):
        def shape_projection(self, qkv, batch):
            return qkv

    class Declines(GatedMLP):
        sums_parts = False

    of = lambda kind: declares(kind.__new__(kind), "sums_parts")  # noqa: E731
    assert [of(k) for k in (GatedMLP, Reuses, Plain, Own, Attention, Shaped, Declines)] == [True, True, False, True, True, True, False]


def test_products_of_many_rows_on_the_host_are_torchs():
    from cie_amd.parts.linear import choose_tiles, linear

    g = torch.Generator().manual_seed(1)
    x, w = torch.randn(200, 512, generator=g).bfloat16(), torch.randn(96, 512, generator=g).bfloat16()
    assert choose_tiles(200, 96, 512, 512) is not None  # (on the GPU this product goes to the tiles)
    assert torch.equal(linear(x, w), torch.nn.functional.linear(x, w))
    assert torch.equal(linear(x, w, into=torch.zeros(200, 96)), torch.nn.functional.linear(x, w))


@pytest.mark.parametrize("rows,columns,k", [(2100, 3584, 18944), (4100, 2048, 11008), (1500, 3584, 18944), (20, 896, 4864),
                                            (70000, 1024, 4096), (64, 152064, 8192), (517, 2048, 11008)])
def test_float32_products_in_stretches_keep_their_workspace_bounded(rows, columns, k):
    from cie_amd.kernels import ops

    bands, band = ops.f32_bands(rows, columns, k)
    assert band % 64 == 0 and (bands - 1) * band < rows <= bands * band
    held = -(-k // ops.F32_STRETCH) * min(rows, band) * columns * 4
    assert held <= ops.F32_WORKSPACE_BYTES or (band == 64 and ops.plan_gemm_f32(rows, columns, k) != 2)
    if (rows, columns, k) == (1500, 3584, 18944):  # (2,005 us in whole tiles, 1,878 in stretches at once)
        assert (bands, band) == (2, 768) and ops.plan_gemm_f32(rows, columns, k) == 2


# (what stands behind it, whether in parts of K, rows, columns, K, us by the library with the kernel behind it, {tiles: us}),
# as measured on MI355X: products for which earlier rules took tiles that were slower than the library, and products whose
# tiles are much the faster ones
MEASURED = [
    ("BRANCH", 8, 613, 3584, 18944, 152.5, {(256, 160, 4): 115.0}),
    ("BRANCH", 8, 680, 3584, 18944, 168.5, {(192, 192, 3): 111.2}),
    ("BRANCH", 8, 768, 3584, 18944, 160.5, {(192, 192, 3): 111.0}),
    ("BRANCH", 8, 768, 896, 4864, 22.4, {(96, 128, 4): 21.9}),
    ("BRANCH", 8, 130, 3584, 3584, 24.1, {(96, 64, 2): 18.0}),
    ("BRANCH", 8, 330, 896, 896, 11.6, {(64, 64, 2): 9.8}),
    ("BRANCH", 8, 360, 2048, 2048, 15.9, {(64, 64, 1): 13.7}),
    ("BRANCH", 8, 400, 3584, 18944, 201.5, {(128, 256, 4): 80.6}),
    ("BRANCH", 1, 512, 4096, 11136, 77.2, {(96, 128, 1): 92.4}),
    ("BRANCH", 1, 512, 2560, 5120, 35.0, {(96, 64, 1): 38.8}),
    ("BRANCH", 1, 2048, 1140, 11136, 85.1, {(96, 128, 1): 94.4}),
    ("NOTHING", 1, 768, 1746, 8192, 43.9, {(96, 64, 1): 46.9}),
    ("NOTHING", 1, 512, 4516, 5632, 42.4, {(96, 128, 1): 47.8}),
    ("GATE", 1, 256, 22016, 2048, 42.0, {(192, 128, 1): 34.2}),
    ("GATE", 1, 777, 37888, 3584, 273.0, {(256, 160, 1): 202.0}),
    ("GATE", 1, 2048, 22016, 2048, 201.0, {(256, 256, 1): 167.8}),
]


@pytest.mark.parametrize("behind,parts,rows,n,k,library,tiles", MEASURED)
def test_tiles_are_taken_where_they_were_measured_to_win(behind, parts, rows, n, k, library, tiles):
    from cie_amd.parts import linear

    picked = linear.choose_tiles(rows, n, k, k, most_parts=parts, behind=getattr(linear, "BEHIND_" + behind))
    assert picked is None or (picked.direct and tiles[picked[:3]] <= 1.03 * library)
    assert picked is not None or min(tiles.values()) > 0.9 * library


# the same at row counts that do not recur, of a short K, where the two models are nearly level
MEASURED_SHORT = [
    ("NOTHING", 1, 1999, 4736, 2048, 45.4, {(256, 160, 1): 38.3}, True),
    ("NOTHING", 1, 2019, 5888, 576, 28.0, {(192, 256, 1): 18.8}, True),
    ("NOTHING", 1, 366, 704, 3392, 16.5, {(64, 64, 1): 11.5}, True),
    ("NOTHING", 1, 1310, 6656, 896, 29.1, {(192, 192, 1): 19.9}, True),
    ("NOTHING", 1, 1315, 17920, 2176, 92.5, {(192, 192, 1): 106.9}, False),
    ("NOTHING", 1, 1807, 19200, 1024, 76.5, {(192, 192, 1): 88.4}, False),
    ("NOTHING", 1, 1518, 8704, 1664, 41.5, {(256, 256, 1): 46.8}, False),
    ("NOTHING", 1, 1067, 11264, 3008, 66.4, {(256, 256, 1): 76.8}, False),
    ("GATE", 1, 1202, 16512, 3904, 258.6, {(192, 256, 1): 159.3}, True),
    ("GATE", 1, 524, 23168, 3456, 145.3, {(192, 192, 1): 100.9}, True),
    ("BRANCH", 1, 345, 1024, 4032, 26.1, {(64, 64, 1): 17.7}, True),
    ("BRANCH", 1, 565, 960, 3904, 26.9, {(64, 64, 1): 18.4}, True),
]


@pytest.mark.parametrize("behind,parts,rows,n,k,library,tiles,taken", MEASURED_SHORT)
def test_tiles_of_a_short_k_are_taken_where_they_were_measured_to_win(behind, parts, rows, n, k, library, tiles, taken):
    from cie_amd.parts import linear

    picked = linear.choose_tiles(rows, n, k, k, most_parts=parts, behind=getattr(linear, "BEHIND_" + behind))
    assert (picked is not None) == taken
    assert picked is None or (picked.direct and tiles[picked[:3]] <= 1.03 * library)


@pytest.mark.parametrize("behind", ["NOTHING", "GATE", "BRANCH", "ROTATION"])
def test_the_tiles_that_are_chosen_are_tiles_there_are(behind):
    """Over rows, widths and K: a form that the kernel has, parts of K that all have some, sums within their limit, and the
    tiles that load straight into LDS only for sizes they take; every other K has the other tiles or the library."""
    from cie_amd.kernels import ops
    from cie_amd.parts import linear

    taken = 0
    for rows in (129, 200, 256, 613, 777, 1024, 1999, 2048, 5000):
        for n in (32, 98, 896, 2048, 4608, 22016, 37888):
            for k in (64, 512, 896, 2048, 3584, 4104, 11008, 18944, 29568):
                for most in (1, 8):
                    picked = linear.choose_tiles(rows, n, k, k + 64, most_parts=most, behind=getattr(linear, "BEHIND_" + behind))
                    if picked is None:
                        continue
                    taken += 1
                    assert picked.direct == (k % 64 == 0) and 1 <= picked.parts <= most
                    assert picked[:2] in (ops.DIRECT_SHAPES if picked.direct else ops.TILE_SHAPES)
                    stretch = -(-(-(-k // picked.parts)) // 64) * 64
                    assert stretch * (picked.parts - 1) < k
                    assert picked.parts == 1 or not picked.direct or picked.parts * rows * n * 4 <= linear.PARTS_BYTES
    assert taken > 400
    # operands of 2^31 numbers and more are not the tiles' whose places are 32-bit numbers of bytes
    for rows, n, k, stride in ((256, 1 << 21, 1024, 1024), (1 << 20, 64, 1024, 2048)):
        assert not ops.direct_fits(rows, n, k, stride)
        picked = linear.choose_tiles(rows, n, k, stride)
        assert picked is None or not picked.direct


# (product, columns, rows, K, {(row tiles, waves, column tiles): us}) of 17 to 128 rows, as measured on MI355X
BLOCKS = [
    ("rope", 768, 59, 792, {(2, 4, 1): 5.64, (4, 4, 1): 7.76}),
    ("rope", 1536, 36, 1008, {(2, 4, 1): 5.71, (1, 4, 2): 5.75, (4, 4, 1): 7.36}),
    ("rope", 768, 122, 8176, {(2, 8, 1): 16.04, (1, 8, 2): 17.47, (4, 8, 2): 30.83}),
    ("rope", 4608, 118, 512, {(4, 4, 2): 8.15, (1, 4, 2): 10.53, (2, 4, 2): 10.61, (2, 4, 1): 11.24}),
    ("rope", 6144, 100, 64, {(4, 4, 2): 6.45, (1, 4, 2): 9.72, (2, 4, 2): 10.2}),
    ("rope", 10240, 50, 136, {(4, 4, 2): 6.73, (1, 4, 2): 8.61, (2, 4, 2): 10.2}),
    ("rope", 5120, 107, 600, {(4, 4, 2): 9.74, (1, 4, 2): 11.05, (2, 4, 2): 11.78}),
    ("rope", 5120, 83, 520, {(2, 4, 2): 7.77, (4, 4, 2): 9.35, (1, 4, 2): 9.76}),
    ("rope", 3072, 117, 800, {(4, 8, 2): 7.44, (2, 4, 2): 7.54, (1, 4, 2): 7.75, (4, 4, 2): 8.97}),
    ("plain", 128, 104, 904, {(2, 4, 1): 4.27, (4, 4, 1): 6.21}),
    ("plain", 912, 33, 864, {(2, 4, 1): 4.48, (4, 4, 1): 5.52}),
    ("plain", 4496, 34, 280, {(4, 4, 1): 5.61, (2, 4, 1): 6.3}),
    ("plain", 2224, 43, 352, {(4, 4, 1): 4.09, (2, 4, 1): 4.69}),
    ("plain", 4832, 35, 416, {(4, 4, 1): 5.33, (2, 4, 1): 6.49}),
    ("plain", 4000, 75, 352, {(4, 4, 1): 5.15, (2, 4, 1): 6.13}),
]


@pytest.mark.parametrize("product,n,rows,k,times", BLOCKS)
def test_blocks_of_rows_are_those_that_were_measured_to_win(product, n, rows, k, times):
    from cie_amd.kernels import ops

    if product == "rope":
        row_tiles, waves, one_tile = ops.plan_qkv_rope(rows, n // 32, k)
        plan = (row_tiles, waves, 1 if one_tile else 2)
    else:
        plan = ops.plan_fused(rows, n // 16, k)
    assert times[plan] <= 1.04 * min(times.values())


@pytest.mark.parametrize("rows", [1, 10, 16])
def test_few_rows_take_a_pair_of_column_tiles_where_that_was_measured_to_win(rows):
    """q/k/v of a short K, whose workgroups make the norm of the rows, or read them."""
    from cie_amd.kernels import ops

    one_tile = lambda k, folded: ops.plan_qkv_rope(rows, 72, k, folded)[2]  # noqa: E731
    assert [one_tile(k, True) for k in (64, 512, 824, 1024, 1032)] == [False, False, False, False, True]
    assert [one_tile(k, False) for k in (64, 512, 520, 824, 1024)] == [False, False, True, True, True]


def decode_form(monkeypatch, q_heads, kv_heads, dim, rows, longest, bound=None, unmerged=False, page=16):
    """(waves a part, parts, whether they come back unmerged) of a step of ``rows`` single tokens over up to ``longest`` keys, launch by
    launch, or as captured for up to ``bound`` keys."""
    from cie_amd.engine.batch import PagedView, StepBatch
    from cie_amd.engine.graphs import StaticPlan
    from cie_amd.kernels import ops
    from cie_amd.parts import attention

    ints = lambda values: torch.tensor(list(values), dtype=torch.int32)  # noqa: E731
    starts = [longest - 1 - i % min(longest, 7) for i in range(rows)]
    step = StepBatch(tokens=rows, sequences=rows, token_ids=ints([0] * rows), positions=ints(starts), seq_of_token=ints(range(rows)),
                     seq_slot=ints(range(rows)), seq_start=ints(starts), seq_q_len=ints([1] * rows), q_start_loc=ints(range(rows + 1)),
                     logit_rows=ints([0]), host_slots=list(range(rows)), host_starts=starts, host_q_lens=[1] * rows,
                     static_plan=None if bound is None else StaticPlan(ints(range(rows)), ints([0] * rows), ints([longest]), bound))
    view = PagedView(torch.empty(1, kv_heads, page, dim), torch.empty(1, kv_heads, dim, page), ints([0] * rows).view(rows, 1), page)
    calls = []
    monkeypatch.setattr(ops, "paged_attention_mfma", lambda *a, **k: calls.append((k["tile_waves"], k["n_splits"], not k["merge"])))
    out = attention.attend(torch.empty(rows, (q_heads + 2 * kv_heads) * dim, dtype=torch.bfloat16), step, view, q_heads, kv_heads, dim, None,
                           dim ** -0.5, unmerged=unmerged)
    (form,) = calls
    assert form[2] == isinstance(out, attention.Shares) and (form[1] > 1 or not form[2])
    return form


@pytest.mark.parametrize("heads", [(16, 2, 128), (14, 2, 64)])
@pytest.mark.parametrize("rows", [17, 24, 32, 47])
def test_a_captured_steps_keys_are_not_cut_by_its_bound_alone(heads, rows, monkeypatch):
    """Some dozens of pairs: parts of one wave, which are the faster ones over few keys, whatever the limit (below the one from which
    every step has four waves); launch by launch the keys are known, and many of them are four waves'."""
    for bound in (1024, 1500, 2047):
        for longest in (60, 300, 1000):
            waves, parts, _ = decode_form(monkeypatch, *heads, rows, longest, bound)
            assert (waves, parts > 1) == (1, True)
    assert decode_form(monkeypatch, *heads, rows, 1600)[0] == 4
    assert decode_form(monkeypatch, *heads, rows, 60, 4096)[0] == 4
    assert decode_form(monkeypatch, *heads, rows, 300, 304)[:2] == (4, 1)  # (whole: one kernel and no merge)


@pytest.mark.parametrize("page", [8, 16])
def test_shares_that_are_planned_for_the_output_product_are_left_to_it(page, monkeypatch):
    """Up to 16 single tokens, at bounds that give more parts than the output product takes: a form of which it takes all, or, with
    pages that have no such form, the one with a merge of its own."""
    for heads in ((8, 1, 128), (16, 1, 64), (16, 2, 128), (14, 2, 64), (28, 4, 128), (32, 8, 64)):
        for rows in range(1, 17):
            for bound in (None, 300, 1000, 2040, 4096, 16384, 32768, 131072):
                longest = 20000 if bound is None else min(bound, 1000)
                waves, parts, unmerged = decode_form(monkeypatch, *heads, rows, longest, bound, unmerged=True, page=page)
                if page >= 16:
                    assert unmerged == (parts > 1)
                elif parts > 1 and not unmerged:
                    assert (waves, parts) == decode_form(monkeypatch, *heads, rows, longest, bound, page=page)[:2]


def test_which_portions_take_the_form_through_lds():
    from cie_amd.parts.attention import takes_prompt_form

    assert takes_prompt_form(192, 200, 8, True, 256)  # many tiles: whatever is beside them
    assert not takes_prompt_form(191, 100_000, 8, False, 256) and not takes_prompt_form(191, 100_000, 32, False, 256)
    assert takes_prompt_form(191, 100, 0, True, 256) and takes_prompt_form(141, 100, 33, False, 256)
    assert not takes_prompt_form(140, 685, 0, False, 256) and takes_prompt_form(140, 686, 0, False, 256)
    assert not takes_prompt_form(140, 100_000, 0, True, 256)  # (a captured step's keys are not known)
    assert not takes_prompt_form(0, 100_000, 0, False, 256)


@pytest.mark.parametrize("window,page", [(None, 16), (1024, 32), (1024, 16)])
@pytest.mark.parametrize("singles,single_start,portion,portion_start,through_lds", [
    (40, 3999, 200, 0, False),    # 50 tiles over 200 keys: the 40 tokens' 4,000 keys are not theirs
    (40, 99, 200, 1800, True),    # ... over 2,000
    (40, 99, 200, 1700, False),   # (95,000 tiles x keys)
    (0, 0, 200, 1800, True), (0, 0, 400, 1000, True)])
def test_the_keys_of_the_portions_choose_their_form(monkeypatch, window, page, singles, single_start, portion, portion_start, through_lds):
    """Single tokens beside the portions have a launch of their own here; their contexts do not choose the portions' form.  (A
    window of 1,024 keys leaves the portions some 1,088; with pages of 16 few tiles do not take the form for its keys.)"""
    from cie_amd.engine.batch import PagedView, StepBatch
    from cie_amd.kernels import ops
    from cie_amd.parts import attention

    waves = []
    monkeypatch.setattr(ops, "compute_units", lambda *_: 256)
    monkeypatch.setattr(ops, "paged_attention_mfma", lambda *a, **k: waves.append((k["tokens_per_tile"], k["tile_waves"])))
    q_lens, starts = [1] * singles + [portion], [single_start] * singles + [portion_start]
    total = sum(q_lens)
    some = torch.zeros(total + 1, dtype=torch.int32)
    batch = StepBatch(tokens=total, sequences=len(q_lens), token_ids=some, positions=some, seq_of_token=some, seq_slot=some,
                      seq_start=some, seq_q_len=some, q_start_loc=some, logit_rows=some, host_slots=list(range(len(q_lens))),
                      host_starts=starts, host_q_lens=q_lens)
    pool = torch.zeros((1, 2, page, 128), dtype=torch.bfloat16)
    view = PagedView(pool, pool.transpose(2, 3), some[None], page)
    attention.attend(torch.zeros((total, 20 * 128), dtype=torch.bfloat16), batch, view, 16, 2, 128, window, 0.1)
    keys = portion_start + portion if window is None else min(portion_start + portion, window + 64)
    tiles = -(-portion * 8 // 64) * 2
    if window is not None:
        through_lds = tiles >= 0.55 * 256 or (page == 32 and tiles * keys >= 96_000)
    assert [w for tokens, w in waves if tokens > 1] == [ops.PROMPT_WAVES if through_lds else ops.TILE_WAVES]


@pytest.mark.parametrize("rows", [17, 41, 64, 65, 128])
@pytest.mark.parametrize("n,k", [(896, 4864), (2048, 11008), (3584, 18944), (5120, 5120), (64, 64), (9728, 896), (22016, 2048), (40000, 64)])
@pytest.mark.parametrize("most", [1, 8])
def test_tiles_of_few_rows_meet_the_units_once(rows, n, k, most):
    from cie_amd.kernels import ops
    from cie_amd.parts.linear import plan_few_tiles

    form = plan_few_tiles(rows, n, k, most, 256)
    if form is None:
        assert min(-(-n // 128) * -(-rows // r) for r in ((64,) if rows <= 64 else (64, 128))) > 256
        return
    columns, tile_rows, parts = form
    assert (columns, tile_rows) in ops.DIRECT_FEW_SHAPES and parts <= most
    assert -(-n // columns) * -(-rows // tile_rows) * parts <= 256
    assert -(-(-(-k // parts)) // 64) * 64 * (parts - 1) < k  # (no part without k)
    assert -(-(-(-n // columns) * -(-rows // tile_rows)) // 8) * parts <= 32  # (and an eighth of the tiles an eighth of the units)


@pytest.mark.parametrize("rows,n,k,gate,tiles", [
    # (us, the other way and the tiles, measured)
    (64, 2048, 11008, False, True), (96, 2048, 11008, False, True), (128, 3584, 18944, False, True), (72, 896, 4864, False, True),
    (96, 5120, 5120, False, True),
    (64, 5120, 22016, False, False),   # 51.7, 59.4
    (48, 6144, 8192, False, False),    # 23.0, 26.0
    (56, 8128, 8192, False, False),    # 27.4, 29.9
    (64, 6144, 24576, False, False),   # 64.5, 70.8
    (64, 9728, 896, True, True), (128, 22016, 2048, True, True), (56, 20480, 1024, True, True),
    (64, 28672, 6144, True, False),    # 65.3, 78.1
    (72, 28672, 6144, True, False),    # 71.7, 80.0
    (112, 1024, 6144, True, False),    # 15.3, 18.2
    (112, 1120, 5120, True, False),    # 14.7, 16.8
    (128, 16384, 5120, True, False)])  # 49.4, 52.4
def test_tiles_of_few_rows_where_they_are_the_faster_ones(monkeypatch, rows, n, k, gate, tiles):
    from cie_amd.kernels import ops
    from cie_amd.parts import linear

    monkeypatch.setattr(ops, "compute_units", lambda *_: 256)
    assert ((linear._gate_tiles if gate else linear._cut_tiles)(rows, n, k, 256) is not None) == tiles


def test_tiles_of_few_rows_cut_a_short_k_little():
    """4,096 x 4,096, 96 rows: 8 parts of 128 x 128 20.3 us, 2 of 64 x 64 13.7, the streaming waves 16.4."""
    from cie_amd.parts.linear import plan_few_tiles

    assert plan_few_tiles(96, 4096, 4096, 8, 256)[2] <= 4


@pytest.mark.parametrize("blocks,width,sequences,takes", [
    (16, 128, 128, True), (16, 128, 129, False), (20, 128, 128, False), (32, 64, 128, True), (40, 64, 112, False),
    (8, 256, 160, True), (8, 256, 161, False), (16, 160, 128, True), (4, 640, 128, True)])
def test_which_steps_of_single_tokens_make_their_gates_themselves(monkeypatch, blocks, width, sequences, takes):
    """Up to four workgroups a unit for blocks of up to 128 numbers, up to five for wider ones."""
    from cie_amd.kernels import ops

    monkeypatch.setattr(ops, "compute_units", lambda *_: 256)
    u = torch.zeros((sequences, blocks * width), dtype=torch.bfloat16)
    weight = torch.zeros((blocks, 2 * width, width), dtype=torch.bfloat16)
    assert ops.steps_gated_recurrence(u, weight, sequences, width, 4) == takes
