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
    from cie_amd.parts.linear import linear, plan_tiles

    g = torch.Generator().manual_seed(1)
    x, w = torch.randn(200, 512, generator=g).bfloat16(), torch.randn(96, 512, generator=g).bfloat16()
    assert plan_tiles(200, 96, 512) is not None  # (on the GPU this product goes to the tiles)
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


# (what, rows, columns, K, us by the library with the kernel behind it, {tiles: us}), as measured on MI355X: products for
# which an earlier rule took tiles that were slower than the library (the first of each), and tiles that are not
MEASURED = [
    ("down", 613, 3584, 18944, 151.2, {(128, 256, 3): 193.0, (128, 128, 3): 134.1}),
    ("down", 680, 3584, 18944, 169.8, {(128, 256, 3): 195.3, (128, 128, 3): 138.4}),
    ("down", 768, 3584, 18944, 161.5, {(128, 256, 3): 198.8, (128, 128, 3): 145.2}),
    ("down", 768, 896, 4864, 23.1, {(128, 64, 3): 28.3}),
    ("o", 130, 3584, 3584, 20.4, {(128, 64, 3): 23.5, (64, 64, 3): 19.4}),
    ("o", 330, 896, 896, 12.1, {(64, 64, 3): 11.2, (64, 64, 1): 10.6, (64, 64, 2): 10.2}),
    ("o", 360, 2048, 2048, 16.3, {(128, 64, 2): 17.8, (64, 64, 1): 16.6}),
]


@pytest.mark.parametrize("what,rows,n,k,library,tiles", MEASURED)
def test_tiles_are_not_taken_where_they_were_measured_to_lose(what, rows, n, k, library, tiles):
    from cie_amd.parts.linear import BEHIND_BRANCH, plan_tiles

    picked = plan_tiles(rows, n, k, most_parts=8, behind=BEHIND_BRANCH)
    assert picked is None or tiles[picked] <= 1.03 * library
