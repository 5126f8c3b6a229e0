"""The kernel library's host side without a GPU: the entry points' argument types are read from the sources."""

from __future__ import annotations

import ctypes

import pytest

from cie_amd.kernels import library


def test_signatures_of_all_entry_points_are_read_from_the_sources():
    found = library.entry_point_signatures()
    text = "".join(path.read_text() for path in library.sources())
    assert len(found) == text.count("CIE_API int ") >= 14
    # (stream, dtype, gate_up, out, tokens, intermediate, row_sumsq, parts, hidden, eps)
    p, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    assert found["cie_silu_mul"] == [p, i, p, p, i, i, p, i, i, f]
    assert found["cie_gemm_library"][-2:] == [ctypes.c_size_t, i]
    assert all(types[0] is p for types in found.values())  # every entry point takes the stream first


@pytest.mark.parametrize("params", ["void* stream, double x", "void* stream, unsigned int n", "void* stream, int"])
def test_a_parameter_that_is_not_understood_is_an_error(tmp_path, monkeypatch, params):
    source = tmp_path / "odd.hip"
    source.write_text(f"CIE_API int cie_odd({params}) {{ return 0; }}\n")
    monkeypatch.setattr(library, "sources", lambda: [source])
    with pytest.raises(library.KernelLibraryError, match="cie_odd"):
        library.entry_point_signatures()


def test_a_product_of_no_rows_launches_nothing_and_widens_nothing():
    """Steps of prompt portions that end before their prompts want no logits: the output head is given no
    rows.  No kernel runs (none could, here without a GPU) and the weight is not touched."""
    import torch

    from cie_amd.parts.linear import linear

    weight = torch.zeros((32, 16), dtype=torch.bfloat16)
    rows = torch.empty((0, 16), dtype=torch.bfloat16)
    logits = linear(rows, weight, None, out_dtype=torch.float32)
    assert logits.shape == (0, 32) and logits.dtype == torch.float32
    gated = linear(rows, weight, None, epilogue="silu")
    assert gated.shape == (0, 16) and gated.dtype == torch.bfloat16


def test_the_fallback_build_folder_must_be_this_users_own(tmp_path, monkeypatch):
    """The folder under the temporary directory has a name anyone can guess: one that others can write
    into (or that is no folder of this user's) is neither built into nor loaded from."""
    import os

    folder = tmp_path / "cie_amd_build_me"
    monkeypatch.setattr(library, "_fallback_dir", lambda: folder)
    assert library._build_dirs()[-1] == folder and folder.stat().st_mode & 0o777 == 0o700
    os.chmod(folder, 0o777)  # as if someone else had made it before us
    assert folder not in library._build_dirs()
    os.chmod(folder, 0o755)
    assert folder in library._build_dirs()
    folder.rmdir()
    folder.symlink_to(tmp_path)  # a link is no folder of ours, wherever it points
    assert folder not in library._build_dirs()


def test_cut_products_and_silu_products_plan_by_compute_units():
    """The cut of a long K: workgroups of four waves, about one for each compute unit, no part shorter than
    ``PART_K``; the SiLU product: the fewest pairs of tiles that meet on one compute unit.  The shapes that were
    measured keep their measured choice."""
    from cie_amd.parts.linear import plan_shared_parts, plan_shared_silu

    assert plan_shared_parts(128, 11008) == (1, 4, 8)     # the 3B down product
    assert plan_shared_parts(224, 18944) == (1, 4, 4)     # 7B
    assert plan_shared_parts(320, 13824) == (2, 4, 6)     # 14B
    assert plan_shared_parts(6, 328) == (1, 4, 1) and plan_shared_parts(3, 4096) == (1, 4, 4)
    assert plan_shared_parts(500, 1 << 20) == (2, 4, 4) and plan_shared_parts(1, 1 << 20) == (1, 4, 16)
    assert plan_shared_silu(688) == (3, True)      # 3B: 230 workgroups of three waves
    assert plan_shared_silu(1184) == (3, False)    # 7B: two turns either way, three waves are less per turn
    assert plan_shared_silu(864) == (4, True)      # 14B: 216 workgroups of four
    assert plan_shared_silu(1) == (2, True)        # a narrow one: no idle waves


def test_narrow_products_of_a_long_k_take_more_parts():
    """Stretches of 512 k where eight workgroups and more stand side by side and units are left; none without K of its own."""
    from cie_amd.parts.linear import plan_shared_parts

    assert plan_shared_parts(56, 4864) == (1, 4, 10)      # the 0.5B down product
    assert plan_shared_parts(96, 8960) == (1, 4, 10)      # 1.5B: as many as there are units for
    assert plan_shared_parts(28, 4096) == (1, 4, 4) and plan_shared_parts(29, 4096) == (1, 4, 8)  # seven workgroups, eight
    assert plan_shared_parts(64, 11008) == (1, 4, 15) and plan_shared_parts(113, 4104) == (1, 4, 7)
    for tiles in (1, 3, 28, 29, 32, 40, 56, 63, 64, 96, 113, 128, 224, 257, 320, 511):
        for k in (*range(4096, 9000, 8), 8960, 11008, 13824, 16400, 18944, 29568):
            _, _, parts = plan_shared_parts(tiles, k)
            stretch = -(-(-(-k // parts)) // 128) * 128   # what the kernel gives each part
            assert 1 <= parts <= 16 and stretch * (parts - 1) < k <= stretch * parts, (tiles, k)


def test_float32_results_share_rows_only_where_the_units_have_work():
    """Heads take the form whose waves own 128 columns a workgroup; a router, an expert's gate, a mixer's or an entry's
    float32 rows, whose few workgroups would walk all of K one after another, do not (17 to 80 rows take it at any width)."""
    from cie_amd.parts.linear import shares_rows_f32

    for n, k in ((1, 2048), (32, 2048), (64, 5120), (2048, 2048), (2048, 4096), (4096, 8192), (16384, 1024)):
        assert not any(shares_rows_f32(rows, n, k) for rows in (*range(1, 17), *range(81, 129))), (n, k)
        assert all(shares_rows_f32(rows, n, k) for rows in (17, 64, 80))
    for n, k in ((151936, 896), (151936, 2048), (152064, 3584), (152064, 5120)):
        assert [rows for rows in range(1, 200) if shares_rows_f32(rows, n, k)] == list(range(4, 97))
    assert not shares_rows_f32(4, 40000, 2048) and not shares_rows_f32(16, 40000, 2048)  # a second turn of a few units
    assert not shares_rows_f32(8, 73728, 2048) and shares_rows_f32(9, 73728, 2048)
    assert shares_rows_f32(81, 65536, 4096) and not shares_rows_f32(81, 65536, 5120)


def test_a_widened_head_is_made_once_and_let_go_with_its_weight():
    import gc

    import torch

    from cie_amd.parts import linear

    weight = torch.ones((5, 3), dtype=torch.bfloat16)
    first = linear._widened(weight)
    assert first.dtype == torch.float32 and linear._widened(weight) is first
    key = id(weight)
    del weight
    gc.collect()
    assert key not in linear._WIDENED
