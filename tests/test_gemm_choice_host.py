"""The library's automatic GEMM choices (host code of csrc/gemm.hip), without a
GPU: split counts for every depth the entry points take, the entry that
linear() calls, and which products the mid-size kernel takes."""

from __future__ import annotations

import pytest
import torch

KINDS = ["bf16", "int8", "mxfp8"]


@pytest.fixture(scope="module")
def gemm():
    from ltx_amd import _lib
    from ltx_amd.kernels import gemm

    if not _lib.LIB_PATH.exists():
        pytest.skip("libltx_hip.so not built")
    return gemm


@pytest.mark.parametrize("m,n,k,kind,least", [
    (77, 2048, 188160, "bf16", 5),   # 188160 / 4 is no multiple of 128
    (26, 2048, 188160, "bf16", 5),
    (59, 248, 8448, "int8", 3),      # 8448 = 128 * 66
    (1, 648, 10368, "int8", 3),      # 10368 = 128 * 81
    (68, 4096, 3840, "mxfp8", 2),    # no multiple of 512: 128x128 tiles
    (68, 2048, 1280, "mxfp8", 2),
    (2, 448, 20224, "mxfp8", 2),
    (3, 3480, 4736, "int8", 2),      # 37 units, split in halves of 64 k
])
def test_few_row_products_split_at_any_depth(gemm, m, n, k, kind, least):
    assert gemm.auto_splits(m, n, k, kind) >= least


@pytest.mark.parametrize("kind", KINDS)
def test_split_counts_are_counts_the_entry_points_take(gemm, kind):
    unit = 128 if kind == "mxfp8" else 64
    for m in (1, 26, 77, 256, 300, 1024):
        for n in (8, 264, 2048, 4128):
            for k in range(unit, 20000, 11 * unit):
                s = gemm.auto_splits(m, n, k, kind)
                assert 1 <= s <= 64 and k % (unit * s) == 0
                assert s == 1 or k // s >= 256


@pytest.mark.parametrize("m,n,k,splits", [(68, 2048, 8192, 4), (121, 2048, 2048, 4), (256, 4096, 4096, 1),
                                          (257, 2048, 8192, 1), (68, 2048, 512, 1)])
def test_explicit_128_tiles_still_split(gemm, monkeypatch, m, n, k, splits):
    """linear() on explicit 128x128 tiles splits few-row products by the
    block budget of those tiles."""
    calls = []
    monkeypatch.setattr(gemm._lib, "call", lambda name, *args, detail="": calls.append((name, args)))
    monkeypatch.setattr(gemm._lib, "stream_of", lambda t: 0)
    weight = gemm.LinearWeight(kind="bf16", w=torch.empty((n, k), dtype=torch.bfloat16))
    gemm.linear(torch.empty((m, k), dtype=torch.bfloat16), weight, tile=gemm.TILE_128)
    (name, args), = calls
    assert name == ("ltx_gemm_splitk_bf16" if splits > 1 else "ltx_gemm_bf16")
    assert splits == 1 or args[15] == splits


def _rows(gemm, m, n, k, kind, splits=1):
    """Tile height of an automatic launch on the mid-size kernel, 0: another kernel."""
    return gemm._lib.lib().ltx_gemm_auto_rows(m, n, k, gemm._WFORMAT[kind], splits)


@pytest.mark.parametrize("kind", KINDS)
def test_shallow_products_of_many_tiles_keep_the_older_kernels(gemm, kind):
    """The latent projections (K = 128): the mid-size kernel only where its
    64-row tiles are one round."""
    for m, n in ((700, 4096), (1296, 4096), (1728, 4096), (1296, 2048)):
        assert _rows(gemm, m, n, 128, kind) == 0 and _rows(gemm, m, n, 256, kind) == 0
    if kind != "mxfp8":  # MXFP8: whole groups of 512
        assert _rows(gemm, 700, 2048, 128, kind) == 64 and _rows(gemm, 68, 2048, 256, kind) == 64
    assert _rows(gemm, 1296, 4096, 512, kind) > 0
