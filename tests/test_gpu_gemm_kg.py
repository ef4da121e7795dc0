"""The mid-size projection kernel (csrc/gemm_kg.hip) through the automatic
tile choice, at the edges of its tiles: each tile height (64, 128, 192 rows; the
test asks the library that its shape gets it), one row past a tile, half a tile
and one row more (a wave tile wholly past M or N), the fewest units of its rings
and counts that are no multiple of four, single pass and split-K.

Bounds: the in-GEMM dequantisation, an identity product (one product 1.0 * w per
output) and products of small whole numbers (every partial sum is exact) are
exact; the epilogues match the oracle at the GEMM gate of test_gpu_gemm.py (bf16
outputs of fp32 sums in another order).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import bf16_from_torch
from test_gpu_gemm import _bf, _check, _decoded, _t, _weight_matrix
from oracle import quant as oq
from oracle.bf16 import bf16r

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS = ["bf16", "int8", "mxfp8"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("K,N", [(512, 384), (1536, 264), (640, 136), (128, 128)])
def test_identity_returns_decoded_weight(kind, K, N):
    """C = I @ W'^T; K = 640 and 128 are not whole scale groups of MXFP8
    weights (those take the older tile kernels)."""
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(K + N)
    wt = gemm.make_weight(_t(_weight_matrix(rng, N, K)), kind=kind)
    out = gemm.linear(torch.eye(K, dtype=torch.bfloat16, device=DEV), wt, splits=1)
    np.testing.assert_array_equal(bf16_from_torch(out), bf16_from_torch(gemm.dequantize(wt)).T)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("epi", ["bias", "gelu", "sigmoid2", "residual", "residual_round"])
@pytest.mark.parametrize("M,K,N,splits", [(1, 512, 136, 1), (65, 1536, 264, 1), (100, 512, 4128, 1), (300, 1024, 4096, 1),
                                          (1024, 512, 4096, 1), (1297, 512, 4096, 1), (70, 2048, 520, 4),
                                          (130, 1024, 392, 2)])
def test_epilogues(kind, epi, M, K, N, splits):
    from ltx_amd.kernels import gemm

    codes = {"bias": gemm.EPI_BIAS, "gelu": gemm.EPI_GELU, "sigmoid2": gemm.EPI_SIGMOID2,
             "residual": gemm.EPI_RESIDUAL, "residual_round": gemm.EPI_RESIDUAL_ROUND}
    rng = np.random.default_rng(M + N + K + len(epi))
    x, W = _bf(rng, (M, K)), _bf(rng, (N, K), 0.05)
    b = bf16r(rng.standard_normal(N).astype(np.float32) * 0.1)
    res, g = _bf(rng, (M, N)), rng.standard_normal(N).astype(np.float32) * 0.5
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    sig = N - 40 if epi == "bias" else None
    # the output in a wider, longer buffer whose other elements must survive
    buf = torch.full((M + 3, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    out = buf[:M, :N]
    if epi.startswith("residual"):
        out.copy_(_t(res))
        gemm.linear(_t(x), wt, epilogue=codes[epi], out=out, residual=out, gate=_t(g, torch.float32), splits=splits)
    else:
        gemm.linear(_t(x), wt, epilogue=codes[epi], out=out, sigmoid_from=sig, splits=splits)
    assert (buf[M:] == 7.0).all() and (buf[:, N:] == 7.0).all()
    qlin = kind == "mxfp8"
    ref = oq.linear(x, _decoded(kind, W), b, epilogue=epi, residual=res, gate=g, round_then_bias=qlin)
    if sig is not None:
        ref[:, sig:] = oq.linear(x, _decoded(kind, W), b, epilogue="sigmoid2", round_then_bias=qlin)[:, sig:]
    _check(bf16_from_torch(out), ref, min_exact=0.85)


def _whole(rng, shape, lo, hi):
    return rng.integers(lo, hi + 1, shape).astype(np.float32)


# (tile height, splits, M, N): M one row, half a tile or half a tile and one row
# past whole tiles, N 8 or 72 columns past 128
HEIGHTS = [(64, 1, 1, 72), (64, 1, 33, 136), (64, 2, 32, 72), (64, 4, 65, 264),
           (128, 1, 385, 4680), (128, 1, 3392, 520), (128, 1, 449, 4168),
           (128, 2, 257, 3272), (128, 2, 2752, 264), (128, 4, 129, 2760), (128, 4, 2112, 200), (128, 4, 65, 4104),
           (192, 1, 769, 4680), (192, 1, 1056, 3656), (192, 1, 1057, 3656),
           (192, 2, 385, 4168), (192, 2, 5472, 264), (192, 4, 385, 2120), (192, 4, 288, 2760), (192, 4, 4129, 136)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("depth", ["fewest", "odd"])
@pytest.mark.parametrize("bm,splits,M,N", HEIGHTS)
def test_each_tile_height_at_its_edges(bm, splits, M, N, depth, kind):
    """Whole-number operands: x in [-1, 2], weights that each format holds
    exactly, so outputs are the oracle's bits in any order of the sums.
    ``odd``: 10 (bf16), 5 (int8) or 12 (MXFP8) units; ``fewest``: 2, 1 or 4
    (in a single pass of the taller tiles 8, 4 or 4: below, other kernels)."""
    from ltx_amd import _lib
    from ltx_amd.kernels import gemm

    per = {"odd": (640, 1536), "fewest": (128 if splits > 1 or bm == 64 else 512, 512)}[depth][kind == "mxfp8"]
    K = per * splits
    assert _lib.lib().ltx_gemm_auto_rows(M, N, K, gemm._WFORMAT[kind], splits) == bm
    print(f"{kind} {M} x {K} -> {N} rows {bm} splits {splits}", flush=True)
    rng = np.random.default_rng(M + N + K)
    x, W = _whole(rng, (M, K), -1, 2), _whole(rng, (N, K), -4, 4)
    if kind == "int8":  # 127 in every row: a scale of exactly one
        W[:, 0] = 127.0
    b, res = _whole(rng, N, -8, 8), _whole(rng, (M, N), -64, 64)
    gate = np.float32(0.5) * np.ones(N, np.float32)
    np.testing.assert_array_equal(_decoded(kind, W), W)
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    buf = torch.full((M + 2, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    out = buf[:M, :N]
    qlin = kind == "mxfp8"
    gemm.linear(_t(x), wt, out=out, splits=splits)
    ref = oq.linear(x, W, b, epilogue="bias", round_then_bias=qlin)
    np.testing.assert_array_equal(bf16_from_torch(out), ref)
    gemm.linear(_t(x), wt, epilogue=gemm.EPI_RESIDUAL, out=out, residual=_t(res), gate=_t(gate, torch.float32),
                splits=splits)
    ref = oq.linear(x, W, b, epilogue="residual", residual=res, gate=gate, round_then_bias=qlin)
    np.testing.assert_array_equal(bf16_from_torch(out), ref)
    assert (buf[M:] == 7.0).all() and (buf[:, N:] == 7.0).all()


@pytest.mark.parametrize("kind", KINDS)
def test_tile_heights_and_strides_agree(kind):
    """The k order of an output does not depend on the tile height: rows of a
    300-row and a 1297-row product (64- and 192-row tiles) of the same inputs
    are the same bits, from contiguous and from strided activations."""
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(3)
    x = _t(_bf(rng, (1297, 1024)))
    wt = gemm.make_weight(_t(_bf(rng, (4096, 1024), 0.05)), kind=kind)
    wide = torch.zeros((1297, 1032), dtype=torch.bfloat16, device=DEV)
    wide[:, :1024] = x
    full = gemm.linear(x, wt, splits=1)
    assert torch.equal(full, gemm.linear(wide[:, :1024], wt, splits=1))
    assert torch.equal(full[:300], gemm.linear(x[:300], wt, splits=1))


def test_auto_splits_only_where_tiles_leave_cus_idle():
    from ltx_amd.kernels import gemm

    assert gemm.auto_splits(3456, 4096, 4096, "mxfp8") == 1
    assert gemm.auto_splits(1296, 4096, 16384, "mxfp8") == 1
    assert gemm.auto_splits(0, 4096, 4096, "mxfp8") == 1
    s = gemm.auto_splits(68, 2048, 8192, "mxfp8")
    assert s > 1 and 8192 % (512 * s) == 0
