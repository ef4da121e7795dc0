"""The mid-size projection kernel (csrc/gemm_kg.hip) through the automatic
tile choice, at the edges of its tiles: every tile height (64, 128, 192 rows),
one row, partial tiles in both directions, a wave tile wholly past M or N, the
fewest units of its rings (K = 128 bf16 / int8, 512 MXFP8) and an odd number
of units, and its split-K form.

Bounds: the in-GEMM dequantisation and an identity product are exact (one
product 1.0 * w per output); the epilogues match the oracle at the GEMM gate
of test_gpu_gemm.py (bf16 outputs of fp32 sums in another order).
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
