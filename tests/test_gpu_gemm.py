"""GPU parity of the weight-format kernels and the projection GEMMs.

* Encoders/decoders: bit-exact against the oracle (oracle/quant.py).
* In-GEMM dequantisation: bit-exact, shown with A = identity, for which
  C = I @ W'^T is exactly the decoded weight transposed.
* GEMM + epilogues: bf16 tolerance against the fp32-accumulating oracle --
  normwise max relative error <= 1e-2 (the bf16 tolerance gate), cosine >=
  0.9999 and >= 90 % of outputs bit-identical (the remainder differ by the
  fp32 summation order moving a value across a bf16 rounding boundary).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import bf16_from_torch, cos_sim, max_rel_err, ulp_diff_bf16
from oracle import quant as oq
from oracle.bf16 import bf16r

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf(rng, shape, scale=1.0):
    return bf16r(rng.standard_normal(shape).astype(np.float32) * np.float32(scale))


def _t(a, dtype=torch.bfloat16):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dtype).to(DEV)


def _weight_matrix(rng, n, k):
    W = _bf(rng, (n, k), 0.02)
    W[1] = 0.0                       # zero row / zero blocks
    W[2, :64] = bf16r(np.linspace(-3, 3, 64, dtype=np.float32))  # wide range
    W[3, 32:64] = 0.0
    return W


def test_int8_encoder_and_decoder_bitexact():
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(0)
    W = _weight_matrix(rng, 512, 4096)
    wt = gemm.make_weight(_t(W), kind="int8")
    torch.cuda.synchronize()
    q, s = oq.int8_quantize(W)
    np.testing.assert_array_equal(wt.scale.cpu().numpy(), s)
    np.testing.assert_array_equal(wt.w.cpu().numpy(), q)
    deq = bf16_from_torch(gemm.dequantize(wt))
    np.testing.assert_array_equal(deq, oq.int8_dequantize(q, s))


def test_mxfp8_encoder_and_decoder_bitexact():
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(1)
    W = _weight_matrix(rng, 512, 4096)
    W[4, :32] = bf16r(np.array([448.0 * 2 ** -3] + [1e-3] * 31, np.float32))
    wt = gemm.make_weight(_t(W), kind="mxfp8")
    torch.cuda.synchronize()
    codes, scales = oq.mxfp8_quantize(W)
    np.testing.assert_array_equal(wt.scale.cpu().numpy(), scales)
    np.testing.assert_array_equal(wt.w.cpu().numpy(), codes)
    deq = bf16_from_torch(gemm.dequantize(wt))
    np.testing.assert_array_equal(deq, oq.mxfp8_dequantize(codes, scales))


def test_mxfp8_decoder_all_codes_bitexact():
    """Every E4M3 code under a spread of E8M0 scales decodes exactly."""
    from ltx_amd import _lib

    codes = np.tile(np.arange(256, dtype=np.uint8), 8).reshape(64, 32)  # 64 blocks
    scales = np.array([127, 128, 126, 100, 150, 60, 200, 1] * 8, np.uint8).reshape(64, 1)
    ct, st = _t(codes, torch.uint8), _t(scales, torch.uint8)
    out = torch.empty((64, 32), dtype=torch.bfloat16, device=DEV)
    _lib.call("ltx_dequantize_mxfp8_bf16", ct.data_ptr(), 32, st.data_ptr(), 1, 64, 32, out.data_ptr(), 32,
              _lib.stream_of(out))
    got = bf16_from_torch(out)
    ref = oq.mxfp8_dequantize(codes, scales)
    finite = ~np.isnan(ref)
    np.testing.assert_array_equal(got[finite], ref[finite])
    assert np.isnan(got[~finite]).all()


@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp8"])
@pytest.mark.parametrize("tile", [1, 2, 3, 4])
def test_gemm_identity_returns_decoded_weight(kind, tile):
    """C = I @ W'^T: each output is one product 1.0 * w' plus exact zeros."""
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(2)
    K, N = 512, 384
    W = _weight_matrix(rng, N, K)
    wt = gemm.make_weight(_t(W), kind=kind)
    eye = torch.eye(K, dtype=torch.bfloat16, device=DEV)
    out = gemm.linear(eye, wt, tile=tile)
    deq = gemm.dequantize(wt)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bf16_from_torch(out), bf16_from_torch(deq).T)


def _decoded(kind, W):
    if kind == "bf16":
        return W
    if kind == "int8":
        return oq.int8_dequantize(*oq.int8_quantize(W))
    return oq.mxfp8_dequantize(*oq.mxfp8_quantize(W))


def _check(got, ref, min_exact=0.9):
    assert max_rel_err(got, ref) <= 1e-2
    assert cos_sim(got, ref) >= 0.9999
    assert (ulp_diff_bf16(got, ref) == 0).mean() >= min_exact


@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp8"])
@pytest.mark.parametrize("K,N", [(4096, 4096), (4096, 16384), (16384, 4096), (4096, 2048), (2048, 4096)])
def test_gemm_block_shapes(kind, K, N):
    """The projection shapes of one video block at M = 3456 tokens (the last
    two: the A2V query and output projections, 112 and 224 tiles of 256 x 256:
    by the automatic tile choice the mid-size kernel for 8-bit weights, and
    the 8-wave kernel)."""
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(K + N)
    M = 3456
    x = _bf(rng, (M, K))
    W = _bf(rng, (N, K), 0.02)
    b = bf16r(rng.standard_normal(N).astype(np.float32) * 0.02)
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    out = gemm.linear(_t(x), wt)
    torch.cuda.synchronize()
    ref = oq.linear(x, _decoded(kind, W), b, round_then_bias=kind == "mxfp8")
    _check(bf16_from_torch(out), ref)


@pytest.mark.parametrize("epi", ["bias", "gelu", "sigmoid2", "residual", "residual_round"])
@pytest.mark.parametrize("tile", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["bf16", "mxfp8"])
def test_gemm_epilogues(epi, tile, kind):
    """Every epilogue, with a non-zero bias: single rounding for bf16 weights
    (mx.addmm), bias after the bf16 product for MXFP8 (nn.QuantizedLinear)."""
    from ltx_amd.kernels import gemm

    codes = {"bias": gemm.EPI_BIAS, "gelu": gemm.EPI_GELU, "sigmoid2": gemm.EPI_SIGMOID2,
             "residual": gemm.EPI_RESIDUAL, "residual_round": gemm.EPI_RESIDUAL_ROUND}
    rng = np.random.default_rng(3)
    M, K, N = 700, 1024, 1536
    x = _bf(rng, (M, K))
    W = _bf(rng, (N, K), 0.05)
    b = bf16r(rng.standard_normal(N).astype(np.float32) * 0.1)
    res = _bf(rng, (M, N))
    g = rng.standard_normal(N).astype(np.float32) * 0.5
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    assert wt.qlinear == (kind == "mxfp8")
    rt, gt = _t(res), _t(g, torch.float32)
    if epi.startswith("residual"):  # in place on the residual stream
        out = gemm.linear(_t(x), wt, epilogue=codes[epi], out=rt, residual=rt, gate=gt, tile=tile)
        assert out.data_ptr() == rt.data_ptr()
    else:
        out = gemm.linear(_t(x), wt, epilogue=codes[epi], tile=tile)
    torch.cuda.synchronize()
    ref = oq.linear(x, _decoded(kind, W), b, epilogue=epi, residual=res, gate=g,
                    round_then_bias=kind == "mxfp8")
    _check(bf16_from_torch(out), ref, min_exact=0.85)
    if kind == "mxfp8" and epi != "sigmoid2":  # the other rounding form is measurably further away
        alt = oq.linear(x, _decoded(kind, W), b, epilogue=epi, residual=res, gate=g)
        assert (ulp_diff_bf16(bf16_from_torch(out), ref) == 0).mean() > \
            (ulp_diff_bf16(bf16_from_torch(out), alt) == 0).mean()


@pytest.mark.parametrize("M,K,N", [(1, 4096, 4096), (68, 2048, 2048), (68, 2048, 6144), (256, 4096, 8192),
                                   (3456, 4096, 32), (3456, 4096, 128), (3456, 128, 4096), (130, 64, 8)])
def test_gemm_edge_shapes(M, K, N):
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(M + K + N)
    x = _bf(rng, (M, K))
    W = _bf(rng, (N, K), 0.03)
    b = rng.standard_normal(N).astype(np.float32) * 0.02
    wt = gemm.make_weight(_t(W), _t(b, torch.float32))
    out = gemm.linear(_t(x), wt)
    torch.cuda.synchronize()
    _check(bf16_from_torch(out), oq.linear(x, W, b))


def test_gemm_strided_operands():
    """A and C as column slices of wider row-major buffers (fused QKV layout)."""
    from ltx_amd.kernels import gemm

    rng = np.random.default_rng(4)
    M, K, N = 1000, 2048, 1024
    big_x = _bf(rng, (M, 3 * K))
    W = _bf(rng, (N, K), 0.03)
    wt = gemm.make_weight(_t(W))
    xt = _t(big_x)
    outbuf = torch.zeros((M, 3 * N), dtype=torch.bfloat16, device=DEV)
    gemm.linear(xt[:, K:2 * K], wt, out=outbuf[:, 2 * N:])
    torch.cuda.synchronize()
    got = bf16_from_torch(outbuf)
    _check(got[:, 2 * N:], oq.linear(big_x[:, K:2 * K], W))
    assert not got[:, :2 * N].any()


def test_gemm_rejects_bad_shapes():
    from ltx_amd import _lib
    from ltx_amd.kernels import gemm

    wt = gemm.make_weight(torch.zeros((64, 100 * 0 + 96), dtype=torch.bfloat16, device=DEV))
    with pytest.raises(_lib.LtxKernelError):  # K = 96 is not a multiple of 64
        gemm.linear(torch.zeros((4, 96), dtype=torch.bfloat16, device=DEV), wt)


@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp8"])
@pytest.mark.parametrize("epi", ["bias", "gelu", "sigmoid2", "residual", "residual_round"])
@pytest.mark.parametrize("M,K,N,splits", [(68, 2048, 8192, 4), (68, 8192, 2048, 16), (1, 4096, 1024, 8),
                                          (100, 2048, 2080, 2), (256, 4096, 4096, 4)])
def test_gemm_splitk(kind, epi, M, K, N, splits):
    """Split-K (fp32 partials summed in split order, then the epilogue) against
    the oracle and the single-pass kernel; the gate-logit columns too."""
    from ltx_amd.kernels import gemm

    print(f"splitk {kind} {epi} M={M} K={K} N={N} s={splits}", flush=True)
    codes = {"bias": gemm.EPI_BIAS, "gelu": gemm.EPI_GELU, "sigmoid2": gemm.EPI_SIGMOID2,
             "residual": gemm.EPI_RESIDUAL, "residual_round": gemm.EPI_RESIDUAL_ROUND}
    rng = np.random.default_rng(M + K + N)
    x = _bf(rng, (M, K))
    W = _bf(rng, (N, K), 0.02)
    b = bf16r(rng.standard_normal(N).astype(np.float32) * 0.1)
    res = _bf(rng, (M, N))
    g = rng.standard_normal(N).astype(np.float32) * 0.5
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    sig = N - 32 if epi == "bias" else None

    def run(s):
        if epi.startswith("residual"):
            rt = _t(res)
            return gemm.linear(_t(x), wt, epilogue=codes[epi], out=rt, residual=rt, gate=_t(g, torch.float32),
                               splits=s)
        return gemm.linear(_t(x), wt, epilogue=codes[epi], splits=s, sigmoid_from=sig)

    split, single = bf16_from_torch(run(splits)), bf16_from_torch(run(1))
    torch.cuda.synchronize()
    ref = oq.linear(x, _decoded(kind, W), b, epilogue=epi, residual=res, gate=g, round_then_bias=kind == "mxfp8")
    if sig is not None:  # head-gate columns
        ref[:, sig:] = oq.linear(x, _decoded(kind, W), b, epilogue="sigmoid2", round_then_bias=kind == "mxfp8")[:, sig:]
    _check(split, ref, min_exact=0.85)
    assert (ulp_diff_bf16(split, single) == 0).mean() >= 0.85


def test_gemm_splitk_rejects_bad_splits():
    from ltx_amd.kernels import gemm
    from ltx_amd._lib import LtxKernelError

    wt = gemm.make_weight(torch.zeros((64, 2048), dtype=torch.bfloat16, device=DEV), kind="mxfp8")
    x = torch.zeros((4, 2048), dtype=torch.bfloat16, device=DEV)
    with pytest.raises(LtxKernelError):
        gemm.linear(x, wt, splits=32)  # 2048 % (128 * 32) != 0 for MXFP8


# ---- the 8-wave kernel (tile 5; 128-row tiles: tile 6) ----------------------
@pytest.mark.parametrize("rows", [256, 128])
@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp8"])
@pytest.mark.parametrize("K,N", [(64, 264), (192, 256), (320, 384), (512, 384), (1024, 520), (4096, 256)])
def test_gemm8_identity_returns_decoded_weight(kind, K, N, rows):
    """C = I @ W'^T through the 8-wave kernel (256- and 128-row tiles): the
    per-fragment dequantisation (scales from LDS, eight stages per octet for
    MXFP8) is bit-exact, and bf16 weights come back unchanged; K = 512 is one
    octet, 4096 eight; N = 520 leaves a ragged last tile.  The short K (bf16
    and int8 only: MXFP8 needs whole octets) cover the stage-ring remainders:
    bf16 stages are 32 deep in a ring of four, 8-bit ones 64 deep in three."""
    from ltx_amd.kernels import gemm

    if kind == "mxfp8" and K % 512:
        pytest.skip("MXFP8 on the 8-wave kernel needs K % 512 == 0")
    tile = gemm.TILE_G8 if rows == 256 else gemm.TILE_G8_128

    rng = np.random.default_rng(K + N)
    W = _weight_matrix(rng, N, K)
    W[5] = bf16r(np.logspace(-6, 2, K, dtype=np.float32) * np.sign(rng.standard_normal(K)).astype(np.float32))
    wt = gemm.make_weight(_t(W), kind=kind)
    eye = torch.eye(K, dtype=torch.bfloat16, device=DEV)
    print(f"gemm8 identity {kind} K={K} N={N} rows={rows}", flush=True)
    out = gemm.linear(eye, wt, tile=tile)
    deq = gemm.dequantize(wt)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(bf16_from_torch(out), bf16_from_torch(deq).T)


@pytest.mark.parametrize("rows", [256, 128])
@pytest.mark.parametrize("epi", ["bias", "gelu", "sigmoid2", "residual", "residual_round"])
@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp8"])
@pytest.mark.parametrize("M,K,N", [(700, 1024, 1288), (3456, 4096, 768)])
def test_gemm8_epilogues(epi, kind, M, K, N, rows):
    """Every epilogue through the 8-wave kernel (256- and 128-row tiles),
    ragged M and N, against the oracle, with the 2*sigmoid head-gate columns
    of a fused projection for the bias epilogue; in place on the residual
    stream for the gated forms."""
    from ltx_amd.kernels import gemm

    tile = gemm.TILE_G8 if rows == 256 else gemm.TILE_G8_128

    codes = {"bias": gemm.EPI_BIAS, "gelu": gemm.EPI_GELU, "sigmoid2": gemm.EPI_SIGMOID2,
             "residual": gemm.EPI_RESIDUAL, "residual_round": gemm.EPI_RESIDUAL_ROUND}
    print(f"gemm8 {kind} {epi} M={M} K={K} N={N} rows={rows}", flush=True)
    rng = np.random.default_rng(M + N + len(epi))
    x = _bf(rng, (M, K))
    W = _bf(rng, (N, K), 0.05)
    b = bf16r(rng.standard_normal(N).astype(np.float32) * 0.1)
    res = _bf(rng, (M, N))
    g = rng.standard_normal(N).astype(np.float32) * 0.5
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    sig = N - 40 if epi == "bias" else None
    rt = _t(res)
    if epi.startswith("residual"):
        out = gemm.linear(_t(x), wt, epilogue=codes[epi], out=rt, residual=rt, gate=_t(g, torch.float32),
                          tile=tile)
        assert out.data_ptr() == rt.data_ptr()
    else:
        out = gemm.linear(_t(x), wt, epilogue=codes[epi], tile=tile, sigmoid_from=sig)
    torch.cuda.synchronize()
    qlin = kind == "mxfp8"
    ref = oq.linear(x, _decoded(kind, W), b, epilogue=epi, residual=res, gate=g, round_then_bias=qlin)
    if sig is not None:
        ref[:, sig:] = oq.linear(x, _decoded(kind, W), b, epilogue="sigmoid2", round_then_bias=qlin)[:, sig:]
    _check(bf16_from_torch(out), ref, min_exact=0.85)
    # the same product as the 4-wave kernel up to the fp32 summation order
    ref_old = gemm.linear(_t(x), wt, epilogue=codes[epi], tile=gemm.TILE_256, sigmoid_from=sig,
                          **({"out": _t(res), "residual": _t(res), "gate": _t(g, torch.float32)}
                             if epi.startswith("residual") else {}))
    assert (ulp_diff_bf16(bf16_from_torch(out), bf16_from_torch(ref_old)) <= 1).mean() >= 0.99


@pytest.mark.parametrize("M,N", [(3456, 16384), (1296, 16384), (6144, 4096)])
@pytest.mark.parametrize("epi", ["bias", "gelu", "residual", "residual_round"])
@pytest.mark.parametrize("kind", ["bf16", "int8", "mxfp8"])
def test_gemm8_row_split_matches_one_launch(kind, epi, M, N):
    """At 3456 and 1296 rows x 16384 columns and 6144 rows x 4096 columns the
    automatic choice runs the first rows in 256-row tiles and the rest (384 /
    272 / 2048 rows) by a second launch of the 128-row form, whose activation,
    output and residual rows are offset views of the same buffers:
    bit-identical to one launch of 256-row tiles for every epilogue, in place
    on the residual for the gated forms, and the bias form with head-gate
    columns."""
    from ltx_amd.kernels import gemm

    codes = {"bias": gemm.EPI_BIAS, "gelu": gemm.EPI_GELU, "residual": gemm.EPI_RESIDUAL,
             "residual_round": gemm.EPI_RESIDUAL_ROUND}
    K = 512
    print(f"gemm8 row split {kind} {epi} M={M} N={N}", flush=True)
    rng = np.random.default_rng(M + len(epi))
    x = _t(_bf(rng, (M, K)))
    wt = gemm.make_weight(_t(_bf(rng, (N, K), 0.05)), _t(rng.standard_normal(N).astype(np.float32) * 0.1,
                                                        torch.float32), kind=kind)
    outs = []
    for tile in (gemm.TILE_AUTO, gemm.TILE_G8):
        if epi.startswith("residual"):
            r = _t(_bf(np.random.default_rng(7), (M, N)))
            g = _t(np.random.default_rng(8).standard_normal(N).astype(np.float32) * 0.5, torch.float32)
            out = gemm.linear(x, wt, epilogue=codes[epi], out=r, residual=r, gate=g, tile=tile)
            assert out.data_ptr() == r.data_ptr()
        else:
            out = gemm.linear(x, wt, epilogue=codes[epi], tile=tile, sigmoid_from=N - 40 if epi == "bias" else None)
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.isfinite(outs[0].float()).all()
    assert torch.equal(outs[0], outs[1])


def test_gemm8_rejects_what_it_does_not_cover():
    from ltx_amd import _lib
    from ltx_amd.kernels import gemm

    for kind, k in (("mxfp8", 1152),):  # MXFP8 K not a multiple of 512
        wt = gemm.make_weight(torch.zeros((256, k), dtype=torch.bfloat16, device=DEV), kind=kind)
        for tile in (gemm.TILE_G8, gemm.TILE_G8_128):
            with pytest.raises(_lib.LtxKernelError, match="unsupported"):
                gemm.linear(torch.zeros((300, k), dtype=torch.bfloat16, device=DEV), wt, tile=tile)
