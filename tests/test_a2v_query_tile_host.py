"""The block's A2V query projection runs on the 8-wave kernel where that is one
partial round (100-159 tiles of 256x256), on the automatic choice elsewhere and
in an attention module on its own.  Host only: the projection call is recorded,
not run."""

from __future__ import annotations

import pytest
import torch

from ltx_amd.kernels import gemm
from ltx_amd.model.transformer import attention, transformer


class _Recorded(Exception):
    pass


def _projection(monkeypatch, tokens, kind="bf16", fused=True, **kw):
    """(function, tile) of the query projection of a 4096 -> 32 x 64 module."""
    def record(name):
        def call(x, weight, *args, tile=gemm.TILE_AUTO, **kwargs):
            raise _Recorded(name, tile)
        return call

    monkeypatch.setattr(attention, "FUSED_QNORM", fused)
    for name in ("linear", "linear_rowss"):
        monkeypatch.setattr(gemm, name, record(name))
    dtype = torch.bfloat16 if kind == "bf16" else torch.uint8
    weight = gemm.LinearWeight(kind=kind, w=torch.empty((2080, 4096), dtype=dtype))
    attn = attention.Attention(4096, 2048, 32, 64, weight, None, None, None, None)
    x, ctx = torch.empty((tokens, 4096), dtype=torch.bfloat16), torch.empty((68, 2048), dtype=torch.bfloat16)
    with pytest.raises(_Recorded) as rec:
        attn.core(x, ctx, **kw)
    return rec.value.args


@pytest.mark.parametrize("kind", ["bf16", "mxfp8"])
def test_query_tile(monkeypatch, kind):
    q = dict(q_tile=transformer.A2V_Q_TILE)
    assert transformer.A2V_Q_TILE == gemm.TILE_G8
    assert _projection(monkeypatch, 3456, kind, **q) == ("linear_rowss", gemm.TILE_G8)
    assert _projection(monkeypatch, 3456, kind, fused=False, **q) == ("linear", gemm.TILE_G8)
    assert _projection(monkeypatch, 3456, kind) == ("linear_rowss", gemm.TILE_AUTO)
    for tokens in (1296, 6144, 14640):  # below 100 tiles; 160 and more: row split
        assert _projection(monkeypatch, tokens, kind, **q)[1] == gemm.TILE_AUTO


def test_quantised_rows_have_no_choice():
    weight = gemm.LinearWeight(kind="mxfp8", w=torch.empty((2080, 4096), dtype=torch.uint8))
    rows = gemm.MxRows(torch.empty((3456, 4096), dtype=torch.uint8), torch.empty((3456, 128), dtype=torch.uint8))
    assert not gemm.single_g8_round(rows, weight)


def test_block_asks_for_it():
    """Every A2V core call of the block passes the tile."""
    import inspect

    src = inspect.getsource(transformer.BasicAVTransformerBlock)
    calls = src.count("self.audio_to_video_attn.core(")
    assert calls == 3 and src.count("q_tile=A2V_Q_TILE") == calls
