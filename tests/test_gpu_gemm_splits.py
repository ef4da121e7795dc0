"""Automatic split-K at depths that are no power-of-two multiple of a kernel's
unit (odd counts on the mid-size kernel, halves on 128x128 tiles), against the
oracle at the GEMM gate of test_gpu_gemm.py: bf16 outputs of fp32 sums in
another order.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import bf16_from_torch
from test_gpu_gemm import _bf, _check, _decoded, _t
from oracle import quant as oq
from oracle.bf16 import bf16r

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,M,K,N", [("bf16", 77, 18816, 264), ("bf16", 1, 10368, 648), ("int8", 9, 8448, 136),
                                        ("int8", 3, 4736, 392), ("mxfp8", 68, 3840, 520), ("mxfp8", 129, 1280, 264),
                                        ("mxfp8", 33, 10752, 200)])
def test_automatic_splits_at_odd_depths(kind, M, K, N):
    from ltx_amd.kernels import gemm

    assert gemm.auto_splits(M, N, K, kind) > 1
    rng = np.random.default_rng(K + N)
    x, W = _bf(rng, (M, K)), _bf(rng, (N, K), 0.05)
    b = bf16r(rng.standard_normal(N).astype(np.float32) * 0.1)
    wt = gemm.make_weight(_t(W), _t(b, torch.float32), kind=kind)
    out = gemm.linear(_t(x), wt)
    ref = oq.linear(x, _decoded(kind, W), b, epilogue="bias", round_then_bias=kind == "mxfp8")
    _check(bf16_from_torch(out), ref, min_exact=0.85)
