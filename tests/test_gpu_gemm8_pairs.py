"""The 8-wave kernel's rings of stage pairs (csrc/gemm.hip): identity products,
exact (one product 1.0 * w per output), at the depths where the order of the
rings can go wrong -- one stage, an odd stage count (half a pair of int8 codes),
every remainder of a ring turn -- with both tile heights and strided weights.
That no load leaves its row is not visible in outputs (the bytes of a missing
stage are never multiplied); the host checks enumerate the addresses.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import bf16_from_torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", ["TILE_G8", "TILE_G8_128"])
@pytest.mark.parametrize("kind,K", [("int8", 64), ("int8", 128), ("int8", 192), ("int8", 320), ("int8", 448),
                                    ("int8", 832), ("mxfp8", 512), ("mxfp8", 1024), ("mxfp8", 1536),
                                    ("bf16", 64), ("bf16", 128), ("bf16", 192), ("bf16", 448)])
def test_identity_at_ring_remainders(kind, K, tile):
    from ltx_amd.kernels import gemm

    N = 264
    gen = torch.Generator(device="cuda").manual_seed(K)
    wt = gemm.make_weight(torch.randn((N, K), generator=gen, device="cuda").bfloat16(), kind=kind)
    ref = bf16_from_torch(gemm.dequantize(wt)).T
    wide = torch.zeros((N, K + 64), dtype=wt.w.dtype, device="cuda")
    wide[:, 64:] = wt.w
    wt.w = wide[:, 64:]
    x = torch.eye(K, dtype=torch.bfloat16, device="cuda")
    out = gemm.linear(x, wt, tile=getattr(gemm, tile))
    np.testing.assert_array_equal(bf16_from_torch(out), ref)
