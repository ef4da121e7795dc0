"""The split-KV combine at split counts around its batches of four, two and one
splits and query counts around its one- and four-wave workgroups (385 x 8 heads
of 64: the first four-wave launch): against the single pass on the same inputs,
and bit-identical between runs.

Bound: both forms round P to bf16 once per key and the output once; they differ
in the running maximum that P is scaled by, so by bf16 roundings of P
(2^-9 each, averaged over the keys) and one of the output: max relative error
<= 1e-2, the gate of the attention tests.
"""

from __future__ import annotations

import pytest
import torch

from _util import max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("tq,H,dh", [(1, 1, 64), (1, 2, 128), (9, 3, 64), (130, 2, 128), (385, 8, 64)])
def test_combine_matches_single_pass(splits, tq, H, dh):
    from ltx_amd.kernels import attention as A

    gen = torch.Generator(device="cuda").manual_seed(tq + splits)
    q, k, v = (torch.randn((t, H * dh), generator=gen, device="cuda").bfloat16() for t in (tq, 577, 577))
    g = torch.rand((tq, H), generator=gen, device="cuda").bfloat16()
    out = A.flash_attention(q, k, v, H, gate=g, splits=splits)
    one = A.flash_attention(q, k, v, H, gate=g, splits=1)
    again = A.flash_attention(q, k, v, H, gate=g, splits=splits)
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))
    assert max_rel_err(out.float().cpu().numpy(), one.float().cpu().numpy()) <= 1e-2
