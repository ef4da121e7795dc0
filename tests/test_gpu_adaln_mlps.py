"""The grouped timestep MLPs (ltx_adaln_mlps_f32) give the bits of one
sinusoid and three GEMV calls per MLP: both row widths of the kernel, a row
count that is no multiple of a workgroup's pass, mixed groups, more jobs than
one call takes, and replays of a captured call.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _mlp(dim, num, gen):
    from ltx_amd.model.transformer.timestep_embedding import AdaLayerNormSingle

    m = AdaLayerNormSingle(dim, num, generator=gen, std=0.05)
    for b in (m.b1, m.b2, m.b):
        b.normal_(0.0, 0.1, generator=gen)
    return m


def _one_by_one(m, t, mult):
    from ltx_amd import _lib

    s = _lib.stream_of(t)
    sin, h1, h2 = (torch.empty(n, device="cuda") for n in (256, m.dim, m.dim))
    out = torch.empty(m.num_embeddings * m.dim, device="cuda")
    _lib.call("ltx_timestep_embedding_f32", t.data_ptr(), 1, mult, sin.data_ptr(), 256, s)
    for x, w, b, y, k, n, flags in ((sin, m.w1, m.b1, h1, 256, m.dim, _lib.GEMV_SILU_OUTPUT),
                                    (h1, m.w2, m.b2, h2, m.dim, m.dim, 0),
                                    (h2, m.w, m.b, out, m.dim, out.numel(), _lib.GEMV_SILU_INPUT)):
        _lib.call("ltx_gemv_f32_bf16w", x.data_ptr(), 1, k, w.data_ptr(), b.data_ptr(), y.data_ptr(), n, flags, s)
    return out, h2


@pytest.mark.parametrize("shapes", [[(4096, 2)], [(2048, 9), (4096, 1)], [(8, 1)], [(264, 3), (2056, 1), (2048, 1)],
                                    [(64 + 8 * i, 1 + i % 3) for i in range(11)]])
def test_grouped_equals_one_by_one(shapes):
    from ltx_amd.model.transformer.timestep_embedding import run_mlps

    gen = torch.Generator(device="cuda").manual_seed(len(shapes))
    mlps = [_mlp(d, n, gen) for d, n in shapes]
    ts = [torch.tensor([0.03 + 0.09 * i], device="cuda") for i in range(len(mlps))]
    jobs = [(m, t, 1000.0, torch.full((m.num_embeddings * m.dim,), 7.0, device="cuda"),
             torch.empty(m.dim, device="cuda") if i % 2 == 0 else None) for i, (m, t) in enumerate(zip(mlps, ts))]
    run_mlps(jobs)

    def check():
        for m, t, mult, out, emb in jobs:
            ref, ref_emb = _one_by_one(m, t, mult)
            assert torch.equal(out, ref)
            assert emb is None or torch.equal(emb, ref_emb)

    check()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run_mlps(jobs)
    for step in range(3):
        for t in ts:
            t.mul_(0.7)
        graph.replay()
        check()
