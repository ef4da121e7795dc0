"""The timestep MLPs' descriptors (run_mlps), without a launch: the scratch rows
that the kernels write as fp32 are disjoint and inside their allocation, also
where a program has set another default dtype."""

from __future__ import annotations

import ctypes

import pytest
import torch

from ltx_amd.model.transformer import timestep_embedding as te


@pytest.mark.parametrize("default", [torch.float32, torch.bfloat16, torch.float64])
def test_scratch_rows(monkeypatch, default):
    dims = [64 + 8 * (i % 3) for i in range(11)]  # more jobs than one call takes
    row = lambda n: torch.zeros(n, dtype=torch.float32)  # noqa: E731
    before = torch.get_default_dtype()
    torch.set_default_dtype(default)
    try:
        mlps = [te.AdaLayerNormSingle(d, 2, device="cpu") for d in dims]
    finally:
        torch.set_default_dtype(before)
    assert all(b.dtype == torch.float32 for m in mlps for b in (m.b1, m.b2, m.b))
    jobs = [(m, row(1), 1000.0, row(2 * m.dim), row(m.dim) if i % 2 else None) for i, m in enumerate(mlps)]
    allocated, spans, empty = [], [], torch.empty

    def recorded(*args, **kwargs):
        t = empty(*args, **kwargs)
        allocated.append((t.data_ptr(), t.numel() * t.element_size()))
        return t

    def call(name, mlp_array, count, stream, detail=""):
        assert name == "ltx_adaln_mlps_f32"
        args = (te._MlpArgs * count).from_address(mlp_array)
        start, size = allocated[-1]
        for a in args:
            job = jobs[len(spans)]
            rows = [a.h1] + ([a.h2] if job[4] is None else [])
            assert job[4] is None or a.h2 == job[4].data_ptr()
            assert all(start <= r and r + 4 * a.dim <= start + size for r in rows)
            assert all(b - a_ >= 4 * a.dim for a_, b in zip(sorted(rows), sorted(rows)[1:]))
            spans.append((min(rows), max(rows) + 4 * a.dim))

    monkeypatch.setattr(te.torch, "empty", recorded)
    monkeypatch.setattr(te._lib, "call", call)
    monkeypatch.setattr(te._lib, "stream_of", lambda t: 0)
    torch.set_default_dtype(default)
    try:
        te.run_mlps(jobs)
    finally:
        torch.set_default_dtype(before)
    assert len(spans) == len(jobs) and len(allocated) == 2
    for part in (sorted(spans[:8]), sorted(spans[8:])):
        assert all(a[1] <= b[0] for a, b in zip(part, part[1:]))
