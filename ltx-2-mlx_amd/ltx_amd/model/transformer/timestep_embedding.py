"""AdaLN timestep MLPs on the per-step scalar timestep (timestep_embedding.py).

``AdaLayerNormSingle(t) -> (emb (N*D), embedded_timestep (D))`` with
sinusoid(256, flip_sin_to_cos, shift 0) -> linear_1 -> SiLU -> linear_2
(= embedded_timestep) -> SiLU -> linear(D -> N*D) (:126-201).  The three
layers run as fp32-activation / bf16-weight GEMV kernels, each layer of all the
MLPs of a step in one launch (:func:`run_mlps`); the final layer writes
straight into a slice of the caller's modulation-row buffer.
"""

from __future__ import annotations

import ctypes

import torch

from ... import _lib

SINUSOID_DIM = 256
MAX_MLPS = 8  # per ltx_adaln_mlps_f32 call


class _MlpArgs(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("t", "w1", "b1", "w2", "b2", "w", "b", "h1", "h2", "out")] + [
        ("dim", ctypes.c_int64), ("num", ctypes.c_int64), ("multiplier", ctypes.c_float)]


def run_mlps(jobs: list, scratch: list | None = None) -> None:
    """Run independent timestep MLPs together: each job is (mlp, t_value,
    multiplier, out, embedded or None), as for ``AdaLayerNormSingle.__call__``;
    ``scratch``: (hidden, embedded) fp32 rows per job (default: allocated)."""
    for i in range(0, len(jobs), MAX_MLPS):
        part = jobs[i:i + MAX_MLPS]
        dev = part[0][3].device
        rows = (torch.empty((len(part), 2, max(j[0].dim for j in part)), dtype=torch.float32, device=dev)
                if scratch is None else scratch[i:i + MAX_MLPS])
        args = (_MlpArgs * len(part))()
        for a, h, (m, t, mult, out, embedded) in zip(args, rows, part):
            h2 = h[1] if embedded is None else embedded
            a.t, a.w1, a.b1, a.w2, a.b2 = t.data_ptr(), m.w1.data_ptr(), m.b1.data_ptr(), m.w2.data_ptr(), m.b2.data_ptr()
            a.w, a.b, a.h1, a.h2, a.out = m.w.data_ptr(), m.b.data_ptr(), h[0].data_ptr(), h2.data_ptr(), out.data_ptr()
            a.dim, a.num, a.multiplier = m.dim, m.num_embeddings, float(mult)
        _lib.call("ltx_adaln_mlps_f32", ctypes.addressof(args), len(part), _lib.stream_of(part[0][3]),
                  detail=f"{len(part)} timestep MLPs")


class AdaLayerNormSingle:
    def __init__(self, dim: int, num_embeddings: int, *, device="cuda", generator: torch.Generator | None = None,
                 std: float = 0.02, init: str = "random"):
        g = generator

        def rnd(shape):
            if init == "empty":  # storage for a checkpoint loader
                return torch.empty(shape, dtype=torch.bfloat16, device=device)
            return (torch.randn(shape, generator=g, device=device, dtype=torch.float32) * std).to(torch.bfloat16)

        def zeros(n):
            return torch.zeros(n, dtype=torch.float32, device=device)

        self.dim = dim
        self.num_embeddings = num_embeddings
        self.w1, self.b1 = rnd((dim, SINUSOID_DIM)), zeros(dim)
        self.w2, self.b2 = rnd((dim, dim)), zeros(dim)
        self.w, self.b = rnd((num_embeddings * dim, dim)), zeros(num_embeddings * dim)

    def nbytes(self) -> int:
        return sum(t.numel() * t.element_size() for t in (self.w1, self.b1, self.w2, self.b2, self.w, self.b))

    def __call__(self, t_value: torch.Tensor, multiplier: float, out: torch.Tensor,
                 embedded: torch.Tensor | None = None, scratch: tuple | None = None) -> None:
        """t_value: fp32 device scalar (1,); writes emb (N*D) into ``out`` and,
        if given, embedded_timestep (D) into ``embedded``."""
        run_mlps([(self, t_value, multiplier, out, embedded)], None if scratch is None else [scratch[1:]])
