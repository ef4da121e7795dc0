"""The denoise path's workloads, as cases that a timing program can prepare, run and check.

A case is a dict of plain values.  ``prepare(case, seed)`` builds what a program holds before the call
(resident weights, RoPE tables, modulation rows, activations; for the whole step the captured HIP graph),
``run(state)`` is one pass through the public entry points, ``exact(case, seed)`` the same result in
float64 with plain torch, ``work(case)`` the bytes and flops that no implementation can do without.

Kinds:
  modulate        the fused AdaLN operator and the gated residual add on (1, T, C) rows
  self_attention  the gated self-attention module (fused QKV projection, QK-norm + RoPE, attention, output)
  text_attention  the text cross-attention module
  a2v / v2a       the cross-modal attention modules (video queries on audio keys, and the reverse)
  feed_forward    Linear -> GELU -> Linear
  connector       text features through the register-extended 1-D connector (the prompt's encoding)
  block           one audio+video block, ``passes`` sequences stacked by rows (a guided step's passes)
  step            a captured denoise step: patchify, timestep MLPs, ``layers`` blocks, heads, Euler
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "ltx-2-mlx_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

VIDEO, AUDIO = dict(dim=4096, heads=32, dim_head=128), dict(dim=2048, heads=32, dim_head=64)
EPS = 1e-6


def listed() -> list[dict]:
    return [
        # one AdaLN + gated add of a 512x288x65 clip's video rows: a launch is a few microseconds
        dict(name="modulate_1296", kind="modulate", tokens=1296, channels=4096),
        # the same operators on a long clip's rows
        dict(name="modulate_14640", kind="modulate", tokens=14640, channels=4096),
        # the audio stream of a 768x512x65 clip: few rows, the weight bytes dominate
        dict(name="audio_feed_forward_68_mxfp8", kind="feed_forward", stream="audio", tokens=68, weights="mxfp8"),
        dict(name="audio_self_attention_68_mxfp8", kind="self_attention", stream="audio", tokens=68,
             weights="mxfp8"),
        # audio queries over all video tokens: few queries, many keys
        dict(name="v2a_68x3456_mxfp8", kind="v2a", tokens=3456, audio=68, weights="mxfp8"),
        # text conditioning of a 512x288x65 clip (9 x 9 x 16 tokens, no multiple of a tile)
        dict(name="text_attention_1296x256_mxfp8", kind="text_attention", stream="video", tokens=1296, text=256,
             weights="mxfp8"),
        # the video self-attention of a 768x512x121 clip
        dict(name="self_attention_6144_mxfp8", kind="self_attention", stream="video", tokens=6144,
             weights="mxfp8"),
        # the feed-forward of a 768x512x65 clip with int8 weights
        dict(name="feed_forward_3456_int8", kind="feed_forward", stream="video", tokens=3456, weights="int8"),
        # a prompt's encoding: 77 text tokens extended to 1024 rows, bf16 weights as the connector loads them
        dict(name="connector_77_bf16", kind="connector", text=77, weights="bf16"),
        # a whole block on a short low-resolution clip, bf16 weights, called eagerly: many small launches
        dict(name="block_384_bf16", kind="block", tokens=384, audio=26, text=256, weights="bf16", passes=1),
        # the three stacked passes (prompt, negative prompt, perturbed) of a guided step at 512x288x65
        dict(name="block_guided_1296_mxfp8", kind="block", tokens=1296, audio=68, text=256, weights="mxfp8",
             passes=3),
        # the distilled step at 768x512x65 as it is served: captured once, replayed per step
        dict(name="step_768x512x65_mxfp8", kind="step", height=512, width=768, frames=65, text=256,
             weights="mxfp8", layers=4, sigma_index=6),
    ]


def draw(rng) -> dict:
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("modulate", "self_attention", "self_attention", "text_attention", "a2v", "v2a",
                       "feed_forward", "feed_forward", "connector", "block", "block", "step"))
    weights = rng.choice(("mxfp8", "mxfp8", "bf16", "int8"))
    video, audio, text = log_int(200, 6144), log_int(24, 160), rng.choice((rng.randint(16, 512), 256))
    if kind == "modulate":
        return dict(kind=kind, tokens=log_int(24, 14640), channels=rng.choice((4096, 2048)))
    if kind in ("self_attention", "feed_forward", "text_attention"):
        stream = rng.choice(("video", "video", "audio"))
        case = dict(kind=kind, stream=stream, tokens=video if stream == "video" else audio, weights=weights)
        return dict(case, text=text) if kind == "text_attention" else case
    if kind in ("a2v", "v2a"):
        return dict(kind=kind, tokens=video, audio=audio, weights=weights)
    if kind == "connector":
        return dict(kind=kind, text=rng.randint(8, 1400), weights="bf16")
    if kind == "block":
        passes = rng.choice((1, 1, 2, 3))
        return dict(kind=kind, tokens=log_int(96, 3456 // passes), audio=audio, text=text, weights=weights,
                    passes=passes)
    height, width = 32 * rng.randint(6, 16), 32 * rng.randint(8, 24)
    return dict(kind=kind, height=height, width=width, frames=8 * rng.randint(1, 8) + 1, text=text,
                weights=weights, layers=rng.choice((1, 2)), sigma_index=rng.randint(4, 7))


# ---- inputs -------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rows(gen, *shape, std=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * std).bfloat16()


def _biases(gen, weights):
    for w in weights:  # the random initialisation's biases are zero, a checkpoint's are not
        w.bias.normal_(0.0, 0.02, generator=gen)


def _attention(case, gen, query, context, heads, dim_head):
    from ltx_amd.loader.weights import build_attention

    attn = build_attention(query, context, heads, dim_head, gen=gen, device="cuda", weight_format=case["weights"])
    _biases(gen, attn.weights())
    for norm in (attn.q_norm, attn.k_norm):
        norm.uniform_(0.6, 1.4, generator=gen)
    return attn


def _grid(tokens):
    """A (frames, height, width) latent grid of at least ``tokens`` tokens in the usual 3:2 shape."""
    height = max(1, round((tokens / 13.5) ** 0.5)) if tokens >= 96 else 4
    width = max(1, round(1.5 * height))
    return -(-tokens // (height * width)), height, width


def _positions(tokens=0, audio=0):
    from ltx_amd.model.transformer.rope import audio_positions, video_positions

    return (video_positions(*_grid(tokens), 24.0)[:, :, :tokens] if tokens else None,
            audio_positions(audio) if audio else None)


def _tables(positions, dim, max_pos):
    from ltx_amd.model.transformer.rope import rope_tables

    return rope_tables(positions, dim, max_pos, "cuda", factored=True)


def _video_pe(tokens):
    return _tables(_positions(tokens)[0], VIDEO["dim"], (20, 2048, 2048))


def _audio_pe(audio):
    return _tables(_positions(0, audio)[1], AUDIO["dim"], (20,))


def _cross_pe(tokens, audio):
    vp, ap = _positions(tokens, audio)
    return _tables(vp[:, :1], AUDIO["dim"], (20,)), _tables(ap[:, :1], AUDIO["dim"], (20,))


def _inputs(case, seed) -> dict:
    """The operands of a case, from its seed alone."""
    gen, kind = _gen(seed), case["kind"]
    if kind == "modulate":
        t, c = case["tokens"], case["channels"]
        rows = [torch.randn((1, 1, c), generator=gen, device="cuda") * 0.1 for _ in range(3)]
        return dict(x=_rows(gen, 1, t, c), branch=_rows(gen, 1, t, c), scale=rows[0], shift=rows[1], gate=rows[2])
    if kind in ("self_attention", "text_attention"):
        cfg = VIDEO if case["stream"] == "video" else AUDIO
        text = kind == "text_attention"
        attn = _attention(case, gen, cfg["dim"], cfg["dim"] if text else None, cfg["heads"], cfg["dim_head"])
        pe = None if text else (_video_pe if cfg is VIDEO else _audio_pe)(case["tokens"])
        return dict(attn=attn, x=_rows(gen, case["tokens"], cfg["dim"]),
                    context=_rows(gen, case["text"], cfg["dim"]) if text else None, pe=pe, k_pe=None)
    if kind in ("a2v", "v2a"):
        vpe, ape = _cross_pe(case["tokens"], case["audio"])
        video, audio = _rows(gen, case["tokens"], VIDEO["dim"]), _rows(gen, case["audio"], AUDIO["dim"])
        if kind == "a2v":
            attn = _attention(case, gen, VIDEO["dim"], AUDIO["dim"], AUDIO["heads"], AUDIO["dim_head"])
            return dict(attn=attn, x=video, context=audio, pe=vpe, k_pe=ape)
        attn = _attention(case, gen, AUDIO["dim"], VIDEO["dim"], AUDIO["heads"], AUDIO["dim_head"])
        return dict(attn=attn, x=audio, context=video, pe=ape, k_pe=vpe)
    if kind == "feed_forward":
        from ltx_amd.loader.weights import build_ff

        dim = (VIDEO if case["stream"] == "video" else AUDIO)["dim"]
        ff = build_ff(dim, gen=gen, device="cuda", weight_format=case["weights"])
        _biases(gen, ff.weights())
        return dict(ff=ff, x=_rows(gen, case["tokens"], dim))
    if kind == "connector":
        from ltx_amd.model.text_encoder.connector import Embeddings1DConnector

        conn = Embeddings1DConnector(num_layers=1, weight_format=case["weights"],
                                     positional_embedding_max_pos=[4096], seed=seed)
        for b in conn.transformer_1d_blocks:
            _biases(gen, b.attn1.weights() + b.ff.weights())
        conn.rope(conn.extended_length(case["text"]))  # built once per length
        return dict(connector=conn, x=_rows(gen, 1, case["text"], VIDEO["dim"]))
    if kind == "block":
        from ltx_amd.model.transformer.transformer import BasicAVTransformerBlock, TransformerArgs, TransformerConfig

        cfgs = [TransformerConfig(c["dim"], c["heads"], c["dim_head"], c["dim"], True, True) for c in (VIDEO, AUDIO)]
        block = BasicAVTransformerBlock(0, *cfgs, weight_format=case["weights"], generator=gen)
        _biases(gen, block.linear_weights())
        for a in block.attentions():
            for norm in (a.q_norm, a.k_norm):
                norm.uniform_(0.6, 1.4, generator=gen)
        p, args = case["passes"], []
        cross = _cross_pe(case["tokens"], case["audio"])
        for cfg, t, pe, xpe in ((VIDEO, case["tokens"], _video_pe(case["tokens"]), cross[0]),
                                (AUDIO, case["audio"], _audio_pe(case["audio"]), cross[1])):
            d = cfg["dim"]
            temb = torch.randn((16, d), generator=gen, device="cuda") * 0.3
            args.append(TransformerArgs(
                x=_rows(gen, p, t, d) if p > 1 else _rows(gen, t, d),
                context=_rows(gen, p, case["text"], d) if p > 1 else _rows(gen, case["text"], d),
                timesteps=temb[None, None, :9], prompt_timestep=temb[None, None, 9:11],
                cross_scale_shift_timestep=temb[None, None, 11:15], cross_gate_timestep=temb[None, None, 15:],
                positional_embeddings=pe, cross_positional_embeddings=xpe))
        return dict(block=block, video=args[0], audio=args[1])
    from ltx_amd.model.transformer.model import LTXModel
    from ltx_amd.pipeline import DenoiseState

    model = LTXModel(num_layers=case["layers"], weight_format=case["weights"], seed=seed)
    state = DenoiseState(model, case["height"], case["width"], case["frames"], text_tokens=case["text"], seed=seed)
    for b in model.transformer_blocks:
        _biases(gen, b.linear_weights())
    # modulation of a trained model's size (the random tables leave every gate near zero)
    for t in (model.video_tables, model.audio_tables):
        t.normal_(0.0, 0.3, generator=gen)
    return dict(model=model, state=state, pes=model.rope(state.video_positions, state.audio_positions))


def _perturbations(passes):
    """A guided step's passes: plain, negative prompt, and (third) video self-attention skipped."""
    from ltx_amd.components.perturbations import (BatchedPerturbationConfig, PerturbationConfig,
                                                  create_stg_perturbation)

    if passes < 3:
        return None
    return BatchedPerturbationConfig([PerturbationConfig.empty()] * (passes - 1) + [create_stg_perturbation()])


def _step(s, sigma_index):
    from ltx_amd.components.diffusion_steps import EulerDiffusionStep

    model, st = s["model"], s["state"]
    now, then = st.sigmas[sigma_index], st.sigmas[sigma_index + 1]
    v, a = model.velocity(st.video_latent, st.video_context, st.sigmas_dev[sigma_index:sigma_index + 1], s["pes"],
                          st.audio_latent, st.audio_context)
    euler = EulerDiffusionStep()
    return [v, a, euler.step_from_velocity(st.video_latent, v, now, then),
            euler.step_from_velocity(st.audio_latent, a, now, then)]


def prepare(case: dict, seed: int) -> dict:
    s = dict(_inputs(case, seed), kind=case["kind"])
    if case["kind"] == "block":
        s["perturbations"] = _perturbations(case["passes"])
    if case["kind"] == "step":
        _step(s, case["sigma_index"])  # once outside capture, as the denoise loops do
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = _step(s, case["sigma_index"])
    return s


def run(s: dict):
    kind = s["kind"]
    if kind == "modulate":
        from ltx_amd.kernels import adaln_norm_fused, gated_add_fused

        y = adaln_norm_fused(s["x"], s["scale"], s["shift"], EPS)
        return [y, gated_add_fused(s["x"], s["branch"], s["gate"])]
    if kind in ("self_attention", "text_attention", "a2v", "v2a"):
        return s["attn"](s["x"], s["context"], pe=s["pe"], k_pe=s["k_pe"])
    if kind == "feed_forward":
        return s["ff"](s["x"])
    if kind == "connector":
        return s["connector"](s["x"])[0]
    if kind == "block":
        video, audio = s["block"](s["video"], s["audio"], perturbations=s["perturbations"])
        return [video.x, audio.x]
    s["graph"].replay()
    return s["out"]


# ---- the least work -----------------------------------------------------------------------------------


def _linear_work(fmt, m, n, k):
    bits = dict(bf16=16.0, int8=8.0, mxfp8=8.25)[fmt]
    return n * k * bits / 8 + 4 * n * (2 if fmt == "int8" else 1), 2.0 * m * n * k


def _attention_work(fmt, tq, tk, query, context, heads, dim_head, passes=1, own=True):
    """Weights' bytes and flops; ``own``: the keys come from the queries' rows."""
    inner = heads * dim_head
    parts = ([_linear_work(fmt, passes * tq, 3 * inner + heads, query)] if own else
             [_linear_work(fmt, passes * tq, inner + heads, query),
              _linear_work(fmt, passes * tk, 2 * inner, context)])
    parts.append(_linear_work(fmt, passes * tq, query, inner))
    return sum(b for b, _ in parts), sum(f for _, f in parts) + 4.0 * passes * tq * tk * inner


def _block_work(fmt, tv, ta, text, passes=1, skipped=0):
    v, a = VIDEO, AUDIO
    parts = [_attention_work(fmt, tv, tv, v["dim"], 0, v["heads"], v["dim_head"], passes - skipped),
             _attention_work(fmt, tv, text, v["dim"], v["dim"], v["heads"], v["dim_head"], passes, False),
             _attention_work(fmt, ta, ta, a["dim"], 0, a["heads"], a["dim_head"], passes),
             _attention_work(fmt, ta, text, a["dim"], a["dim"], a["heads"], a["dim_head"], passes, False),
             _attention_work(fmt, tv, ta, v["dim"], a["dim"], a["heads"], a["dim_head"], passes, False),
             _attention_work(fmt, ta, tv, a["dim"], v["dim"], a["heads"], a["dim_head"], passes, False)]
    for t, d in ((tv, v["dim"]), (ta, a["dim"])):
        parts += [_linear_work(fmt, passes * t, 4 * d, d), _linear_work(fmt, passes * t, d, 4 * d)]
    return sum(b for b, _ in parts), sum(f for _, f in parts)


def _step_tokens(case):
    frames = (case["frames"] - 1) // 8 + 1
    return frames * (case["height"] // 32) * (case["width"] // 32), math.ceil(case["frames"] / 24.0 * 25.0)


def work(case: dict) -> dict:
    kind, fmt = case["kind"], case.get("weights")
    if kind == "modulate":
        n = case["tokens"] * case["channels"]
        return dict(bytes=2.0 * n * 4 + 12 * case["channels"], flops=0.0)  # x, branch in; both results out
    if kind in ("self_attention", "text_attention"):
        c, t = (VIDEO if case["stream"] == "video" else AUDIO), case["tokens"]
        own = kind == "self_attention"
        b, f = _attention_work(fmt, t, t if own else case["text"], c["dim"], c["dim"], c["heads"], c["dim_head"],
                               1, own)
        return dict(bytes=b + 2.0 * c["dim"] * (2 * t + (0 if own else case["text"])), flops=f)
    if kind in ("a2v", "v2a"):
        tv, ta = case["tokens"], case["audio"]
        tq, tk, q, c = (tv, ta, 4096, 2048) if kind == "a2v" else (ta, tv, 2048, 4096)
        b, f = _attention_work(fmt, tq, tk, q, c, AUDIO["heads"], AUDIO["dim_head"], 1, False)
        return dict(bytes=b + 2.0 * (2 * tq * q + tk * c), flops=f)
    if kind == "feed_forward":
        d, t = (VIDEO if case["stream"] == "video" else AUDIO)["dim"], case["tokens"]
        parts = (_linear_work(fmt, t, 4 * d, d), _linear_work(fmt, t, d, 4 * d))
        return dict(bytes=sum(b for b, _ in parts) + 4.0 * t * d, flops=sum(f for _, f in parts))
    if kind == "connector":
        t, c = math.ceil(max(1024, case["text"]) / 128) * 128, VIDEO
        b, f = _attention_work(fmt, t, t, c["dim"], 0, c["heads"], c["dim_head"])
        for n, k in ((16384, 4096), (4096, 16384)):
            b, f = b + _linear_work(fmt, t, n, k)[0], f + _linear_work(fmt, t, n, k)[1]
        return dict(bytes=b + 2.0 * c["dim"] * (case["text"] + 128 + t), flops=f)
    if kind == "block":
        p, tv, ta = case["passes"], case["tokens"], case["audio"]
        b, f = _block_work(fmt, tv, ta, case["text"], p, 1 if p >= 3 else 0)
        return dict(bytes=b + 2.0 * p * (4096 * (2 * tv + case["text"]) + 2048 * (2 * ta + case["text"])), flops=f)
    tv, ta = _step_tokens(case)
    b, f = _block_work(fmt, tv, ta, case["text"])
    mlps = sum(2.0 * (256 * d + 4 * d * d + 16 * d * d) for d in (4096, 2048))  # bf16 timestep MLPs
    mlps += 2.0 * 3 * 256 * (4096 + 2048)
    ends = sum(2.0 * 128 * d * 2 for d in (4096, 2048))  # patchify and output projections
    io = 2.0 * 128 * 3 * (tv + ta) + 2.0 * case["text"] * (4096 + 2048)
    return dict(bytes=case["layers"] * b + mlps + ends + io,
                flops=case["layers"] * f + 2.0 * 2 * 128 * (tv * 4096 + ta * 2048))


def tolerance(case: dict):
    # bf16 results of chained products; about four times the error against float64
    return dict(rel={"modulate": 0.007, "feed_forward": 0.012, "connector": 0.016, "block": 0.016,
                     "step": 0.02}.get(case["kind"], 0.016))


# ---- the results in float64 ---------------------------------------------------------------------------


def _decoded(w):
    """The bf16 values that a resident weight stands for, as float64."""
    if w.kind == "bf16":
        return w.w.double()
    if w.kind == "int8":
        return (w.w.float() * w.scale[:, None]).bfloat16().double()
    codes = w.w.view(torch.float8_e4m3fn).float().double()
    return codes * torch.exp2(w.scale.double() - 127.0).repeat_interleave(32, 1)


def _lin(x, w):
    return x @ _decoded(w).T + w.bias.double()


def _rms(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rope(x, pe, heads):
    if pe is None:
        return x
    cos, sin = pe[0].double(), pe[1].double()
    if len(pe) == 3:  # per-axis rows and each token's row of every axis
        idx = pe[2].long()
        cos = math.prod(cos[idx[:, a]] for a in range(idx.shape[1]))
        sin = sum(sin[idx[:, a]] for a in range(idx.shape[1]))
    t, d = x.shape
    half = d // heads // 2
    cos, sin = (y[:t].reshape(t, heads, half) for y in (cos, sin))
    a, b = x.view(t, heads, 2, half).unbind(2)
    return torch.stack((a * cos - b * sin, a * sin + b * cos), 2).reshape(t, d)


def _attend(attn, x, context=None, pe=None, k_pe=None):
    """The module's result with its output projection."""
    inner, heads = attn.inner_dim, attn.heads
    if attn.self_attention:
        q, k, v, g = _lin(x, attn.proj_q).split((inner, inner, inner, heads), 1)
        k_pe = pe
    else:
        q, g = _lin(x, attn.proj_q).split((inner, heads), 1)
        k, v = _lin(context, attn.proj_kv).split((inner, inner), 1)
    q = _rope(_rms(q) * attn.q_norm.double(), pe, heads)
    k = _rope(_rms(k) * attn.k_norm.double(), k_pe, heads)
    out = torch.empty_like(q)
    dh = inner // heads
    for h in range(heads):
        c = slice(h * dh, (h + 1) * dh)
        p = torch.softmax(q[:, c] @ k[:, c].T.contiguous() / math.sqrt(dh), -1)
        out[:, c] = (p @ v[:, c].contiguous()) * (2 * torch.sigmoid(g[:, h:h + 1]))
    return _lin(out, attn.to_out)


def _ff(ff, x):
    return _lin(torch.nn.functional.gelu(_lin(x, ff.project_in), approximate="tanh"), ff.project_out)


def _block(block, vx, ax, vctx, actx, rv, ra, vpe, ape, vxpe, axpe, skip=False):
    """One pass of a block; rv, ra: its (16, D) modulation rows."""
    def mod(x, r, scale, shift):
        return _rms(x) * (1 + r[scale]) + r[shift]

    def stream(x, ctx, r, self_attn, text_attn, pe, skip):
        if not skip:
            x = x + r[2] * _attend(self_attn, mod(x, r, 1, 0), pe=pe)
        c = ctx * (1 + r[10]) + r[9]
        return x + r[8] * _attend(text_attn, mod(x, r, 7, 6), c)

    vx = stream(vx, vctx, rv, block.attn1, block.attn2, vpe, skip)
    ax = stream(ax, actx, ra, block.audio_attn1, block.audio_attn2, ape, False)
    v_in, a_in = (mod(vx, rv, 11, 12), mod(vx, rv, 13, 14)), (mod(ax, ra, 11, 12), mod(ax, ra, 13, 14))
    vx = vx + rv[15] * _attend(block.audio_to_video_attn, v_in[0], a_in[0], vxpe, axpe)
    ax = ax + ra[15] * _attend(block.video_to_audio_attn, a_in[1], v_in[1], axpe, vxpe)
    return (vx + rv[5] * _ff(block.ff, mod(vx, rv, 4, 3)),
            ax + ra[5] * _ff(block.audio_ff, mod(ax, ra, 4, 3)))


def _mlp(m, t):
    """(embedding rows, embedded timestep) of one timestep MLP."""
    e = torch.exp(-math.log(10000.0) * torch.arange(128, dtype=torch.float64, device="cuda") / 128)
    x = torch.cat((torch.cos(t * e), torch.sin(t * e)))
    silu = torch.nn.functional.silu
    emb = m.w2.double() @ silu(m.w1.double() @ x + m.b1.double()) + m.b2.double()
    return (m.w.double() @ silu(emb) + m.b.double()).view(-1, m.dim), emb


def _exact_step(s, case):
    model, st = s["model"], s["state"]
    now, then = st.sigmas[case["sigma_index"]], st.sigmas[case["sigma_index"] + 1]
    vpe, vxpe, ape, axpe = s["pes"]
    xs, embs, rows = [], [], []
    for lat, proj, mlps, tables in (
            (st.video_latent, model.patchify_proj, (model.adaln_single, model.prompt_adaln_single,
             model.av_ca_video_scale_shift_adaln_single, model.av_ca_a2v_gate_adaln_single), model.video_tables),
            (st.audio_latent, model.audio_patchify_proj, (model.audio_adaln_single, model.audio_prompt_adaln_single,
             model.av_ca_audio_scale_shift_adaln_single, model.av_ca_v2a_gate_adaln_single), model.audio_tables)):
        out = [_mlp(m, now * 1000.0) for m in mlps]
        xs.append(_lin(lat.double(), proj))
        embs.append(out[0][1])
        rows.append(torch.cat([r for r, _ in out]) + tables.double())
    ctx = st.video_context.double(), st.audio_context.double()
    for i, b in enumerate(model.transformer_blocks):
        xs = _block(b, *xs, *ctx, rows[0][i], rows[1][i], vpe, ape, vxpe, axpe)
    vel = []
    for x, table, emb, proj in ((xs[0], model.scale_shift_table, embs[0], model.proj_out),
                                (xs[1], model.audio_scale_shift_table, embs[1], model.audio_proj_out)):
        n = torch.nn.functional.layer_norm(x, x.shape[-1:], eps=EPS)
        vel.append(_lin(n * (1 + table[1].double() + emb) + table[0].double() + emb, proj))
    return vel + [lat.double() + (then - now) * v for lat, v in zip((st.video_latent, st.audio_latent), vel)]


def exact(case: dict, seed: int):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "modulate":
        x = s["x"].double()
        return [_rms(x) * (1 + s["scale"].double()) + s["shift"].double(),
                x + s["branch"].double() * s["gate"].double()]
    if kind in ("self_attention", "text_attention", "a2v", "v2a"):
        context = None if s["context"] is None else s["context"].double()
        return _attend(s["attn"], s["x"].double(), context, s["pe"], s["k_pe"])
    if kind == "feed_forward":
        return _ff(s["ff"], s["x"].double())
    if kind == "connector":
        conn = s["connector"]
        x, total = s["x"][0], conn.extended_length(case["text"])
        tiled = conn.learnable_registers.repeat(total // conn.num_learnable_registers, 1)
        x = torch.cat((x, tiled[x.shape[0]:])).double()
        for b in conn.transformer_1d_blocks:
            x = x + _attend(b.attn1, _rms(x), pe=conn.rope(total))
            x = x + _ff(b.ff, _rms(x))
        return _rms(x)[None]
    if kind == "block":
        block, out = s["block"], []
        rows = []
        for a, tables in ((s["video"], block.video_tables), (s["audio"], block.audio_tables)):
            temb = torch.cat([t[0, 0] for t in (a.timesteps, a.prompt_timestep, a.cross_scale_shift_timestep,
                                                a.cross_gate_timestep)])
            rows.append(temb.double() + tables.double())
        v, a, p = s["video"], s["audio"], case["passes"]
        for i in range(p):
            ops = [t if p == 1 else t[i] for t in (v.x, a.x, v.context, a.context)]
            out.append(_block(block, *(t.double() for t in ops), *rows, v.positional_embeddings,
                              a.positional_embeddings, v.cross_positional_embeddings,
                              a.cross_positional_embeddings, skip=p >= 3 and i == p - 1))
        return [torch.stack(x) if p > 1 else x[0] for x in zip(*out)]
    return _exact_step(s, case)
