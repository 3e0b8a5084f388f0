"""The work whose speed counts: what an engine has this framework do, call by call.

Every case is one call sequence of a serving step at the sizes engines run: decode
attention from a handful of short sequences to a full batch of long ones, a prefill chunk
alone and a whole prompt, a packed step of chunks and decodes, decodes that share a cached
prefix, and the W4A16 feed-forward block from one token to a packed step's worth.
``listed()`` names fixed ones, ``draw()`` gives others of the same ranges.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from slipstream_amd import workloads
from slipstream_amd.kernels import (
    fused_rmsnorm,
    packed_attention,
    paged_attention_decode,
    paged_attention_prefill,
    paged_attention_shared_prefix,
)
from slipstream_amd.paged_cache import build_packed_step
from slipstream_amd.quantized import W4A16Linear, W4A16MLP, quantize_weight

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
ROPE_THETA = 500000.0


def listed() -> list[dict]:
    return [
        # a few chats on a small model: 14/2 heads of 64 in fp16, short contexts; one launch's latency
        {"name": "decode_small", "kind": "decode", "batch": 8, "n_q": 14, "n_kv": 2, "head_dim": 64, "block": 16,
         "dtype": "fp16", "ctx_lo": 32, "ctx_hi": 512},
        # a half-filled batch at an odd size, 28/4 heads, larger blocks
        {"name": "decode_medium", "kind": "decode", "batch": 37, "n_q": 28, "n_kv": 4, "head_dim": 128, "block": 32,
         "dtype": "bf16", "ctx_lo": 64, "ctx_hi": 4096},
        # the full decode batch of a 32/8-head model, contexts spread over 16 to 8192 tokens
        {"name": "decode_large", "kind": "decode", "batch": 256, "n_q": 32, "n_kv": 8, "head_dim": 128, "block": 16,
         "dtype": "bf16", "ctx_lo": 16, "ctx_hi": 8192},
        # one prefill chunk by itself, as an engine runs a chunked prompt: 256 new tokens over what is there
        {"name": "prefill_chunk", "kind": "prefill", "batch": 1, "n_q": 32, "n_kv": 8, "head_dim": 128, "block": 16,
         "dtype": "bf16", "tq": 256, "prior": 1777},
        # a long prompt in one call, odd length, nothing cached
        {"name": "prefill_prompt", "kind": "prefill", "batch": 1, "n_q": 32, "n_kv": 8, "head_dim": 128, "block": 16,
         "dtype": "bf16", "tq": 6001, "prior": 0},
        # a mixed step of a continuous batch: chunks and decodes in one token stream, RoPE and KV write included
        {"name": "packed_step", "kind": "packed", "n_prefill": 4, "chunk": 512, "n_decode": 192, "n_q": 32, "n_kv": 8,
         "head_dim": 128, "block": 16, "dtype": "bf16", "ctx_lo": 128, "ctx_hi": 4096},
        # decodes behind one system prompt: every table starts with the same cached blocks
        {"name": "shared_prefix", "kind": "prefix", "batch": 128, "n_q": 28, "n_kv": 4, "head_dim": 128, "block": 16,
         "dtype": "bf16", "prefix": 2048, "ctx_lo": 64, "ctx_hi": 512},
        # the quantized feed-forward block for one token; three layers' weights in turn, captured as decode loops are
        {"name": "mlp_token", "kind": "mlp", "m": 1, "hidden": 4096, "inter": 14336, "group": 128, "dtype": "bf16",
         "layers": 3, "graph": True},
        # the same for a small batch, and with the finer groups some checkpoints have on a small model
        {"name": "mlp_small_groups", "kind": "mlp", "m": 11, "hidden": 896, "inter": 4864, "group": 64,
         "dtype": "fp16", "layers": 3, "graph": True},
        {"name": "mlp_batch", "kind": "mlp", "m": 24, "hidden": 4096, "inter": 14336, "group": 128, "dtype": "bf16",
         "layers": 3, "graph": True},
        # a decode batch of an odd size, called as it is
        {"name": "mlp_decodes", "kind": "mlp", "m": 197, "hidden": 4096, "inter": 14336, "group": 128,
         "dtype": "bf16", "layers": 1, "graph": False},
        # every token of a packed step (4 chunks of 512 and 192 decodes)
        {"name": "mlp_step", "kind": "mlp", "m": 2240, "hidden": 4096, "inter": 14336, "group": 128, "dtype": "bf16",
         "layers": 1, "graph": False},
    ]


HEADS = [(14, 2, 64), (28, 4, 128), (32, 8, 128)]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "packed", "prefix", "mlp", "mlp", "mlp"])
    if kind == "mlp":
        small = rng.random() < 0.3
        hidden, inter = (896, 4864) if small else (128 * _log_int(rng, 8, 32), 128 * _log_int(rng, 16, 112))
        m = _log_int(rng, 1, 2240)
        layers = 3 if m <= 64 else 1
        return {"kind": kind, "m": m, "hidden": hidden, "inter": inter,
                "group": rng.choice([32, 64]) if m <= 64 and rng.random() < 0.25 else 128,
                "dtype": rng.choice(["bf16", "bf16", "fp16"]), "layers": layers, "graph": m <= 64}
    n_q, n_kv, d = rng.choice(HEADS)
    case = {"kind": kind, "n_q": n_q, "n_kv": n_kv, "head_dim": d,
            "dtype": rng.choice(["bf16", "bf16", "fp16"]), "block": rng.choice([16, 16, 32])}
    if kind == "decode":
        batch = _log_int(rng, 1, 256)
        hi = _log_int(rng, 64, 8192)
        case.update(batch=batch, ctx_lo=rng.randint(1, 64), ctx_hi=hi)
    elif kind == "prefill":
        tq = _log_int(rng, 16, 4096)
        case.update(batch=rng.randint(1, 4) if tq <= 1024 else 1, tq=tq, prior=rng.choice([0, rng.randint(1, 4096)]))
    elif kind == "packed":
        case.update(n_prefill=rng.randint(1, 4), chunk=_log_int(rng, 32, 512), n_decode=_log_int(rng, 4, 192),
                    ctx_lo=rng.randint(16, 128), ctx_hi=_log_int(rng, 256, 4096))
    else:
        case.update(batch=_log_int(rng, 8, 128), prefix=32 * _log_int(rng, 8, 64), ctx_lo=rng.randint(1, 64),
                    ctx_hi=_log_int(rng, 64, 512))
    return case


# ---- inputs --------------------------------------------------------------------------


def _lengths(case: dict, count: int) -> list[int]:
    """Context lengths of a case: fixed by the case, so that its work is the same for every
    seed -- lognormal about the geometric middle of the range, as chat lengths spread."""
    rng = np.random.default_rng([count, case["ctx_lo"], case["ctx_hi"]])
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    if hi / lo > 64:
        x = np.rint(rng.lognormal(mean=math.log(hi / 8.0), sigma=1.0, size=count))
        return np.clip(x, lo, hi).astype(int).tolist()
    return rng.integers(lo, hi + 1, size=count).tolist()


def _step_lengths(case: dict) -> tuple[list[int], list[int]]:
    """(context lengths, query lengths) of every sequence of an attention case."""
    if case["kind"] == "decode":
        ctx = _lengths(case, case["batch"])
        return ctx, [1] * len(ctx)
    if case["kind"] == "prefix":
        ctx = [case["prefix"] + s for s in _lengths(case, case["batch"])]
        return ctx, [1] * len(ctx)
    if case["kind"] == "prefill":
        return [case["prior"] + case["tq"]] * case["batch"], [case["tq"]] * case["batch"]
    dec = _lengths(case, case["n_decode"])  # decodes first, then the chunks, as a scheduler packs them
    rng = np.random.default_rng([case["n_prefill"], case["chunk"]])
    chunks = [int(p) + case["chunk"] for p in rng.integers(0, 4097, size=case["n_prefill"])]
    return dec + chunks, [1] * len(dec) + [case["chunk"]] * len(chunks)


def _prepare_attention(case: dict, seed: int) -> dict:
    ctx, ql = _step_lengths(case)
    batch = workloads.build_batch(
        ctx, ql, n_q=case["n_q"], n_kv=case["n_kv"], head_dim=case["head_dim"], block_size=case["block"],
        dtype=DTYPES[case["dtype"]], device="cuda", seed=seed, std=1.0,
        shared_prefix_blocks=case["prefix"] // case["block"] if case["kind"] == "prefix" else 0)
    state = {"kind": case["kind"], "batch": batch}
    if case["kind"] == "packed":
        pos = torch.cat([torch.arange(c - q, c) for c, q in zip(ctx, ql)]).to(torch.float32)
        half = torch.arange(0, case["head_dim"], 2, dtype=torch.float32) / case["head_dim"]
        angle = torch.outer(pos, ROPE_THETA ** -half)
        angle = torch.cat([angle, angle], dim=-1).to("cuda")
        state["cos"], state["sin"] = angle.cos().to(batch.q.dtype), angle.sin().to(batch.q.dtype)
        state["query_lens"] = torch.tensor(ql, dtype=torch.int32, device="cuda")
        state["prior_lens"] = batch.context_lens - state["query_lens"]
    else:
        state["q"] = batch.padded_q().contiguous()
    return state


def _prepare_mlp(case: dict, seed: int) -> dict:
    """Weights N(0, 1/fan-in) put through the framework's own quantizer, as a checkpoint's
    were; activations N(0, 1) with a few large channels, as hidden states have."""
    dt = DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def linear(n: int, k: int) -> W4A16Linear:
        w = torch.randn(n, k, generator=gen, device="cuda", dtype=torch.float32) * k ** -0.5
        qweight, scales, qzeros = quantize_weight(w, case["group"])
        return W4A16Linear(qweight, scales.to(torch.float16), qzeros, case["group"])

    layers = []
    hidden, inter = case["hidden"], case["inter"]
    for _ in range(case["layers"]):
        mlp = W4A16MLP(linear(inter, hidden), linear(inter, hidden), linear(hidden, inter))
        big = torch.ones(hidden, device="cuda")
        big[torch.randint(0, hidden, (4,), generator=gen, device="cuda")] = 8.0
        x = (torch.randn(case["m"], hidden, generator=gen, device="cuda") * big).to(dt)
        attn = torch.randn(case["m"], hidden, generator=gen, device="cuda").to(dt)
        norm = (1.0 + 0.1 * torch.randn(hidden, generator=gen, device="cuda")).to(dt)
        layers.append({"mlp": mlp, "x": x, "attn": attn, "norm": norm})
    state = {"kind": "mlp", "layers": layers, "graph": None}
    if case["graph"]:
        state["stream"] = stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _run_layers(state)  # workspaces exist before the capture
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=stream):
            state["out"] = _run_layers(state)
    return state


def prepare(case: dict, seed: int) -> dict:
    return _prepare_mlp(case, seed) if case["kind"] == "mlp" else _prepare_attention(case, seed)


# ---- one pass ------------------------------------------------------------------------


def _run_layers(state: dict) -> list[torch.Tensor]:
    """The feed-forward half of a decoder layer: norm of (x + attention output), then the
    gated MLP on int4 weights."""
    with torch.no_grad():
        return [s["mlp"](fused_rmsnorm(s["x"], s["norm"], s["attn"])) for s in state["layers"]]


def run(state: dict):
    if state["kind"] == "mlp":
        if state["graph"] is None:
            return _run_layers(state)
        state["graph"].replay()
        return state["out"]
    b = state["batch"]
    if state["kind"] == "packed":
        step = build_packed_step(b.block_tables, state["prior_lens"], state["query_lens"], b.block_size,
                                 b.total_tokens, b.max_query_len)
        out = packed_attention(b.q, b.k_new, b.v_new, state["cos"], state["sin"], b.kv_cache, step, 0, b.scale,
                               b.block_size)
        return [out, b.kv_cache]
    if state["kind"] == "prefix":
        return paged_attention_shared_prefix(state["q"], b.kv_cache, b.block_tables, b.context_lens, 0, b.scale,
                                             b.block_size, b.shared_blocks)
    attend = paged_attention_decode if state["kind"] == "decode" else paged_attention_prefill
    return attend(state["q"], b.kv_cache, b.block_tables, b.context_lens, 0, b.scale, b.block_size)


# ---- what a pass cannot do without ---------------------------------------------------


def work(case: dict) -> dict:
    if case["kind"] == "mlp":
        h, i, m, g = case["hidden"], case["inter"], case["m"], case["group"]
        weights = 3 * h * i
        per_layer = weights // 2 + weights // g * 6 + 2 * (3 * m * h + h)  # x, attn, out; the norm's weight
        return {"bytes": case["layers"] * per_layer, "flops": case["layers"] * 2 * m * weights}
    ctx, ql = _step_lengths(case)
    n_q, n_kv, d = case["n_q"], case["n_kv"], case["head_dim"]
    tokens = sum(ql)
    kv_tokens = sum(ctx)
    if case["kind"] == "prefix":
        kv_tokens -= case["prefix"] * (case["batch"] - 1)
    blocks = sum(-(-c // case["block"]) for c in ctx)
    nbytes = 2 * (kv_tokens * 2 * n_kv * d + 2 * tokens * n_q * d) + 4 * blocks + 4 * len(ctx)
    if case["kind"] == "packed":  # new K and V read, cos and sin read (the written rows are in kv_tokens)
        nbytes += 2 * (tokens * 2 * n_kv * d + 2 * tokens * d)
    flops = sum(4 * n_q * d * (q * (c - q) + q * (q + 1) // 2) for c, q in zip(ctx, ql))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict) -> dict:
    # measured against exact(): the rounding of the 16-bit results and of the
    # probabilities or the block's intermediate values, times about four
    if case["kind"] == "mlp":
        return {"rel": 1.6e-2 if case["dtype"] == "bf16" else 2e-3, "max": 0.1 if case["dtype"] == "bf16" else 1.5e-2}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.5e-3, "max": 0.1 if case["dtype"] == "bf16" else 1.5e-2}


# ---- the same in 64 bits, with torch alone -------------------------------------------


def _rotate(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos.unsqueeze(1) + turned * sin.unsqueeze(1)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float) -> torch.Tensor:
    """Causal attention of the last ``q.shape[0]`` tokens: q [Tq, n_q, D], k and v [ctx, n_kv, D]."""
    tq, n_q, d = q.shape
    ctx, n_kv, _ = k.shape
    rep = n_q // n_kv
    out = torch.empty_like(q)
    last = torch.arange(ctx - tq, ctx, device=q.device)
    hidden = torch.arange(ctx, device=q.device)[None, :] > last[:, None]
    for h in range(n_kv):
        kt = k[:, h].t().contiguous()
        vh = v[:, h].contiguous()
        for r in range(rep):
            scores = (q[:, h * rep + r].contiguous() @ kt) * scale
            out[:, h * rep + r] = scores.masked_fill_(hidden, -math.inf).softmax(dim=-1) @ vh
    return out


def _attend_one(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float) -> torch.Tensor:
    """The same for one query token: q [1, n_q, D]."""
    n_kv, d = k.shape[1], k.shape[2]
    qh = q[0].view(n_kv, -1, d)
    scores = torch.matmul(qh, k.permute(1, 2, 0).contiguous()) * scale
    return torch.matmul(scores.softmax(dim=-1), v.transpose(0, 1).contiguous()).reshape(1, -1, d)


def _exact_attention(case: dict, seed: int):
    state = _prepare_attention(case, seed)
    b = state["batch"]
    q, k_new = b.q.double(), b.k_new.double()
    if case["kind"] == "packed":
        cos, sin = state["cos"].double(), state["sin"].double()
        q, k_new = _rotate(q, cos, sin), _rotate(k_new, cos, sin)
    out, at = torch.empty_like(q), 0
    for ctx, ql, table in zip(b.ctx_host, b.query_lens, b.tables_host):
        pages = torch.tensor(table, device="cuda")
        k, v = (b.kv_cache[0, i, pages].reshape(-1, b.n_kv, b.head_dim)[:ctx].double() for i in (0, 1))
        if case["kind"] == "packed":
            k[ctx - ql:], v[ctx - ql:] = k_new[at : at + ql], b.v_new[at : at + ql].double()
        out[at : at + ql] = (_attend_one if ql == 1 else _attend)(q[at : at + ql], k, v, b.scale)
        at += ql
    if case["kind"] == "packed":
        return [out, None]
    return out.view(b.batch, -1, b.n_q, b.head_dim)


def _dense(lin: W4A16Linear) -> torch.Tensor:
    shifts = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    q = ((lin.qweight.unsqueeze(-1) >> shifts) & 15).flatten(1).double()
    scales, zeros = (t.double().repeat_interleave(lin.group_size, dim=1) for t in (lin.scales, lin.qzeros))
    return (q - zeros) * scales


def _exact_mlp(case: dict, seed: int):
    out = []
    for s in _prepare_mlp(dict(case, graph=False), seed)["layers"]:
        h = s["x"].double() + s["attn"].double()
        h = h * (h.square().mean(dim=-1, keepdim=True) + 1e-6).rsqrt() * s["norm"].double()
        gate, up = (h @ _dense(s["mlp"].gate_up_proj).t()).split(case["inter"], dim=-1)
        out.append((gate * gate.sigmoid() * up) @ _dense(s["mlp"].down_proj).t())
    return out


def exact(case: dict, seed: int):
    return _exact_mlp(case, seed) if case["kind"] == "mlp" else _exact_attention(case, seed)
