"""The calls a program on this framework makes, at the sizes it makes them, for timing and comparing builds.

A case is one call of a public entry point with its sizes:

* ``step``       ``SharedFastWeightPool.chunk_step``: the write and readout of one chunk (streaming a turn);
* ``layer``      ``uTTTLayer.forward`` with writes: every chunk of a sequence through one layer;
* ``block``      ``uTTTBlock.forward`` with writes: attention and the layer;
* ``attention``  ``SlidingWindowAttention.forward``: prompt attention, with and without a KV cache;
* ``readout``    ``SharedFastWeightPool.forward_readout``: the frozen fast-weight read of a prompt;
* ``decode``     ``BatchedDecoder.step``: one token for each of many users, from one captured step;
* ``prefill``    ``uTTTModel.forward`` with writes: a batch of prompts, the last token's logits and the new state;
* ``evolve``     ``evolve_batched``: ragged turns of several users, their gates and elastic pull.

Widths come from the benchmark's model configurations and from ``uTTTConfig``'s defaults; weights are the
models' own initialisation, states are personalised (W near W_0, momentum not zero).
"""
from __future__ import annotations

import math
import random

import torch
import torch.nn.functional as F

from utttcompanion_amd import (FastWeightState, SharedFastWeightPool, SlidingWindowAttention, uTTTBlock, uTTTConfig,
                               uTTTLayer, uTTTModel)
from utttcompanion_amd.decoder import BatchedDecoder
from utttcompanion_amd.evolve import evolve_batched

EPS = 1e-5
BETA = 0.9
CLIP = 1.0
LR, DECAY = 0.015, 0.005
VOCAB = 32000
THETA = 10000.0

# d_model, d_ff, heads, kv heads, window
WIDTHS = {
    "w512": (512, 1024, 8, 4, 256),      # one fp32 block of the benchmark
    "w768": (768, 2048, 12, 4, 512),     # the 151M model
    "w1024": (1024, 2816, 16, 4, 512),   # uTTTConfig's defaults
    "w2048": (2048, 5504, 16, 4, 1024),  # the 1.58B model
}


def _width(case):
    return WIDTHS[case["width"]]


def listed():
    return [
        # one user's short chunk while a turn is streamed: the smallest write, launches and latency
        dict(name="step_1x37", kind="step", width="w768", rows=1, tokens=37, dtype="bf16"),
        # a whole block in fp32, sixteen chunk writes of one row: research and parity runs
        dict(name="block_fp32_1x1024", kind="block", width="w512", rows=1, tokens=1024, chunk=64, dtype="fp32",
             masked=False),
        # one layer over a padded batch, the module API of a program with its own model loop
        dict(name="layer_8x512", kind="layer", width="w768", rows=8, tokens=512, chunk=64, dtype="bf16", masked=True),
        # the longer write chunks of the shipped training configurations, with a ragged tail
        dict(name="layer_c128_2x600", kind="layer", width="w1024", rows=2, tokens=600, chunk=128, dtype="bf16",
             masked=False),
        # a follow-up turn on top of a full KV cache, odd length
        dict(name="attention_3x777_cached", kind="attention", width="w768", rows=3, tokens=777, history=512,
             dtype="bf16"),
        # long prompts
        dict(name="attention_4x4096", kind="attention", width="w2048", rows=4, tokens=4096, history=0, dtype="bf16"),
        # two users' short prompts read straight through the fp32 masters
        dict(name="readout_2x333", kind="readout", width="w768", rows=2, tokens=333, dtype="bf16", copies=False,
             shared=False),
        # long prompts of the large model prepared for inference (versioned bf16 read copies)
        dict(name="readout_4x2048", kind="readout", width="w2048", rows=4, tokens=2048, dtype="bf16", copies=True,
             shared=False),
        # batched serving: 32 users, ragged contexts, one token each
        dict(name="decode_32", kind="decode", width="w768", rows=32, layers=12, shortest=64, longest=2048),
        # a batch of prompts with writes through layers of the 151M model, not a whole number of chunks (four layers
        # here and below: a rounding travels through all that follow, so deeper stacks compare noise)
        dict(name="prefill_8x500", kind="prefill", width="w768", rows=8, tokens=500, layers=4),
        # the headline workload's layers: long prompts with writes
        dict(name="prefill_4x2048", kind="prefill", width="w2048", rows=4, tokens=2048, layers=4),
        # the users' turns after the replies, all at once, through the large model's layers
        dict(name="evolve_8_ragged", kind="evolve", width="w2048", rows=8, shortest=128, longest=2048, layers=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["step", "layer", "layer", "block", "attention", "attention", "readout", "readout", "decode",
                       "prefill", "evolve"])
    width = rng.choice(list(WIDTHS))
    big = width == "w2048"
    if kind == "step":
        return dict(kind=kind, width=width, rows=_log(rng, 1, 4 if big else 16), tokens=rng.randint(1, 64),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind in ("layer", "block"):
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return dict(kind=kind, width=width, rows=1 if dtype == "fp32" else _log(rng, 1, 4 if big else 8),
                    tokens=_log(rng, 100, 1024), chunk=rng.choice([64, 64, 64, 128]), dtype=dtype,
                    masked=rng.random() < 0.5)
    if kind == "attention":
        return dict(kind=kind, width=width, rows=_log(rng, 1, 4), tokens=_log(rng, 33, 4096),
                    history=rng.choice([0, 0, _width({"width": width})[4], rng.randint(1, 255)]), dtype="bf16")
    if kind == "readout":
        return dict(kind=kind, width=width, rows=_log(rng, 1, 4), tokens=_log(rng, 65, 2048),
                    dtype=rng.choice(["bf16", "bf16", "bf16", "fp32"]) if not big else "bf16",
                    copies=rng.random() < 0.5, shared=rng.random() < 0.3)
    if kind == "decode":
        width = rng.choice(["w512", "w768", "w1024"])
        return dict(kind=kind, width=width, rows=_log(rng, 1, 32), layers=rng.choice([6, 12]), shortest=1 + rng.randint(0, 63),
                    longest=rng.randint(64, 2048))
    if kind == "prefill":
        return dict(kind=kind, width=width, rows=_log(rng, 1, 4 if big else 8), tokens=_log(rng, 64, 2048),
                    layers=rng.randint(2, 4))
    return dict(kind=kind, width=width, rows=_log(rng, 2, 8), shortest=rng.randint(33, 128),
                longest=_log(rng, 129, 2048), layers=rng.randint(2, 4))


def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _lengths(case):
    """A ragged batch: lengths over the whole of [shortest, longest], both ends among them."""
    rng = random.Random(case["rows"] * 7919 + case["longest"])
    n = [rng.randint(case["shortest"], case["longest"]) for _ in range(case["rows"])]
    n[0] = case["longest"]
    if len(n) > 1:
        n[1] = case["shortest"]
    return n


def _chunks(tokens, chunk=64):
    return (tokens + chunk - 1) // chunk


# ------------------------------------------------------------------------------------------------
# what a program has in hand
# ------------------------------------------------------------------------------------------------

def _randn(gen, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(dtype)


def _personal_state(pool, rows, gen):
    """``rows`` users' states: W_0 moved by about a tenth, momentum of earlier turns."""
    base = [t.detach().float() for t in pool.base_weights()]
    w = [t[None] + _randn(gen, rows, *t.shape, scale=0.1 * float(t.std())) for t in base]
    s = [_randn(gen, rows, *t.shape, scale=0.002 * float(t.std())) for t in base]
    return FastWeightState(*w, *s, pool.ln_weight.detach().float().clone(), pool.ln_bias.detach().float().clone())


def _settle(module, gen):
    """Routers and norms as training leaves them: not constant."""
    for name, p in module.named_parameters():
        if name.endswith(("w_eta.weight", "w_alpha.weight")):
            p.data.copy_(_randn(gen, *p.shape, scale=0.5 / math.sqrt(p.shape[1])))
        elif name.endswith("norm.weight"):
            p.data.add_(_randn(gen, *p.shape, scale=0.1))


def _mask(case, gen):
    """Right-padded rows: between half and all of the tokens are real."""
    rows, tokens = case["rows"], case["tokens"]
    real = torch.randint(tokens // 2, tokens + 1, (rows,), generator=gen, device="cuda")
    return (torch.arange(tokens, device="cuda")[None] < real[:, None]).float()


def prepare(case, seed):
    d, ff, heads, hkv, window = _width(case)
    kind, dt = case["kind"], _dtype(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    torch.manual_seed(seed)
    st = {"kind": kind}
    if kind in ("prefill", "evolve", "decode"):
        with torch.device("cuda"):
            model = uTTTModel(uTTTConfig(vocab_size=VOCAB, d_model=d, n_layers=case["layers"], n_heads=heads,
                                         n_kv_heads=hkv, d_ff_fast=ff, sliding_window_size=window)).eval()
        model.freeze_slow_weights()
        _settle(model, gen)
        model.to(torch.bfloat16)
        pool = model.fast_weight_pool.float()
        st.update(model=model, state=_personal_state(pool, case["rows"], gen))
        if kind == "prefill":
            st["ids"] = torch.randint(6, VOCAB, (case["rows"], case["tokens"]), generator=gen, device="cuda")
            return st
        rows = [FastWeightState(*(t[i:i + 1] for t in st["state"].tensors()), st["state"].ln_weight,
                                st["state"].ln_bias) for i in range(case["rows"])]
        if kind == "evolve":
            st["turns"] = [torch.randint(6, VOCAB, (n,), generator=gen, device="cuda") for n in _lengths(case)]
            st["states"] = rows
            return st
        lengths = _lengths(case)
        hd = d // heads
        caches = [[tuple(_randn(gen, 1, hkv, min(n, window), hd, dtype=torch.bfloat16) for _ in range(2))
                   for _ in range(case["layers"])] for n in lengths]
        dec = BatchedDecoder(model, rows, max_positions=16384)
        dec.reset(caches, lengths)
        dec.capture()
        # the tokens the users' replies take: given, so that a pass does not hang on a tie of the one before
        st.update(decoder=dec, lengths=lengths, caches=caches, at=0,
                  tokens=torch.randint(6, VOCAB, (64, case["rows"]), generator=gen, device="cuda"))
        return st
    with torch.device("cuda"):
        if kind in ("step", "layer", "block", "readout"):
            pool = SharedFastWeightPool(d, ff, BETA, CLIP, normalize_loss_by_dim=True).eval()
            pool.requires_grad_(False)
            st["pool"] = pool
        if kind == "layer":
            st["layer"] = uTTTLayer(d, case["chunk"], LR, DECAY).eval()
        elif kind == "block":
            st["block"] = uTTTBlock(0, d, heads, hkv, window, case["chunk"], LR, DECAY).eval()
        elif kind == "attention":
            st["attention"] = SlidingWindowAttention(d, heads, hkv, window).eval()
    for name in ("layer", "block", "attention"):
        if name in st:
            st[name].requires_grad_(False)
            _settle(st[name], gen)
            st[name].to(dt)
            if hasattr(st[name], "prepare_for_inference"):
                st[name].prepare_for_inference()
    rows, tokens = case["rows"], case["tokens"]
    if kind == "attention":
        st["x"] = _randn(gen, rows, tokens, d, dtype=dt)
        st["cache"], st["start"] = None, 0
        if case["history"]:
            n = min(case["history"], window)
            st["cache"] = tuple(_randn(gen, rows, hkv, n, d // heads, dtype=dt) for _ in range(2))
            st["start"] = case["history"] + 100
        return st
    if kind == "readout" and case["shared"]:  # new users: W_0 itself, nothing of their own yet
        st["state"] = pool.readonly_state(rows)
    else:
        st["state"] = _personal_state(pool, rows, gen)
    if kind == "step":
        for name in ("q", "k", "v"):
            st[name] = F.rms_norm(_randn(gen, rows, tokens, d), (d,)).to(dt)
        st["eta"] = (LR * torch.sigmoid(_randn(gen, rows, tokens, 1))).to(dt)
        st["alpha"] = (DECAY * torch.sigmoid(_randn(gen, rows, tokens, 1) - 1.386)).to(dt)
        return st
    if kind == "readout":
        pool.fused_inference_readout = case["copies"]
        st["x"] = F.rms_norm(_randn(gen, rows, tokens, d), (d,)).to(dt)
        return st
    st["x"] = _randn(gen, rows, tokens, d, dtype=dt)
    st["mask"] = _mask(case, gen) if case["masked"] else None
    return st


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------

@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "step":
        out, new, surprise = state["pool"].chunk_step(state["state"], state["q"], state["k"], state["v"], state["eta"],
                                                      state["alpha"])
        return out, list(new.tensors()), surprise
    if kind == "layer":
        out, new, surprise = state["layer"](state["x"], state["pool"], state["state"], state["mask"])
        return out, list(new.tensors()), surprise
    if kind == "block":
        out, new, surprise, cache = state["block"](state["x"], state["pool"], state["state"], state["mask"])
        return out, list(new.tensors()), surprise, list(cache)
    if kind == "attention":
        out, cache = state["attention"](state["x"], state["cache"], state["start"])
        return out, list(cache)
    if kind == "readout":
        return state["pool"].forward_readout(state["x"], state["state"])
    if kind == "decode":
        dec = state["decoder"]
        logits = dec.step(state["tokens"][state["at"]])
        state["at"] = (state["at"] + 1) % state["tokens"].shape[0]
        return logits, [list(r) for r in dec.rings]
    if kind == "prefill":
        out = state["model"](state["ids"], state["state"], logits_to_keep=1)
        return out.logits, list(out.fast_state.tensors()), out.layer_surprise_losses, [c[0] for c in out.kv_caches]
    results = evolve_batched(state["model"], state["turns"], state["states"], surprise_threshold=0.5,
                             anchor_lambda=1e-3, max_drift_ratio=0.35, min_chunk_surprise=0.5)
    return [list(r.state.tensors()) for r in results], [r.surprise for r in results]


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------------

def _pairs(tokens, history, window):
    """Visible (query, key) pairs of one row and head."""
    full = max(0, tokens - max(0, window - history))
    part = tokens - full
    return full * window + part * history + part * (part + 1) // 2


def _slow_params(width, layers):
    d, _, heads, hkv, _ = width
    hd = d // heads
    return layers * (d * (heads + 2 * hkv) * hd + heads * hd * d + 4 * d * d + 2 * d)


def work(case):
    d, ff, heads, hkv, window = width = _width(case)
    kind, rows = case["kind"], case["rows"]
    e = 4 if case.get("dtype") == "fp32" else 2
    hd = d // heads
    state = 48 * d * ff * rows  # W and S, read and written
    if kind == "step":
        t = rows * case["tokens"]
        return {"bytes": state + t * (4 * d + 2) * e, "flops": 20 * d * ff * t}
    if kind == "readout":
        t = rows * case["tokens"]
        w = 2 if case["copies"] and not case["shared"] and e == 2 else 4
        return {"bytes": 3 * d * ff * w * (1 if case["shared"] else rows) + 2 * t * d * e, "flops": 6 * d * ff * t}
    if kind == "layer":
        t = rows * case["tokens"]
        return {"bytes": state + _slow_params(width, 1) * e + 2 * t * d * e, "flops": (20 * ff + 8 * d) * d * t}
    if kind in ("attention", "block"):
        t, hist = rows * case["tokens"], min(case.get("history", 0), window - 1)
        params = 2 * d * (heads + hkv) * hd
        flops = 2 * t * params + 4 * hd * heads * rows * _pairs(case["tokens"], hist, window)
        nbytes = params * e + 2 * t * d * e + 2 * rows * hkv * hd * e * (hist + min(window, hist + case["tokens"]))
        if kind == "attention":
            return {"bytes": nbytes, "flops": flops}
        return {"bytes": nbytes + state + 4 * d * d * e, "flops": flops + (20 * ff + 8 * d) * d * t}
    layers = case["layers"]
    params = _slow_params(width, layers)
    if kind == "decode":
        ctx = sum(min(n, window) for n in _lengths(case))
        return {"bytes": 2 * (params + VOCAB * d + 3 * d * ff * rows + 2 * layers * hkv * hd * ctx + rows * VOCAB),
                "flops": rows * (2 * (params + VOCAB * d) + 6 * d * ff * layers) + 4 * hd * heads * layers * ctx}
    lengths = [case["tokens"]] * rows if kind == "prefill" else _lengths(case)
    t = sum(lengths)
    flops = t * (2 * params + 20 * d * ff * layers) + 4 * hd * heads * layers * sum(_pairs(n, 0, window) for n in lengths)
    nbytes = state + 2 * params + 2 * t * d
    if kind == "prefill":
        flops += 2 * rows * VOCAB * d
        nbytes += 2 * VOCAB * d
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "step":
        return {"rel": 1e-2, "max": 0.5}
    if kind in ("layer", "block"):
        return {"rel": 2e-2, "max": 0.5}
    if kind in ("attention", "readout"):
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 3e-2, "max": 0.9}


# ------------------------------------------------------------------------------------------------
# the same in 64 bits, with plain torch
# ------------------------------------------------------------------------------------------------

def _norm(x, weight=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if weight is None else y * weight


def _readout(x, w, ln):
    z = (F.silu(x @ w[1]) * (x @ w[0])) @ w[2]
    return x + F.layer_norm(z, (z.shape[-1],), ln[0], ln[1], EPS)


def _write(k, v, eta, alpha, w, s, ln, mask, gate=0.0):
    """(new W, new S, per-row loss sums, per-row token counts) of one chunk; W and S as lists of 3."""
    dim = k.shape[-1]
    up, pre = k @ w[0], k @ w[1]
    sig = torch.sigmoid(pre)
    hid = pre * sig * up
    z = hid @ w[2]
    cent = z - z.mean(-1, keepdim=True)
    rstd = torch.rsqrt(cent.square().mean(-1, keepdim=True) + EPS)
    zh = cent * rstd
    err = k + zh * ln[0] + ln[1] - v
    loss = 0.5 * err.square().sum(-1) / dim
    m = torch.ones_like(loss) if mask is None else mask
    n = m.sum(1)
    weight = (eta[..., 0] * m / n.clamp_min(1.0)[:, None])[..., None]
    dzh = weight / dim * err * ln[0]
    dz = rstd * (dzh - dzh.mean(-1, keepdim=True) - zh * (dzh * zh).mean(-1, keepdim=True))
    dh = dz @ w[2].transpose(1, 2)
    du = dh * pre * sig
    dg = dh * up * sig * (1 + pre * (1 - sig))
    kt = k.transpose(1, 2)
    grads = [kt @ du, kt @ dg, hid.transpose(1, 2) @ dz]
    clip = torch.rsqrt(sum(g.square().sum((1, 2)) for g in grads) + 1e-8).mul(CLIP).clamp(max=1.0).view(-1, 1, 1)
    decay = 1 - ((alpha[..., 0] * m).sum(1) / n.clamp_min(1.0)).view(-1, 1, 1)
    row = (loss * m).sum(1)
    keep = (n > 0) & ((row / n.clamp_min(1.0) >= gate) if gate > 0 else (n > 0))
    keep = keep.view(-1, 1, 1)
    new_s = [torch.where(keep, BETA * b - clip * g, b) for b, g in zip(s, grads)]
    new_w = [torch.where(keep, decay * a + b, a) for a, b in zip(w, new_s)]
    return new_w, new_s, row, n


def _rotate(x, start):
    """RoPE on (B, H, T, hd) from position ``start``, or from one position for each row."""
    hd, t = x.shape[-1], x.shape[2]
    inv = 1.0 / (THETA ** (torch.arange(0, hd, 2, device=x.device, dtype=torch.float64) / hd))
    pos = torch.as_tensor(start, device=x.device, dtype=torch.float64).view(-1, 1) + torch.arange(t, device=x.device)
    ang = (pos[..., None] * inv)[:, None]
    cos, sin = torch.cat((ang.cos(), ang.cos()), -1), torch.cat((ang.sin(), ang.sin()), -1)
    half = hd // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), -1) * sin


def _attend(q, k, v, window, offset):
    out = torch.empty_like(q)
    rep, t = q.shape[1] // k.shape[1], q.shape[2]
    for i in range(0, t, 256):
        j = min(t, i + 256)
        lo = max(0, offset + i - window + 1)
        kk, vv = (x[:, :, lo:offset + j].repeat_interleave(rep, 1) for x in (k, v))
        dist = (torch.arange(i, j, device=q.device)[:, None] + offset) - torch.arange(lo, offset + j, device=q.device)
        sc = q[:, :, i:j] @ kk.transpose(-1, -2) / math.sqrt(q.shape[-1])
        out[:, :, i:j] = torch.softmax(sc.masked_fill((dist < 0) | (dist >= window), -math.inf), -1) @ vv
    return out


def _double(module):
    return {n: p.detach().double() for n, p in module.named_parameters()}


def _attention(x, p, case, cache, start):
    """(output, rotated keys and values, history first), ``p`` with the names of SlidingWindowAttention."""
    d, _, heads, hkv, window = _width(case)
    b, t, _ = x.shape
    q, k, v = ((x @ p[n + ".weight"].t()).view(b, t, -1, d // heads).transpose(1, 2) for n in ("wq", "wk", "wv"))
    q, k = _rotate(q, start), _rotate(k, start)
    hist = 0
    if cache is not None:
        hist = min(cache[0].shape[2], window - 1)
        k, v = (torch.cat((c[:, :, c.shape[2] - hist:], x), 2) for c, x in zip(cache, (k, v)))
    out = _attend(q, k, v, window, hist)
    return out.transpose(1, 2).reshape(b, t, d) @ p["wo.weight"].t(), (k, v)


def _projections(x, p):
    q, k, v = (x @ p[n + ".weight"].t() for n in ("w_q", "w_k", "w_v"))
    eta = LR * torch.sigmoid(x @ p["w_eta.weight"].t() + p["w_eta.bias"])
    alpha = DECAY * torch.sigmoid(x @ p["w_alpha.weight"].t() + p["w_alpha.bias"])
    return _norm(q, p["q_norm.weight"]), _norm(k, p["k_norm.weight"]), _norm(v), eta, alpha


def _layer(x, p, case, w, s, ln, mask):
    q, k, v, eta, alpha = _projections(x, p)
    outs, losses = [], []
    for i in range(0, x.shape[1], case["chunk"]):
        sl = slice(i, i + case["chunk"])
        outs.append(_readout(q[:, sl], w, ln))
        w, s, row, n = _write(k[:, sl], v[:, sl], eta[:, sl], alpha[:, sl], w, s, ln, None if mask is None else mask[:, sl])
        losses.append(row.sum() / n.sum().clamp_min(1.0))
    return torch.cat(outs, 1) @ p["w_o.weight"].t(), w, s, torch.stack(losses).mean()


def _part(p, prefix):
    return {n[len(prefix):]: t for n, t in p.items() if n.startswith(prefix)}


def _model(model, case, ids, mask, w, s, ln, gate=0.0):
    """(hidden, W, S, per-row loss and token sums (2, rows, layers), keys of every layer) of the chunk-first pass."""
    window = _width(case)[4]
    layers = [_double(m) for m in model.layers]
    emb = model.tok_embeddings.weight.detach()
    caches = [None] * len(layers)
    sums, hidden = 0, []
    for i in range(0, ids.shape[1], 64):
        h = F.embedding(ids[:, i:i + 64], emb).double()
        m = None if mask is None else mask[:, i:i + 64]
        read, sums_c = w, []
        for li, p in enumerate(layers):
            a, kv = _attention(_norm(h, p["attn_norm.weight"]), _part(p, "attn."), case, caches[li], i)
            caches[li] = tuple(t[:, :, -window:] for t in kv)
            h = h + a
            u = _part(p, "uttt.")
            q, k, v, eta, alpha = _projections(_norm(h, p["uttt_norm.weight"]), u)
            h = h + _readout(q, read, ln) @ u["w_o.weight"].t()
            w, s, row, n = _write(k, v, eta, alpha, w, s, ln, m, gate)
            sums_c.append(torch.stack((row, n)))
        sums = sums + torch.stack(sums_c, -1)
        hidden.append(h[:, -1:])
    return hidden[-1], w, s, sums, [c[0] for c in caches]


def exact(case, seed):
    with torch.no_grad():
        return _exact(case, prepare(case, seed))


def _exact(case, st):
    d, ff, heads, hkv, window = _width(case)
    kind = case["kind"]
    if kind == "attention":
        cache = None if st["cache"] is None else tuple(t.double() for t in st["cache"])
        out, kv = _attention(st["x"].double(), _double(st["attention"]), case, cache, st["start"])
        return out, [t[:, :, -window:] for t in kv]
    if kind == "decode":
        return _exact_decode(case, st)
    state = st["state"]
    ten = [t.double() for t in state.tensors()]
    w, s, ln = ten[:3], ten[3:], (state.ln_weight.double(), state.ln_bias.double())
    if kind == "readout":
        return _readout(st["x"].double(), w, ln)
    if kind == "step":
        q, k, v, eta, alpha = (st[n].double() for n in ("q", "k", "v", "eta", "alpha"))
        out = _readout(q, w, ln)
        w, s, row, n = _write(k, v, eta, alpha, w, s, ln, None)
        return out, w + s, row.sum() / n.sum()
    if kind in ("layer", "block"):
        x, mask = st["x"].double(), None if st["mask"] is None else st["mask"].double()
        if kind == "layer":
            out, w, s, surprise = _layer(x, _double(st["layer"]), case, w, s, ln, mask)
            return out, w + s, surprise
        p = _double(st["block"])
        a, kv = _attention(_norm(x, p["attn_norm.weight"]), _part(p, "attn."), case, None, 0)
        h = x + a
        out, w, s, surprise = _layer(_norm(h, p["uttt_norm.weight"]), _part(p, "uttt."), case, w, s, ln, mask)
        return h + out, w + s, surprise, [t[:, :, -window:] for t in kv]
    model = st["model"]
    if kind == "prefill":
        h, w, s, sums, keys = _model(model, case, st["ids"], None, w, s, ln)
        logits = _norm(h, model.norm.weight.double()) @ model.lm_head.weight.double().t()
        surprise = sums[0].sum(0) / sums[1].sum(0)
        return logits, w + s, surprise.tolist(), keys
    lengths = _lengths(case)
    longest = 64 * _chunks(max(lengths))
    ids = torch.zeros((len(lengths), longest), dtype=torch.long, device="cuda")
    mask = torch.zeros((len(lengths), longest), dtype=torch.float64, device="cuda")
    for i, t in enumerate(st["turns"]):
        ids[i, :len(t)] = t
        mask[i, :len(t)] = 1.0
    _, w, s, sums, _ = _model(model, case, ids, mask, w, s, ln, gate=0.5)
    base = [t.double()[None] for t in model.fast_weight_pool.base_weights()]
    surprise = (sums[0] / sums[1]).mean(-1)
    diff = [0.999 * (a - b) for a, b in zip(w, base)]
    drift = torch.sqrt(sum(x.square().sum((1, 2)) for x in diff) + 1e-8)
    scale = (0.35 * torch.sqrt(sum(b.square().sum() for b in base) + 1e-8) / drift).clamp(max=1.0).view(-1, 1, 1)
    w = [b + x * scale for b, x in zip(base, diff)]
    return [[t[i:i + 1] for t in w + s] for i in range(len(lengths))], surprise.tolist()


def _exact_decode(case, st):
    """One step from the given caches: the rings (token p in slot p mod window) and the logits."""
    d, ff, heads, hkv, window = _width(case)
    hd, lengths, model = d // heads, st["lengths"], st["model"]
    ten = [t.double() for t in st["state"].tensors()[:3]]
    ln = (st["state"].ln_weight.double(), st["state"].ln_bias.double())
    h = F.embedding(st["tokens"][0], model.tok_embeddings.weight).double()[:, None]
    rows, rings = len(lengths), []
    for li, m in enumerate(model.layers):
        p = _double(m)
        x = _norm(h, p["attn_norm.weight"])
        q, k, v = ((x @ p["attn.%s.weight" % n].t()).view(rows, 1, -1, hd).transpose(1, 2) for n in ("wq", "wk", "wv"))
        q, k = _rotate(q, lengths), _rotate(k, lengths)
        ring = [torch.zeros((rows, hkv, window, hd), dtype=torch.float64, device="cuda") for _ in range(2)]
        att = torch.empty_like(q)
        for i, n in enumerate(lengths):
            kept = min(n, window)
            slots = torch.arange(n - kept, n, device="cuda") % window
            for r, c, new in zip(ring, st["caches"][i][li], (k, v)):
                r[i, :, slots] = c[0].double()
                r[i, :, n % window] = new[i, :, 0]
            kk, vv = (r[i, :, :min(n + 1, window)].repeat_interleave(heads // hkv, 0) for r in ring)
            att[i] = torch.softmax(q[i] @ kk.transpose(-1, -2) / math.sqrt(hd), -1) @ vv
        rings.append(ring)
        h = h + att.transpose(1, 2).reshape(rows, 1, d) @ p["attn.wo.weight"].t()
        q = _norm(_norm(h, p["uttt_norm.weight"]) @ p["uttt.w_q.weight"].t(), p["uttt.q_norm.weight"])
        h = h + _readout(q, ten, ln) @ p["uttt.w_o.weight"].t()
    logits = _norm(h[:, 0], model.norm.weight.double()) @ model.lm_head.weight.double().t()
    return logits, rings
