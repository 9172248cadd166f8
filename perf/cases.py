"""The workloads that this framework's speed is judged by.

Each case is a call that a program using LoGo on MI355X makes: the
query-sparse attention operator in training and in prefill, the sliding-window
branch, one LoGo attention layer in training and at decode, one decoder layer
of a prompt, and a decode step of the whole causal LM.  ``listed`` names them,
``draw`` gives further sizes and options of the same ranges, ``prepare`` makes
a case's inputs on the GPU from a seed, ``run`` is one pass through the public
entry points, ``exact`` the same result in 64-bit torch arithmetic.
"""

import math

import numpy as np
import torch
import torch.nn.functional as F

from logo_amd.layers import LoGoAttention, LoGoConfig, rope_cos_sin
from logo_amd.model import LoGoDecoderLayer, LoGoForCausalLM
from logo_amd.ops import sq_full_attn, swa_attn
from logo_amd.ops.decode import LogoKVCache

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
MEAN_RUN = 8  # mean length of the spans of selected tokens


def _attn(name, tokens, seqs, heads, kv_heads, k_dim, v_dim, dtype, ratio, per_head=False, backward=True, window=-1):
    """One operator call; window -1: sq_full_attn, else swa_attn over every row."""
    c = {"kind": "attn", "tokens": tokens, "seqs": seqs, "heads": heads, "kv_heads": kv_heads, "k_dim": k_dim,
         "v_dim": v_dim, "dtype": dtype, "ratio": ratio, "per_head": per_head, "backward": backward, "window": window}
    return {"name": name, **c} if name else c


def _layer(name, kind, batch, tokens, heads, kv_heads, head_dim=128, layers=1):
    """kind: layer_train, layer_decode (tokens = cached ones), decoder_prefill, model_decode (tokens = the prompt)."""
    c = {"kind": kind, "batch": batch, "tokens": tokens, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
         "layers": layers}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest call: one short fp32 sequence, each (head, token) row selected by itself; launches count
        _attn("attn_small_fp32", 512, 1, 4, 4, 64, 64, "fp32", 0.5, per_head=True),
        # prefill: forward only, every head with its own selected rows, heads of the 1.5B model
        _attn("attn_prefill_per_head", 8192, 1, 16, 16, 128, 128, "bf16", 0.5, per_head=True, backward=False),
        # a training batch of packed sequences of uneven, odd lengths
        _attn("attn_train_packed", 32373, 4, 16, 16, 128, 128, "bf16", 0.25),
        # training on one long sequence, a quarter of its tokens global
        _attn("attn_train_32k", 32768, 1, 16, 16, 128, 128, "bf16", 0.25),
        # fp16 training with grouped key / value heads of dim 64, medium length
        _attn("attn_train_gqa_fp16", 6001, 2, 16, 4, 64, 64, "fp16", 0.4),
        # the widest head the operator takes
        _attn("attn_train_wide", 8192, 1, 16, 16, 256, 256, "bf16", 0.25),
        # training in full fp32
        _attn("attn_train_fp32", 4096, 1, 16, 16, 128, 128, "fp32", 0.25),
        # the local branch by itself: window 128, packed ragged sequences, forward and backward
        _attn("swa_train", 20011, 3, 16, 16, 128, 128, "bf16", 1.0, window=128),
        # the LoGo attention layer of the 1.5B model in training: all parameters' gradients
        _layer("layer_train", "layer_train", 4, 8192, 16, 16),
        # one decoder layer over a batch of prompts, filling the cache (attention, norms and MLP, no gradients)
        _layer("decoder_prefill", "decoder_prefill", 2, 3001, 16, 16),
        # one layer of a decode step: a full batch with long contexts, about half of the rows global
        _layer("layer_decode", "layer_decode", 32, 16384, 16, 16),
        # a whole decode step of the 24-layer model for a few users with short prompts, replayed from its graph
        _layer("model_decode", "model_decode", 4, 500, 16, 16, layers=24),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("attn", "attn", "attn", "fp32", "wide", "swa", "layer_train", "decoder_prefill", "layer_decode",
                       "model_decode"))
    if kind == "attn":
        heads = rng.choice((4, 8, 16))
        dim = rng.choice((64, 128, 128))
        return _attn(None, _log(rng, 500, 32768), rng.randint(1, 5), heads, heads // rng.choice((1, 1, 2, 4)), dim, dim,
                     rng.choice(("bf16", "bf16", "fp16")), round(rng.uniform(0.1, 0.5), 3),
                     per_head=rng.random() < 0.25, backward=rng.random() < 0.75)
    if kind == "fp32":
        heads, dim = rng.choice((4, 8, 16)), rng.choice((64, 128))
        return _attn(None, _log(rng, 300, 5000), rng.randint(1, 3), heads, heads // rng.choice((1, 2)), dim, dim, "fp32",
                     round(rng.uniform(0.1, 0.5), 3), per_head=rng.random() < 0.25, backward=rng.random() < 0.75)
    if kind == "wide":
        heads = rng.choice((4, 8, 16))
        return _attn(None, _log(rng, 500, 9000), rng.randint(1, 3), heads, heads // rng.choice((1, 2)),
                     rng.choice((160, 192, 256)), rng.choice((128, 256)), "bf16", round(rng.uniform(0.1, 0.4), 3),
                     backward=rng.random() < 0.75)
    if kind == "swa":
        return _attn(None, _log(rng, 500, 32768), rng.randint(1, 5), rng.choice((8, 16)), 8, 128, 128, "bf16", 1.0,
                     backward=rng.random() < 0.75, window=128)
    heads = rng.choice((8, 16))
    if kind == "layer_train":
        return _layer(None, kind, rng.randint(1, 4), _log(rng, 200, 8000), heads, heads // rng.choice((1, 1, 4)))
    if kind == "decoder_prefill":
        return _layer(None, kind, rng.randint(1, 4), _log(rng, 200, 4000), heads, heads // rng.choice((1, 1, 4)))
    if kind == "layer_decode":
        return _layer(None, kind, _log(rng, 1, 32), _log(rng, 200, 16384), heads, heads // rng.choice((1, 1, 4)))
    return _layer(None, kind, _log(rng, 1, 16), _log(rng, 100, 1000), heads, heads, layers=rng.randint(8, 24))


# ---------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(shape, gen, dtype, std=1.0):
    return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)


def _lengths(tokens, seqs, seed):
    """`tokens` cut into `seqs` uneven lengths, fixed by the case (not by the seed): ratios about 1 to 4."""
    w = np.random.RandomState(1000 * seqs + tokens % 997).uniform(1.0, 4.0, seqs)
    cuts = np.floor(np.cumsum(w) / w.sum() * tokens).astype(np.int64)
    cuts[-1] = tokens
    return np.diff(np.concatenate([[0], cuts])).tolist()


def _spans(n, ratio, rng):
    """A selection in spans: runs of selected tokens of mean length MEAN_RUN, gaps to give `ratio`; token 0 selected."""
    gap = MEAN_RUN * (1.0 - ratio) / ratio
    count = int(2 * n / (MEAN_RUN + gap)) + 16
    runs = np.empty(2 * count, dtype=np.int64)
    runs[0::2] = rng.geometric(1.0 / MEAN_RUN, count)
    runs[1::2] = rng.geometric(1.0 / max(gap, 1.0), count)
    sel = np.repeat(np.tile([True, False], count), runs)
    sel = np.concatenate([sel, np.zeros(max(0, n - sel.size), dtype=bool)])[:n]
    return sel


def _attn_inputs(case, seed):
    n, dt, gen = case["tokens"], DTYPES[case["dtype"]], _gen(seed)
    q = _randn((1, n, case["heads"], case["k_dim"]), gen, dt, 0.5)
    k = _randn((1, n, case["kv_heads"], case["k_dim"]), gen, dt, 0.5)
    v = _randn((1, n, case["kv_heads"], case["v_dim"]), gen, dt, 0.5)
    do = _randn((1, n, case["heads"], case["v_dim"]), gen, dt)
    lens = _lengths(n, case["seqs"], seed)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=DEV)
    sel = None
    if case["window"] < 0:
        if case["per_head"]:
            sel = torch.rand((1, n, case["heads"]), generator=gen, device=DEV) < case["ratio"]
            sel[:, 0] = True
        else:
            sel = torch.from_numpy(_spans(n, case["ratio"], np.random.RandomState(seed % (1 << 31)))).to(DEV)[None]
    if case["backward"]:
        for t in (q, k, v):
            t.requires_grad_()
    return {"q": q, "k": k, "v": v, "do": do, "sel": sel, "cu": cu, "lens": lens}


def _config(case, **kw):
    return LoGoConfig(hidden_size=case["heads"] * case["head_dim"], num_attention_heads=case["heads"],
                      num_key_value_heads=case["kv_heads"], num_hidden_layers=case["layers"],
                      intermediate_size=case["heads"] * case["head_dim"] * 11 // 4, window_size=128, **kw)


def _init(module, gen):
    """Linear weights ~ N(0, 0.02), global maps near identity, gate logits of unit variance, norm weights near one."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("_global_proj"):
                p.add_(torch.randn(p.shape, generator=gen, device=DEV) * 0.02)
            elif name.endswith("self_attn.gate_proj.weight") or name == "gate_proj.weight":
                p.copy_(torch.randn(p.shape, generator=gen, device=DEV) / p.shape[1] ** 0.5)
            elif p.dim() == 2:
                p.copy_(torch.randn(p.shape, generator=gen, device=DEV) * 0.02)
            else:
                p.add_(torch.randn(p.shape, generator=gen, device=DEV) * 0.1)
    return module.to(dtype=torch.bfloat16)


def _layer_inputs(case, seed):
    gen, b, t, kind = _gen(seed), case["batch"], case["tokens"], case["kind"]
    # the model's threshold lies low, where a gate near it carries little: which side of it a gate falls then does not
    # depend on 16-bit rounding in the layers before; a single layer selects half of the tokens
    cfg = _config(case, gate_thres_init=0.05 if kind == "model_decode" else 0.5)
    c = cfg.hidden_size
    with torch.device(DEV):
        if kind == "model_decode":
            model = LoGoForCausalLM(cfg)
            model.init_weights(gen)
            model = model.to(dtype=torch.bfloat16).eval()
        elif kind == "decoder_prefill":
            layer = _init(LoGoDecoderLayer(cfg, 0), gen).eval()
        else:
            layer = _init(LoGoAttention(cfg), gen)
    if kind == "layer_train":
        h = _randn((b, t, c), gen, torch.bfloat16).requires_grad_()
        return {"layer": layer.train(), "h": h, "dout": _randn((b, t, c), gen, torch.bfloat16),
                "params": [p for p in layer.parameters()]}
    if kind == "decoder_prefill":
        cache = LogoKVCache(1, b, cfg.num_key_value_heads, cfg.head_dim, t + 64, window=128, device=DEV)
        pos = torch.arange(t, device=DEV)[None].expand(b, t)
        return {"layer": layer, "h": _randn((b, t, c), gen, torch.bfloat16), "cache": cache,
                "pe": rope_cos_sin(pos, cfg.head_dim, cfg.rope_theta, torch.bfloat16)}
    if kind == "layer_decode":
        cache = LogoKVCache(1, b, cfg.num_key_value_heads, cfg.head_dim, t + 64, window=128, device=DEV)
        for x in (cache.global_k[0], cache.global_v[0], cache.local_k[0], cache.local_v[0]):
            x.normal_(0.0, 0.7, generator=gen)
        cache.set_length(t)
        return {"layer": layer.eval(), "h": _randn((b, 1, c), gen, torch.bfloat16), "cache": cache,
                "pe": rope_cos_sin(cache.positions(1), cfg.head_dim, cfg.rope_theta, torch.bfloat16)}
    prompt = torch.randint(0, cfg.vocab_size, (b, t), generator=gen, device=DEV)
    cache = model.new_cache(b, t + 64, device=DEV)
    tok = torch.randint(0, cfg.vocab_size, (b,), generator=gen, device=DEV)
    model.prefill(prompt, cache)
    model.decode_step(tok, cache)
    cache.set_length(t)
    return {"model": model, "cache": cache, "tok": tok, "prompt": t, "step": model.capture_greedy_decode(tok, cache)}


def prepare(case, seed):
    s = _attn_inputs(case, seed) if case["kind"] == "attn" else _layer_inputs(case, seed)
    s["case"] = case
    return s


# ---------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        q, k, v = state["q"], state["k"], state["v"]
        if not case["backward"]:
            with torch.no_grad():
                return _attend(state)
        o = _attend(state)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), state["do"]))
    if kind == "layer_train":
        out, _, _ = state["layer"](state["h"])
        return (out.detach(), *torch.autograd.grad(out, [state["h"]] + state["params"], state["dout"]))
    with torch.no_grad():
        cache = state["cache"]
        if kind == "decoder_prefill":
            cache.reset()
            out = state["layer"](state["h"], past_key_value=cache, position_embeddings=state["pe"])
            cache.set_length(case["tokens"])
            t = case["tokens"]
            return out, cache.global_k[0][:, :, :t], cache.global_v[0][:, :, :t]
        if kind == "layer_decode":
            out, _, _ = state["layer"](state["h"], past_key_value=cache, position_embeddings=state["pe"])
            t = case["tokens"]
            return out, cache.global_k[0][:, :, t], cache.global_v[0][:, :, t]
        # a step behind the cached prompt; the step's token buffer takes the next tokens to score
        cache.set_length(state["prompt"])
        logits, tokens = state["step"]()
        tokens.copy_(state["tok"])
        return logits


def _attend(state):
    if state["case"]["window"] >= 0:
        return swa_attn(state["q"], state["k"], state["v"], state["cu"], window=state["case"]["window"])
    return sq_full_attn(state["q"], state["k"], state["v"], state["sel"], cu_seqlens=state["cu"])


# ---------------------------------------------------------------- what a pass cannot do without


def _pairs(case):
    """Visible (query, key) pairs over all heads, taken at the case's mean selection ratio."""
    total = 0.0
    for n in _lengths(case["tokens"], case["seqs"], 0):
        if case["window"] >= 0:
            w = min(case["window"] + 1, n)
            total += w * (w + 1) / 2 + (n - w) * w
        else:
            total += case["ratio"] * n * (n + 1) / 2
    return total * case["heads"]


def work(case):
    kind = case["kind"]
    if kind == "attn":
        size = 4 if case["dtype"] == "fp32" else 2
        n, dk, dv = case["tokens"], case["k_dim"], case["v_dim"]
        q, o = n * case["heads"] * dk * size, n * case["heads"] * dv * size
        k, v = n * case["kv_heads"] * dk * size, n * case["kv_heads"] * dv * size
        qs, os_ = q * case["ratio"], o * case["ratio"]  # rows read of the selected tokens only
        pairs = _pairs(case)
        nbytes = qs + k + v + o
        flops = 2 * (dk + dv) * pairs
        if case["backward"]:
            nbytes += qs + k + v + 2 * os_ + q + k + v
            flops += (6 * dk + 4 * dv) * pairs
        return {"bytes": nbytes, "flops": flops}
    b, t, h, hk, d = case["batch"], case["tokens"], case["heads"], case["kv_heads"], case["head_dim"]
    c, inter = h * d, h * d * 11 // 4
    weights = c * (h + 2 * hk) * d + c + c * c + (h + 2 * hk) * d * d  # projections, gate, output, global maps
    maps = 2 * (c * (h + 2 * hk) * d + c + c * c) + 2 * (h + 2 * hk) * d * d  # FLOPs of them per token
    if kind in ("layer_train", "decoder_prefill"):
        n = b * t
        pairs = b * h * (0.5 * t * (t + 1) / 2 + min(t, 129) * t)
        if kind == "layer_train":
            return {"bytes": 2 * (4 * n * c + 2 * weights), "flops": 3 * maps * n + 14 * d * pairs}
        return {"bytes": 2 * (2 * n * c + 2 * n * hk * d + weights + 3 * c * inter),
                "flops": (maps + 6 * c * inter) * n + 4 * d * pairs}
    # decode: the cached rows that the step reads, and all weights once; half of a single layer's rows are global, all of the model's
    share = 0.5 if kind == "layer_decode" else 1.0
    rows = b * hk * (share * (t + 1) + min(t + 1, 129))
    flops = maps * b + 4 * d * h * b * (share * (t + 1) + min(t + 1, 129))
    if kind == "layer_decode":
        return {"bytes": 2 * (weights + 2 * rows * d + 2 * b * c), "flops": flops}
    vocab = 32000
    return {"bytes": 2 * (case["layers"] * (weights + 3 * c * inter + 2 * rows * d) + vocab * c + b * vocab),
            "flops": case["layers"] * (flops + 6 * c * inter * b) + 2 * vocab * c * b}


# About four times what these paths differ by from 64-bit arithmetic; 24 layers whose projections are summed in another
# order differ by 0.016.
def tolerance(case):
    if case["kind"] == "attn":
        return {"rel": {"bf16": 0.012, "fp16": 1.6e-3, "fp32": 4e-6}[case["dtype"]]}
    return {"rel": 0.03 if case["kind"] == "model_decode" else 0.025}


# ---------------------------------------------------------------- 64-bit results


class _Attend64(torch.autograd.Function):
    """Softmax attention in float64 on [N, heads, D] tensors: rows [HQ or 1][R] of token indices attend the keys of
    their own segment up to themselves (at most `window` back); other rows are zero."""

    BLOCK = 512

    @staticmethod
    def blocks(rows, lens, window):
        start = 0
        for n in lens:
            mine = rows[(rows >= start) & (rows < start + n)]
            for r in mine.split(_Attend64.BLOCK):
                if r.numel():
                    last = int(r[-1])
                    first = max(start, int(r[0]) - window) if window >= 0 else start
                    keys = torch.arange(first, last + 1, device=r.device)
                    seen = keys[None] <= r[:, None]
                    if window >= 0:
                        seen &= keys[None] >= r[:, None] - window
                    yield r, first, last + 1, seen
            start += n

    @staticmethod
    def probs(q, k, r, a, b, seen, scale):
        s = torch.matmul(q[r].transpose(0, 1), k[a:b].permute(1, 2, 0)) * scale
        return torch.softmax(s.masked_fill(~seen[None], float("-inf")), -1)

    @staticmethod
    def per_head(heads, rows):
        """(head slice, rows): all heads at once where they share their rows."""
        if len(rows) == 1:
            return [(slice(0, heads), rows[0])]
        return [(slice(i, i + 1), r) for i, r in enumerate(rows)]

    @staticmethod
    def forward(ctx, q, k, v, rows, lens, scale, window):
        o = q.new_zeros(q.shape[0], q.shape[1], v.shape[2])
        for hs, rw in _Attend64.per_head(q.shape[1], rows):
            qh, kh, vh = q[:, hs], k[:, hs], v[:, hs]
            for r, a, b, seen in _Attend64.blocks(rw, lens, window):
                p = _Attend64.probs(qh, kh, r, a, b, seen, scale)
                o[r, hs] = torch.matmul(p, vh[a:b].transpose(0, 1)).transpose(0, 1)
        ctx.save_for_backward(q, k, v)
        ctx.rest = (rows, lens, scale, window)
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v = ctx.saved_tensors
        rows, lens, scale, window = ctx.rest
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for hs, rw in _Attend64.per_head(q.shape[1], rows):
            qh, kh, vh, dh = q[:, hs], k[:, hs], v[:, hs], do[:, hs]
            for r, a, b, seen in _Attend64.blocks(rw, lens, window):
                p = _Attend64.probs(qh, kh, r, a, b, seen, scale)
                g = dh[r].transpose(0, 1)
                dv[a:b, hs] += torch.matmul(p.transpose(1, 2), g).transpose(0, 1)
                dp = torch.matmul(g, vh[a:b].permute(1, 2, 0))
                ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale
                dq[r, hs] = torch.matmul(ds, kh[a:b].transpose(0, 1)).transpose(0, 1)
                dk[a:b, hs] += torch.matmul(ds.transpose(1, 2), qh[r].transpose(0, 1)).transpose(0, 1)
        return dq, dk, dv, None, None, None, None


def _attend64(q, k, v, rows, lens, window=-1, scale=None):
    """[N, HQ, K], [N, H, K], [N, H, V] in float64; grouped heads repeated."""
    g = q.shape[1] // k.shape[1]
    if g > 1:
        k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    return _Attend64.apply(q, k, v, rows, lens, q.shape[2] ** -0.5 if scale is None else scale, window)


def _exact_attn(case, seed):
    s = _attn_inputs(case, seed)
    n = case["tokens"]
    q, k, v = (s[x][0].detach().double().requires_grad_() for x in "qkv")
    if s["sel"] is None:
        rows = [torch.arange(n, device=DEV)]
    elif case["per_head"]:
        rows = [torch.nonzero(s["sel"][0, :, h]).flatten() for h in range(case["heads"])]
    else:
        rows = [torch.nonzero(s["sel"][0]).flatten()]
    o = _attend64(q, k, v, rows, s["lens"], case["window"])
    if not case["backward"]:
        return o.detach()[None]
    grads = torch.autograd.grad(o, (q, k, v), s["do"][0].double())
    return (o.detach()[None], *(g[None] for g in grads))


def _norm64(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _rope64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos[..., None, :] + torch.cat((-x[..., half:], x[..., :half]), -1) * sin[..., None, :]


def _inputs64(p, h, cos, sin, heads, kv_heads, d):
    """q, k, v, global q, k, v (rotated) and the gate of hidden states [B, T, C]."""
    b, t, _ = h.shape
    out = []
    for x, n in (("q", heads), ("k", kv_heads), ("v", kv_heads)):
        y = (h @ p[x + "_proj.weight"].T).view(b, t, n, d)
        out += [y, torch.einsum("bthd,hde->bthe", y, p[x + "_global_proj"])]
    q, gq, k, gk, v, gv = out
    q, gq, k, gk = (_rope64(x, cos, sin) for x in (q, gq, k, gk))
    return q, k, v, gq, gk, gv, torch.sigmoid(h @ p["gate_proj.weight"].T)[..., 0]


def _gated(h16, w16, thres):
    """Which tokens the gate selects: the comparison is made on the 16-bit gate, from the 16-bit logit."""
    logit = (h16.double() @ w16.double().T)[..., 0].to(torch.bfloat16)
    return torch.sigmoid(logit) >= thres


def _fuse64(p, local, glob, gate, sel, eps):
    local = _norm64(local, p["context_norm_local.weight"], eps)
    glob = _norm64(glob, p["context_norm_global.weight"], eps)
    g = torch.where(sel, gate, torch.zeros_like(gate))[..., None, None]
    return ((1 - g) * local + g * glob).flatten(-2)


def _params64(module):
    return {n: x.detach().double().requires_grad_() for n, x in module.named_parameters()}


def _sequence64(p, h, cos, sin, sel, eps, heads, kv_heads, d):
    """The attention layer over [B, T, C], and its rotated global k and v."""
    b, t, _ = h.shape
    q, k, v, gq, gk, gv, gate = _inputs64(p, h, cos, sin, heads, kv_heads, d)
    flat = lambda x: x.reshape(b * t, x.shape[2], d)  # noqa: E731
    lens = [t] * b
    local = _attend64(flat(q), flat(k), flat(v), [torch.arange(b * t, device=DEV)], lens, 128)
    glob = _attend64(flat(gq), flat(gk), flat(gv), [torch.nonzero(sel.flatten()).flatten()], lens)
    y = _fuse64(p, local.view(b, t, heads, d), glob.view(b, t, heads, d), gate, sel, eps)
    return y @ p["o_proj.weight"].T, gk, gv


def exact(case, seed):
    if case["kind"] == "attn":
        return _exact_attn(case, seed)
    if case["kind"] == "model_decode":
        return None  # the gates of later layers hang on the rounding of those before
    s = _layer_inputs(case, seed)
    heads, kv_heads, d, eps = case["heads"], case["kv_heads"], case["head_dim"], 1e-5
    b, t, layer = case["batch"], case["tokens"], s["layer"]
    if case["kind"] == "layer_train":
        p, h = _params64(layer), s["h"].detach().double().requires_grad_()
        pos = torch.arange(t, device=DEV)[None].expand(b, t)
        cos, sin = (x.double() for x in rope_cos_sin(pos, d, layer.config.rope_theta, torch.bfloat16))
        sel = _gated(s["h"].detach(), layer.gate_proj.weight.detach(), layer.gate_thres)
        out, _, _ = _sequence64(p, h, cos, sin, sel, eps, heads, kv_heads, d)
        return (out.detach(), *torch.autograd.grad(out, [h] + list(p.values()), s["dout"].double()))
    cos, sin = (x.double() for x in s["pe"])
    with torch.no_grad():
        if case["kind"] == "decoder_prefill":
            p = _params64(layer)
            a = {n[len("self_attn."):]: x for n, x in p.items() if n.startswith("self_attn.")}
            h = s["h"].double()
            x32 = s["h"].float()
            x16 = layer.input_layernorm.weight * (x32 * torch.rsqrt(x32.pow(2).mean(-1, keepdim=True) + eps)).bfloat16()
            sel = _gated(x16, layer.self_attn.gate_proj.weight, layer.self_attn.gate_thres)
            y, gk, gv = _sequence64(a, _norm64(h, p["input_layernorm.weight"], eps), cos, sin, sel, eps, heads, kv_heads, d)
            h = h + y
            x = _norm64(h, p["post_attention_layernorm.weight"], eps)
            m = F.silu(x @ p["mlp.gate_proj.weight"].T) * (x @ p["mlp.up_proj.weight"].T)
            return h + m @ p["mlp.down_proj.weight"].T, gk.transpose(1, 2), gv.transpose(1, 2)
        # layer_decode: the new token behind the cached ones; the ring's slot p % 129 takes position p
        p, h, cache = _params64(layer), s["h"].double(), s["cache"]
        q, k, v, gq, gk, gv, gate = _inputs64(p, h, cos, sin, heads, kv_heads, d)
        sel = _gated(s["h"], layer.gate_proj.weight, layer.gate_thres)
        slot, ring = t % 129, min(t + 1, 129)
        out = []
        for i in range(b):
            parts = []
            for qq, kk, vv, kc, vc, at, n in ((q, k, v, cache.local_k[0], cache.local_v[0], slot, ring),
                                              (gq, gk, gv, cache.global_k[0], cache.global_v[0], t, t + 1)):
                kc, vc = kc[i, :, :n].double(), vc[i, :, :n].double()
                kc[:, at], vc[:, at] = kk[i, 0], vv[i, 0]
                g = heads // kv_heads
                kc, vc = kc.repeat_interleave(g, 0), vc.repeat_interleave(g, 0)
                w = torch.softmax((kc * qq[i, 0][:, None]).sum(-1) * d ** -0.5, -1)
                parts.append((w[..., None] * vc).sum(1))
            out.append(torch.stack(parts))
        both = torch.stack(out, 1)[:, :, None]  # [2, B, 1, H, D]
        glob = both[1] * sel[..., None, None]
        y = _fuse64(p, both[0], glob, gate, sel, eps)
        return y @ p["o_proj.weight"].T, gk[:, 0], gv[:, 0]
