"""The work that users of this package have it do, as cases that can be timed and compared.

Every case is one call, or one short session of calls, through the public entry points at
DeepSeek-V2-Lite's sizes (hidden 2048, 64 routed experts top-6 of intermediate 1408, 2 shared,
16 heads of 128 + 64, latent 512), with seeded random weights N(0, 0.02) and activations N(0, 1):

  moe         moe_layer_forward: the fused MoE layer on T tokens, prepacked tiled weights
  moe_ops     route_dispatch_combine: the seven ops of the reference module one by one, on the
              reference's row-major weights
  projection  mla_projections: the MLA projection block (q, kv_a, latent norm, kv_b, RoPE)
  attention   mla_forward: the full-sequence MLA module, causal or with an additive mask
  layer       decoder_layer_forward: the whole decoder layer
  session     mla_decode_forward on a LatentKVCache: a prompt, then generated tokens one by one
"""
from __future__ import annotations

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "deepseek-v2-lite-cuda_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

HIDDEN, EXPERTS, TOP_K, INTER, SHARED = 2048, 64, 6, 1408, 2
HEADS, NOPE, ROPE, VDIM, LORA = 16, 128, 64, 128, 512
EPS = 1e-6


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # one sequence decoding: the smallest call, bound by latency and launches
        {"name": "moe T=1", "kind": "moe", "T": 1, "skew": False},
        # a small decode batch behind a skewed router, as trained routers are
        {"name": "moe T=16 skewed", "kind": "moe", "T": 16, "skew": True},
        # a larger decode batch of an odd number of sequences
        {"name": "moe T=61 skewed", "kind": "moe", "T": 61, "skew": True},
        # a large decode batch or a short prompt: every expert has a few rows
        {"name": "moe T=250", "kind": "moe", "T": 250, "skew": False},
        # a chunk of a chunked prefill
        {"name": "moe T=1000", "kind": "moe", "T": 1000, "skew": False},
        # the prefill of the headline benchmark
        {"name": "moe T=4096", "kind": "moe", "T": 4096, "skew": False},
        # a program that calls the reference module's ops one by one
        {"name": "moe ops T=600", "kind": "moe_ops", "T": 600},
        # the projection block at the benchmark's size
        {"name": "projection 8x2048", "kind": "projection", "b": 8, "s": 2048},
        # two prompts of a length that is no multiple of anything
        {"name": "attention 2x1111", "kind": "attention", "b": 2, "s": 1111, "mask": False},
        # the whole layer at the benchmark's size: the largest call
        {"name": "layer 4x2048", "kind": "layer", "b": 4, "s": 2048},
        # one user: a prompt, then tokens one by one against the growing cache
        {"name": "session 1x2000+16", "kind": "session", "b": 1, "prompt": 2000, "steps": 16},
        # a batch of users, an odd prompt length
        {"name": "session 16x333+8", "kind": "session", "b": 16, "prompt": 333, "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "moe_ops", "projection", "attention", "attention",
                       "layer", "session", "session"])
    if kind == "moe":
        return {"kind": kind, "T": _log_int(rng, 1, 4096), "skew": rng.random() < 0.5}
    if kind == "moe_ops":
        return {"kind": kind, "T": _log_int(rng, 16, 1000)}
    if kind == "projection":
        s = _log_int(rng, 16, 4096)
        return {"kind": kind, "b": rng.randint(1, max(1, min(8, 16384 // s))), "s": s}
    if kind == "attention":
        s = _log_int(rng, 64, 3000)
        return {"kind": kind, "b": rng.randint(1, max(1, min(8, 6000 // s))), "s": s,
                "mask": rng.random() < 0.3}
    if kind == "layer":
        s = _log_int(rng, 64, 2048)
        return {"kind": kind, "b": rng.randint(1, max(1, min(8, 6000 // s))), "s": s}
    prompt = _log_int(rng, 1, 3000)
    return {"kind": kind, "b": rng.randint(1, max(1, min(32, 6000 // prompt))), "prompt": prompt,
            "steps": rng.randint(2, 16)}


# ----------------------------------------------------------------- inputs --
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000 + int(seed))


def _randn(g, *shape, std=1.0, dtype=torch.bfloat16):
    t = torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)
    return t.mul_(std).to(dtype)


def _moe_inputs(g, T, shared, skew):
    """bf16 router weight, per-expert stacks, shared expert, tokens and router bias."""
    w = {"wg": _randn(g, EXPERTS, HIDDEN, std=0.02),
         "w1": _randn(g, EXPERTS + shared, 2 * INTER, HIDDEN, std=0.02),
         "w2": _randn(g, EXPERTS + shared, HIDDEN, INTER, std=0.02),
         "x": _randn(g, T, HIDDEN), "bias": None}
    if skew:  # a Zipf-like popularity of the experts
        w["bias"] = torch.tensor([-2.2 * math.log(e + 1) for e in range(EXPERTS)],
                                 dtype=torch.float32, device="cuda")
    return w


def _mla_inputs(g):
    """The projection weights; the latent norm's weight is near one, as trained norms are."""
    return {"q": _randn(g, HEADS * (NOPE + ROPE), HIDDEN, std=0.02),
            "kva": _randn(g, LORA + ROPE, HIDDEN, std=0.02),
            "kva_norm": 1.0 + 0.1 * _randn(g, LORA, dtype=torch.float32),
            "kvb": _randn(g, HEADS * (NOPE + VDIM), LORA, std=0.02),
            "o": _randn(g, HIDDEN, HEADS * VDIM, std=0.02)}


def _tables(n):
    from ds_kernels.mla import yarn_cos_sin
    cos, sin = yarn_cos_sin(n)
    return cos.to(torch.bfloat16).cuda(), sin.to(torch.bfloat16).cuda()


def _key_lengths(b, s):
    """Prompt lengths of a right-padded batch."""
    return [s - (i * s) // (3 * b) for i in range(b)]


def _additive_mask(b, s):
    """[b, 1, s, s] bf16: causal, and the padding keys of every prompt masked."""
    keys = torch.arange(s, device="cuda")
    seen = (keys[None, :] <= keys[:, None])[None].expand(b, s, s).clone()
    for i, n in enumerate(_key_lengths(b, s)):
        seen[i, :, n:] = False
    mask = torch.zeros(b, 1, s, s, dtype=torch.bfloat16, device="cuda")
    return mask.masked_fill_(~seen[:, None], float("-inf"))


def _inputs(case, seed):
    """Everything that is drawn from the seed, in the model's own layout."""
    g, kind = _gen(seed), case["kind"]
    if kind == "moe":
        return _moe_inputs(g, case["T"], SHARED, case["skew"])
    if kind == "moe_ops":
        return _moe_inputs(g, case["T"], 0, False)
    if kind == "session":
        w = _mla_inputs(g)
        w["prompt"] = _randn(g, case["b"], case["prompt"], HIDDEN)
        w["tokens"] = [_randn(g, case["b"], 1, HIDDEN) for _ in range(case["steps"])]
        return w
    w = _mla_inputs(g)
    w["x"] = _randn(g, case["b"], case["s"], HIDDEN)
    if kind == "layer":
        w["in_norm"] = 1.0 + 0.1 * _randn(g, HIDDEN, dtype=torch.float32)
        w["post_norm"] = 1.0 + 0.1 * _randn(g, HIDDEN, dtype=torch.float32)
        w["moe"] = _moe_inputs(g, 1, SHARED, False)
    return w


def prepare(case, seed):
    import ds_kernels as dsk
    from ds_kernels import mla as dm
    kind, w = case["kind"], _inputs(case, seed)
    state = {"kind": kind}
    if kind == "moe":
        state.update(x=w["x"], gate=dsk.tile_weights(w["wg"][None])[0],
                     w1=dsk.tile_weights(w["w1"]), w2=dsk.tile_weights(w["w2"]), bias=w["bias"])
        return state
    if kind == "moe_ops":
        state.update(x=w["x"], gate=w["wg"], w1=w["w1"], w2=w["w2"])
        return state
    mla = dm.MLAWeights.from_tensors(w, torch.device("cuda"))
    if kind == "session":
        n = case["prompt"] + case["steps"]
        cos, sin = _tables(n)
        state.update(W=mla, A=dsk.AbsorbedMLAWeights.from_mla(mla), cos=cos, sin=sin,
                     cache=dsk.LatentKVCache.for_inference(case["b"], max_seq=n),
                     prompt=w["prompt"], tokens=w["tokens"])
        return state
    cos, sin = _tables(case["s"])
    state.update(W=mla, x=w["x"], cos=cos, sin=sin)
    if kind == "attention":
        state["mask"] = _additive_mask(case["b"], case["s"]) if case["mask"] else None
    if kind == "layer":
        m = w["moe"]
        state["P"] = dm.DecoderLayerWeights(
            mla=mla, in_norm=w["in_norm"], post_norm=w["post_norm"],
            gate=dsk.tile_weights(m["wg"][None])[0], w1=dsk.tile_weights(m["w1"]),
            w2=dsk.tile_weights(m["w2"]), n_shared_groups=SHARED)
    return state


def run(state):
    import ds_kernels as dsk
    from ds_kernels import mla as dm
    kind = state["kind"]
    if kind == "moe":
        return dsk.moe_layer_forward(state["x"], state["gate"], state["w1"], state["w2"], TOP_K,
                                     SHARED, gate_bias=state["bias"])
    if kind == "moe_ops":
        return dsk.route_dispatch_combine(state["x"], state["gate"], state["w1"], state["w2"],
                                          TOP_K)
    if kind == "projection":
        q_nope, q_rot, k_nope, v, k_rot, _ = dm.mla_projections(
            state["x"], state["W"], state["cos"], state["sin"], with_latent=False)
        return {"q_nope": q_nope, "q_rot": q_rot, "k_nope": k_nope, "v": v, "k_rot": k_rot}
    if kind == "attention":
        return dm.mla_forward(state["x"], state["W"], state["cos"], state["sin"],
                              attention_mask=state["mask"])
    if kind == "layer":
        return dm.decoder_layer_forward(state["x"], state["P"], state["cos"], state["sin"])
    cache = state["cache"]
    cache.reset()
    out = [dsk.mla_decode_forward(state["prompt"], state["W"], cache, state["cos"], state["sin"],
                                  state["A"])]
    for x in state["tokens"]:
        out.append(dsk.mla_decode_forward(x, state["W"], cache, state["cos"], state["sin"],
                                          state["A"]))
    return out


# ------------------------------------------------------------------- work --
def _moe_work(T, shared, skew=False):
    """Weights of the experts that T tokens are expected to reach, tokens in and out; 2 flops
    per weight element and row."""
    if skew:  # how often each expert is chosen under the router bias
        logits = torch.randn(4096, EXPERTS, generator=torch.Generator().manual_seed(0)) * 0.9
        logits -= 2.2 * torch.log(torch.arange(1.0, EXPERTS + 1))
        chosen = torch.topk(logits, TOP_K).indices.flatten()
        freq = torch.bincount(chosen, minlength=EXPERTS).double() / len(logits)
        reached = float((1.0 - (1.0 - freq) ** T).sum())
    else:
        reached = EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** T)
    per = 3 * INTER * HIDDEN
    rows = T * (TOP_K + shared)
    return (2.0 * ((reached + shared) * per + EXPERTS * HIDDEN) + 4.0 * T * HIDDEN,
            2.0 * rows * per + 2.0 * T * EXPERTS * HIDDEN)


_PROJ_IN = (HEADS * (NOPE + ROPE) + LORA + ROPE) * HIDDEN     # q and kv_a weights
_KVB = HEADS * (NOPE + VDIM) * LORA
_O = HIDDEN * HEADS * VDIM


def work(case):
    kind = case["kind"]
    if kind in ("moe", "moe_ops"):
        nbytes, flops = _moe_work(case["T"], SHARED if kind == "moe" else 0,
                                  case.get("skew", False))
        return {"bytes": nbytes, "flops": flops}
    if kind == "session":
        b, p, n = case["b"], case["prompt"], case["steps"]
        tok = b * (p + n)
        keys = b * (p * (p + 1) / 2 + sum(p + i + 1 for i in range(n)))
        # the prompt through all projections; per generated token the projections, the
        # absorbed up-projections and the cached rows
        flops = 2.0 * tok * (_PROJ_IN + _KVB + _O) + 2.0 * HEADS * keys * (NOPE + ROPE + VDIM)
        weights = 2.0 * (_PROJ_IN + _KVB + _O)
        cached = 2.0 * (LORA + ROPE) * b * sum(p + i + 1 for i in range(n))
        return {"bytes": weights * (1 + n) + cached + 4.0 * tok * HIDDEN
                + 2.0 * b * p * (LORA + ROPE), "flops": flops}
    b, s = case["b"], case["s"]
    rows = b * s
    if kind == "projection":
        out = HEADS * (NOPE + ROPE) + HEADS * (NOPE + VDIM) + ROPE
        return {"bytes": 2.0 * (_PROJ_IN + _KVB) + 2.0 * rows * (HIDDEN + out),
                "flops": 2.0 * rows * (_PROJ_IN + _KVB)}
    flops = 2.0 * rows * (_PROJ_IN + _KVB + _O) + b * s * (s + 1.0) * HEADS * (NOPE + ROPE + VDIM)
    nbytes = 2.0 * (_PROJ_IN + _KVB + _O) + 4.0 * rows * HIDDEN
    if kind == "attention":
        return {"bytes": nbytes + (2.0 * b * s * s if case["mask"] else 0.0), "flops": flops}
    mb, mf = _moe_work(rows, SHARED)
    return {"bytes": nbytes + mb - 4.0 * rows * HIDDEN, "flops": flops + mf}


def tolerance(case):
    """bf16 results of bf16 inputs. About four times the measured distance of the outputs from
    the same in 64 bits, which is set by the roundings of the bf16 intermediates."""
    return {"rel": {"moe": 0.012, "moe_ops": 0.016, "projection": 0.012, "attention": 0.022,
                    "layer": 0.016, "session": 0.022}[case["kind"]]}


# ------------------------------------------------------------------ exact --
def _exact_moe(x, wg, w1, w2, shared, bias=None):
    x = x.double()
    logits = x @ wg.double().t()
    if bias is not None:
        logits = logits + bias.double()
    p = torch.softmax(logits, dim=-1)
    top_w, top_i = torch.topk(p, TOP_K, dim=-1)
    out = torch.zeros_like(x)

    def expert(e, rows):
        h = rows @ w1[e].double().t()
        gate, up = h[:, :INTER], h[:, INTER:]
        return (gate * torch.sigmoid(gate) * up) @ w2[e].double().t()

    for e in range(EXPERTS):
        t, k = (top_i == e).nonzero(as_tuple=True)
        if t.numel():
            out.index_add_(0, t, top_w[t, k, None] * expert(e, x[t]))
    for j in range(shared):
        out += expert(EXPERTS + j, x)
    return out


def _exact_rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _exact_rope(x, cos, sin):
    """x [..., s, ROPE] of interleaved pairs -> halves, rotated by the rows of the tables."""
    a, b = x[..., 0::2], x[..., 1::2]
    x = torch.cat([a, b], dim=-1)
    turned = torch.cat([-b, a], dim=-1)
    return x * cos.double() + turned * sin.double()


def _exact_qkv(x, w, s):
    """Per head in 64 bits: q_nope, q_rot, k_nope, v [b, h, s, .] and k_rot [b, 1, s, .]."""
    cos, sin = _tables(s)
    b = x.shape[0]
    x = x.double()
    q = (x @ w["q"].double().t()).view(b, s, HEADS, NOPE + ROPE).transpose(1, 2)
    kva = x @ w["kva"].double().t()
    kv = (_exact_rms(kva[..., :LORA], w["kva_norm"]) @ w["kvb"].double().t())
    kv = kv.view(b, s, HEADS, NOPE + VDIM).transpose(1, 2)
    return (q[..., :NOPE], _exact_rope(q[..., NOPE:], cos, sin), kv[..., :NOPE], kv[..., NOPE:],
            _exact_rope(kva[:, None, :, LORA:], cos, sin))


def _softmax_scale():
    m = 0.1 * 0.707 * math.log(40.0) + 1.0
    return (NOPE + ROPE) ** -0.5 * m * m


def _exact_mla(x, w, mask=None):
    b, s, _ = x.shape
    q_nope, q_rot, k_nope, v, k_rot = _exact_qkv(x, w, s)
    if mask is None:
        mask = torch.full((s, s), float("-inf"), device="cuda", dtype=torch.float64).triu_(1)
        mask = mask.expand(b, 1, s, s)
    out = torch.empty(b, s, HEADS * VDIM, dtype=torch.float64, device="cuda")
    for i in range(b):
        for h in range(HEADS):
            sc = q_nope[i, h] @ k_nope[i, h].t() + q_rot[i, h] @ k_rot[i, 0].t()
            p = torch.softmax(sc * _softmax_scale() + mask[i, 0].double(), dim=-1)
            out[i, :, h * VDIM:(h + 1) * VDIM] = p @ v[i, h]
    return out @ w["o"].double().t()


def exact(case, seed):
    kind, w = case["kind"], _inputs(case, seed)
    if kind == "moe":
        return _exact_moe(w["x"], w["wg"], w["w1"], w["w2"], SHARED, w["bias"])
    if kind == "moe_ops":
        return _exact_moe(w["x"], w["wg"], w["w1"], w["w2"], 0)
    if kind == "projection":
        names = ("q_nope", "q_rot", "k_nope", "v", "k_rot")
        return dict(zip(names, _exact_qkv(w["x"], w, case["s"])))
    if kind == "attention":
        mask = _additive_mask(case["b"], case["s"]) if case["mask"] else None
        return _exact_mla(w["x"], w, mask)
    if kind == "layer":
        m, x = w["moe"], w["x"].double()
        x = x + _exact_mla(_exact_rms(x, w["in_norm"]), w)
        h = _exact_rms(x, w["post_norm"]).view(-1, HIDDEN)
        return x + _exact_moe(h, m["wg"], m["w1"], m["w2"], SHARED).view(x.shape)
    y = _exact_mla(torch.cat([w["prompt"]] + w["tokens"], dim=1), w)
    p = case["prompt"]
    return [y[:, :p]] + [y[:, p + i:p + i + 1] for i in range(case["steps"])]
