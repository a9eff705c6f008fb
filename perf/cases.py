"""The calls whose speed counts: the attention sublayer and the transformer stack, as a
user's program makes them.

A case is a dict of plain values:

``kind``      ``"layer"``: one ``CobraAttentionSublayer`` forward; ``"stack"``: one
              ``CobraTransformer`` forward
``batch``, ``seq_len``, ``d_model``, ``heads``
``ffn_dim``, ``layers``  the stack's (0 for a layer)
``dtype``     of activations and parameters: ``"float16"``, ``"bfloat16"``, ``"float32"``
``causal``    whether a token sees only itself and the tokens before it
``padding``   0.0: no token mask; p > 0: a ``valid_token_mask`` whose sequences hold
              between (1 - p) S and S tokens, the rest padding at the end
``residual``  the layer is asked for its residual too (``return_residual=True``)
``sharp``     factor on the query and key weights: at 1.0 (``nn.Linear``'s own range) a
              logit's standard deviation is about 1/3, at 2.0 about 4/3, at 3.0 about 3,
              which is where trained attention lies

Weights are drawn as ``nn.Linear`` draws them, LayerNorm weights around 1 and biases
around 0 as in a trained model, and inputs from N(0, 1).
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "cobra-gpu-kernel_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

_DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}


def _case(kind, batch, seq_len, d_model, heads, *, ffn_dim=0, layers=0, dtype="float16", causal=False, padding=0.0,
          residual=False, sharp=1.0):
    return {"kind": kind, "batch": batch, "seq_len": seq_len, "d_model": d_model, "heads": heads, "ffn_dim": ffn_dim,
            "layers": layers, "dtype": dtype, "causal": causal, "padding": padding, "residual": residual,
            "sharp": sharp}


def listed():
    cases = {
        # One short sequence: a request on its own, where the launch and the chain of
        # steps inside the kernel are all there is.
        "layer_b1": _case("layer", 1, 128, 128, 4),
        # The benchmark's own workload: a batch of short sequences that covers the chip once.
        "layer_b64": _case("layer", 64, 128, 128, 4),
        # Offline scoring of many short sequences in one call.
        "layer_b10000": _case("layer", 10000, 128, 128, 4),
        # The benchmark's long-context configuration of the narrow model.
        "layer_s1024": _case("layer", 64, 1024, 128, 4),
        # The benchmark's wide configuration, bound by its projections.
        "layer_d1024": _case("layer", 64, 128, 1024, 4),
        # A ragged, padded batch through a causal layer of middle width: what a server
        # with real requests has, odd sizes and a mask.
        "layer_ragged_d512": _case("layer", 37, 333, 512, 8, causal=True, padding=0.5, sharp=2.0),
        # A bf16 decoder layer on a few sequences of ordinary length (prefill).
        "layer_bf16_s2048": _case("layer", 8, 2048, 1024, 16, dtype="bfloat16", causal=True, sharp=2.0),
        # fp32 activations, with the residual handed on to a caller's own feed-forward part.
        "layer_fp32_d256": _case("layer", 64, 128, 256, 8, dtype="float32", residual=True),
        # A width and a head size that are not multiples of 8.
        "layer_odd_d210": _case("layer", 24, 77, 210, 6),
        # One sequence of the benchmark's longest configuration.
        "layer_s100000": _case("layer", 1, 100000, 1024, 16),
        # The whole model, wide: four causal blocks with their feed-forward parts.
        "stack_d1024": _case("stack", 64, 128, 1024, 4, ffn_dim=1024, layers=4, causal=True),
        # The whole model, narrow and long, on a padded batch.
        "stack_s1024": _case("stack", 64, 1024, 128, 4, ffn_dim=128, layers=4, causal=True, padding=0.3, sharp=2.0),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, seq_len, d_model, tokens, most=10000):
    """A batch of 1 up to what ``tokens`` tokens of width 128 hold, over its logarithm."""
    top = max(1, min(most, tokens * 128 // (seq_len * max(128, d_model))))
    return min(top, max(1, _log(rng, 1, top + 0.49)))


def draw(rng):
    """One more case of the same ranges.  The largest of each family stays below the listed
    largest (its tokens x width below layer_b10000's, its operations below layer_s100000's)."""
    family = rng.choice(["short", "short", "long_narrow", "wide", "wide", "odd", "stack", "longest"])
    opt = {"causal": rng.random() < 0.5, "sharp": round(rng.uniform(1.0, 3.0), 2),
           "dtype": rng.choice(["float16", "float16", "bfloat16", "float32"]),
           "padding": rng.choice([0.0, 0.0, round(rng.uniform(0.1, 0.9), 2)])}
    if family == "short":
        d, h = rng.choice([(128, 4), (128, 4), (128, 2), (128, 1), (128, 16), (64, 2), (64, 1)])
        s = _log(rng, 1, 128)
        return _case("layer", _batch(rng, s, d, 1_200_000), s, d, h, residual=rng.random() < 0.2, **opt)
    if family == "long_narrow":
        d, h = rng.choice([(128, 4), (128, 2), (128, 16), (64, 2)])
        s = _log(rng, 129, 4096)
        return _case("layer", _batch(rng, s, d, 131072, 256), s, d, h, residual=rng.random() < 0.2, **opt)
    if family == "wide":
        d = rng.choice([256, 512, 768, 1024, 2048])
        hd = rng.choice([32, 64, 128, 256])
        # Heads of 256 go with short sequences, as in the benchmark's wide configuration.
        h, s = d // hd, _log(rng, 16, 128 if hd == 256 else 4096)
        return _case("layer", _batch(rng, s, d, 262144, 1024), s, d, h, residual=rng.random() < 0.2, **opt)
    if family == "odd":
        d, h = rng.choice([(96, 8), (100, 4), (36, 3), (210, 6), (300, 5)])
        s = _log(rng, 5, 600)
        return _case("layer", _batch(rng, s, d, 65536, 256), s, d, h, **opt)
    if family == "stack":
        d = rng.choice([64, 128, 256, 512, 1024])
        h = d // rng.choice([32, 64])
        s = _log(rng, 16, 1024)
        return _case("stack", _batch(rng, s, d, 131072, 256), s, d, h, ffn_dim=d * rng.choice([1, 1, 4]),
                     layers=rng.randint(2, 4), **opt)
    d = rng.choice([512, 1024])
    return _case("layer", 1, _log(rng, 8192, 80000), d, d // rng.choice([64, 128]), **opt)


# -- inputs -------------------------------------------------------------------------


def _block_names(case):
    """Prefix of each block's parameters."""
    return [""] if case["kind"] == "layer" else [f"layers.{i}." for i in range(case["layers"])]


def _weights(case, g, dev):
    """The state_dict of the case's module, in its dtype, on ``dev``."""
    d, f, dt = case["d_model"], case["ffn_dim"], _DTYPES[case["dtype"]]
    out = {}

    def linear(name, n, k, gain=1.0):
        bound = 1.0 / math.sqrt(k)
        w = (torch.rand(n, k, generator=g, device=dev) * 2 - 1) * bound
        b = (torch.rand(n, generator=g, device=dev) * 2 - 1) * bound
        out[name + ".weight"] = (w * gain).to(dt)
        out[name + ".bias"] = b.to(dt)

    def norm(name):
        out[name + ".weight"] = (1 + 0.1 * torch.randn(d, generator=g, device=dev)).to(dt)
        out[name + ".bias"] = (0.1 * torch.randn(d, generator=g, device=dev)).to(dt)

    for p in _block_names(case):
        norm(p + "norm1")
        for name in ("q_proj", "k_proj"):
            linear(p + "attention." + name, d, d, case["sharp"])
        for name in ("v_proj", "out_proj"):
            linear(p + "attention." + name, d, d)
        norm(p + "norm2")
        if case["kind"] == "stack":
            linear(p + "ffn_in", f, d)
            linear(p + "ffn_out", d, f)
    if case["kind"] == "stack":
        norm("final_norm")
    return out


def _inputs(case, seed, dev):
    """(state_dict, x, mask or None) of a seed."""
    g = torch.Generator(device=dev).manual_seed(seed)
    sd = _weights(case, g, dev)
    b, s, d = case["batch"], case["seq_len"], case["d_model"]
    x = torch.randn(b, s, d, generator=g, device=dev).to(_DTYPES[case["dtype"]])
    mask = None
    if case["padding"] > 0:
        low = max(1, round(s * (1 - case["padding"])))
        length = torch.randint(low, s + 1, (b, 1), generator=g, device=dev)
        mask = torch.arange(s, device=dev)[None, :] < length
    return sd, x, mask


def prepare(case, seed):
    from cobra_amd import CobraAttentionSublayer, CobraTransformer, TransformerConfig

    dev = torch.device("cuda", 0)
    sd, x, mask = _inputs(case, seed, dev)
    if case["kind"] == "layer":
        m = CobraAttentionSublayer(case["d_model"], case["heads"], causal=case["causal"])
    else:
        m = CobraTransformer(TransformerConfig(case["batch"], case["seq_len"], case["d_model"], case["heads"],
                                               case["ffn_dim"], case["layers"], case["causal"]))
    m = m.to(device=dev, dtype=_DTYPES[case["dtype"]]).eval()
    m.load_state_dict(sd, strict=True)
    return {"module": m, "x": x, "mask": mask, "residual": case["residual"]}


def run(state):
    with torch.inference_mode():
        if state["residual"]:
            return state["module"](state["x"], state["mask"], return_residual=True)
        return state["module"](state["x"], state["mask"])


# -- what a pass cannot do without -----------------------------------------------------


def work(case):
    b, s, d, f = case["batch"], case["seq_len"], case["d_model"], case["ffn_dim"]
    t, n = b * s, max(1, case["layers"])
    io = 4 if case["dtype"] == "float32" else 2
    pairs = b * (s * (s + 1) // 2 if case["causal"] else s * s)
    flops = n * (8 * t * d * d + 4 * pairs * d + 4 * t * d * f)
    weights = n * (4 * d * d + 2 * d * f + 9 * d + f) * io
    return {"bytes": 2 * t * d * io + weights + (4 * t * d if case["residual"] else 0) +
            (t if case["padding"] > 0 else 0), "flops": flops}


# -- the exact result ------------------------------------------------------------------


def _attention(q, k, v, causal, mask):
    """softmax(q k^T / sqrt(hd)) v for [B, H, S, hd] in 64 bits, a block of queries of some
    sequences at a time."""
    b, h, s, hd = q.shape
    out = torch.empty_like(q)
    step_b = max(1, (1 << 28) // (h * s * min(s, 2048)))
    for b0 in range(0, b, step_b):
        b1 = min(b, b0 + step_b)
        heads = [slice(0, h)] if h * s * min(s, 2048) <= 1 << 28 else [slice(i, i + 1) for i in range(h)]
        for hs in heads:
            for q0 in range(0, s, 2048):
                q1 = min(s, q0 + 2048)
                end = q1 if causal else s
                kt = k[b0:b1, hs, :end].transpose(-1, -2).contiguous()
                p = torch.matmul(q[b0:b1, hs, q0:q1] * hd ** -0.5, kt)
                if causal:
                    at = torch.arange(s, device=q.device)
                    p.masked_fill_(at[None, :end] > at[q0:q1, None], float("-inf"))
                if mask is not None:
                    p.masked_fill_(~mask[b0:b1, None, None, :end], float("-inf"))
                p.sub_(p.amax(-1, keepdim=True)).exp_()
                out[b0:b1, hs, q0:q1] = torch.matmul(p, v[b0:b1, hs, :end].contiguous()) / p.sum(-1, keepdim=True)
    return out


def _block(case, sd, p, x, mask):
    """(residual after the attention half, and after the whole block)."""
    b, s, d = x.shape
    h = case["heads"]

    def linear(name, a):
        return torch.addmm(sd[p + name + ".bias"], a.reshape(b * s, -1), sd[p + name + ".weight"].t()).view(b, s, -1)

    def norm(name, a):
        return F.layer_norm(a, (d,), sd[p + name + ".weight"], sd[p + name + ".bias"], 1e-5)

    n = norm("norm1", x)
    q, k, v = (linear("attention." + w, n).view(b, s, h, d // h).transpose(1, 2).contiguous()
               for w in ("q_proj", "k_proj", "v_proj"))
    del n
    ctx = _attention(q, k, v, case["causal"], mask).transpose(1, 2).reshape(b, s, d)
    del q, k, v
    branch = linear("attention.out_proj", ctx)
    if mask is not None:
        branch.masked_fill_(~mask[..., None], 0.0)
    r = x + branch
    if case["kind"] == "layer":
        return r, norm("norm2", r)
    out = r + linear("ffn_out", F.gelu(linear("ffn_in", norm("norm2", r))))
    if mask is not None:
        out.masked_fill_(~mask[..., None], 0.0)
    return r, out


def exact(case, seed):
    dev = torch.device("cuda", 0)
    with torch.inference_mode():
        sd, x, mask = _inputs(case, seed, dev)
        sd = {n: w.double() for n, w in sd.items()}
        outs = []
        # Sequences are independent, so many short ones go through in parts.
        step = max(1, (1 << 27) // (case["seq_len"] * case["d_model"]))
        for b0 in range(0, case["batch"], step):
            xd = x[b0:b0 + step].double()
            md = None if mask is None else mask[b0:b0 + step]
            if case["kind"] == "layer":
                r, y = _block(case, sd, "", xd, md)
                outs.append((r, y) if case["residual"] else (y,))
                continue
            for p in _block_names(case):
                _, xd = _block(case, sd, p, xd, md)
            y = F.layer_norm(xd, (case["d_model"],), sd["final_norm.weight"], sd["final_norm.bias"], 1e-5)
            if md is not None:
                y.masked_fill_(~md[..., None], 0.0)
            outs.append((y,))
        whole = tuple(torch.cat(parts) for parts in zip(*outs))
        return whole if case["residual"] else whole[0]


def tolerance(case):
    """About four times the distance from ``exact`` measured over the listed cases and some
    ninety drawn ones.  16-bit outputs: 2.1e-4 (fp16) and 1.66e-3 (bf16) are the rounding of
    the output alone; at ``sharp`` 3 the rounding of q, k and the probabilities brings a layer
    to 2.5e-4 and 2.3e-3 and a stack to 4.3e-4.  float32 activations use fp16 matrix operands:
    1.1e-5 (``sharp`` 1) to 2.1e-4.  Largest elements: 2.1e-3, bf16 1.3e-2."""
    if case["dtype"] == "bfloat16":
        return {"rel": 8e-3 if case["kind"] == "layer" else 1.2e-2, "max": 6e-2}
    return {"rel": 1e-3 if case["kind"] == "layer" else 1.6e-3, "max": 8e-3}
