"""The work this framework is measured on, through its public entry points.

A target model is served in two phases, and both are here, layer by layer and as whole calls:

* decode / speculative verify: 1..16 rows per call (``[anchor] + draft``) against a KV cache of
  hundreds to 32k positions: quantized projections, MLPs, attention over plain and quantized
  caches, the routed-expert block, ``Target.verify``;
* prefill: a prompt of tens to 2048 rows per chunk through the same layers:
  ``QuantizedLinear`` under the prefill scope, causal attention, the routed-expert block,
  ``Target.prefill``.

Sizes are those of the repository's benchmark and tests (hidden 4096 / intermediate 12288 with
32/8 x 128 heads, hidden 5120 / 25600 with 64/8 x 128, 5120 x 17408 and 24/4 x 256, 128 experts
top-8 of 2048 / 768) and generic ones between them.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlx-dspark_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dspark_rocm import fast, ops, quant, skinny_qmm, wide_gemm  # noqa: E402
from dspark_rocm.model import DenseModel, ModelArgs, Target  # noqa: E402
from dspark_rocm.nn import QuantizedLinear  # noqa: E402

DEV = "cuda"
GROUP = 64


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # one projection of a decode step, one row, as a caller holding mlx-format arrays makes it
        dict(name="linear_decode", kind="linear", packed=False, bits=8, m=1, n=4096, k=4096),
        # the MLP of a 4-bit target at an odd verify width, weights packed at load
        dict(name="mlp_verify_4bit", kind="mlp", bits=4, m=11, hidden=5120, inter=17408),
        # verify attention at a long context
        dict(name="attn_verify_32k", kind="attn", hq=32, hk=8, d=128, m=16, keys=32784, kv_bits=16, dtype="bf16"),
        # the same call over an 8-bit cache, head dim 256, ragged length, a 6-row block
        dict(name="attn_verify_kv8", kind="attn", hq=24, hk=4, d=256, m=6, keys=10007, kv_bits=8, dtype="bf16"),
        # the routed experts of one block in a verify step
        dict(name="moe_verify", kind="moe", bits=4, m=16, experts=128, top_k=8, hidden=2048, inter=768),
        # the same block over a prompt chunk
        dict(name="moe_prefill", kind="moe", bits=4, m=500, experts=128, top_k=8, hidden=2048, inter=768),
        # one projection over a short prompt: more rows than a verify block, fewer than a chunk
        dict(name="linear_prompt", kind="prompt", bits=4, m=93, n=17408, k=5120, bias=False),
        # one projection over a full prefill chunk
        dict(name="linear_prefill", kind="prompt", bits=8, m=2048, n=12288, k=4096, bias=False),
        # causal attention of a prefill chunk behind an earlier one
        dict(name="attn_prefill", kind="attn_prefill", hq=32, hk=8, d=128, m=2048, keys=5001, dtype="bf16"),
        # a whole decode step of a small target: launches and host work count
        dict(name="step_small", kind="step", bits=8, m=1, layers=4, hidden=1024, inter=4096, hq=8, hk=2, d=128,
             vocab=8192, context=700, kv_bits=0),
        # a whole verify step of wide layers at a long context
        dict(name="step_verify", kind="step", bits=8, m=16, layers=3, hidden=5120, inter=25600, hq=64, hk=8, d=128,
             vocab=32768, context=16000, kv_bits=0),
        # a whole prompt chunk through a target, logits of its last row
        dict(name="prefill_chunk", kind="prefill", bits=8, m=777, layers=2, hidden=4096, inter=12288, hq=32, hk=8,
             d=128, vocab=32768),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(["linear", "mlp", "attn", "attn", "moe", "moe", "prompt", "prompt", "attn_prefill", "step",
                       "prefill"])
    bits = rng.choice([4, 8])
    if kind == "linear":
        packed = rng.random() < 0.5
        return dict(kind=kind, packed=packed, bits=bits, m=rng.randint(1, 16), n=_log(rng, 256, 16384),
                    k=_log(rng, 512, 16384, 512 if packed else 64))
    if kind == "mlp":
        return dict(kind=kind, bits=bits, m=rng.randint(1, 16), hidden=_log(rng, 1024, 5120, 512),
                    inter=_log(rng, 2048, 25600, 512))
    if kind == "attn":
        hq, hk, d = rng.choice([(32, 8, 128), (64, 8, 128), (24, 4, 256), (16, 8, 256), (8, 2, 64)])
        m = rng.randint(1, 16)
        return dict(kind=kind, hq=hq, hk=hk, d=d, m=m, keys=m + _log(rng, 100, 32768),
                    kv_bits=rng.choice([16, 16, 8, 4]), dtype=rng.choice(["bf16", "bf16", "f16"]))
    if kind == "moe":
        return dict(kind=kind, bits=bits, m=_log(rng, 1, 1000), experts=rng.choice([32, 64, 128]),
                    top_k=rng.choice([4, 8]), hidden=rng.choice([1024, 2048]), inter=128 * rng.randint(3, 8))
    if kind == "prompt":
        return dict(kind=kind, bits=bits, m=_log(rng, 17, 2048), n=_log(rng, 512, 16384), k=_log(rng, 512, 8192, 64),
                    bias=rng.random() < 0.3)
    if kind == "attn_prefill":
        hq, hk, d = rng.choice([(32, 8, 128), (64, 8, 128), (24, 4, 256), (16, 8, 256), (8, 2, 64)])
        m = _log(rng, 17, 2048)
        keys = m + rng.choice([0, _log(rng, 16, 4096)])
        return dict(kind=kind, hq=hq, hk=hk, d=d, m=m, keys=min(keys, 2048 * 5001 * 32 // (m * hq)) if keys > m else m,
                    dtype=rng.choice(["bf16", "bf16", "f16"]))
    hidden = rng.choice([1024, 2048, 4096])
    shape = dict(bits=bits, layers=rng.randint(1, 4), hidden=hidden, inter=hidden * rng.randint(2, 4), hq=hidden // 128,
                 hk=max(1, hidden // 512), d=128, vocab=_log(rng, 4096, 32768, 64))
    if kind == "step":
        return dict(shape, kind=kind, m=rng.randint(1, 16), context=_log(rng, 64, 16384),
                    kv_bits=rng.choice([0, 0, 8, 4]))
    return dict(shape, kind=kind, layers=min(2, shape["layers"]), m=_log(rng, 17, 1024))


# ------------------------------------------------------------------ inputs

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.bfloat16, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


def _quantized(g, n, k, bits, experts=None):
    w, s, b = quant.random_quantized(n * (experts or 1), k, bits, generator=g, device=DEV)
    if experts is None:
        return w, s, b
    return tuple(t.reshape(experts, n, -1) for t in (w, s, b))


def _target(case, seed):
    args = ModelArgs(hidden_size=case["hidden"], num_hidden_layers=case["layers"], intermediate_size=case["inter"],
                     num_attention_heads=case["hq"], num_key_value_heads=case["hk"], head_dim=case["d"],
                     vocab_size=case["vocab"], bits=case["bits"], lm_head_bits=8)
    model = DenseModel.random(args, device=DEV, seed=seed)
    return Target(model, max_rows=16, kv_bits=case.get("kv_bits") or None)


def prepare(case, seed):
    g = _gen(seed)
    kind, m = case["kind"], case["m"]
    st = {"case": case}
    if kind == "linear":
        st["w"] = _quantized(g, case["n"], case["k"], case["bits"])
        st["x"] = _randn(g, m, case["k"])
        if case["packed"]:
            st["packed"] = ops.qmm_pack(*st["w"], bits=case["bits"])
    elif kind == "mlp":
        h, i, bits = case["hidden"], case["inter"], case["bits"]
        st["gate"], st["up"], st["down"] = _quantized(g, i, h, bits), _quantized(g, i, h, bits), _quantized(g, h, i, bits)
        st["pair"] = ops.qmm_pack_swiglu(st["gate"], st["up"], bits=bits)
        st["packed_down"] = ops.qmm_pack(*st["down"], bits=bits)
        st["x"] = _randn(g, m, h)
    elif kind in ("attn", "attn_prefill"):
        hq, hk, d, keys, dt = case["hq"], case["hk"], case["d"], case["keys"], _DTYPES[case["dtype"]]
        cap = (keys + 255) // 256 * 256                    # a cache's buffer, of which keys rows are filled
        k, v = _randn(g, 1, hk, cap, d, dtype=dt), _randn(g, 1, hk, cap, d, dtype=dt)
        if case.get("kv_bits", 16) != 16:
            k, v = (quant.quantize_rows(t, case["kv_bits"], GROUP, dt) for t in (k, v))
            st["k"], st["v"] = (tuple(t[:, :, :keys] for t in x) for x in (k, v))
        else:
            st["k"], st["v"] = k[:, :, :keys], v[:, :, :keys]
        st["q"] = _randn(g, 1, hq, m, d, dtype=dt, scale=2.0)
    elif kind == "moe":
        e, h, i, bits = case["experts"], case["hidden"], case["inter"], case["bits"]
        st["gate"], st["up"], st["down"] = (_quantized(g, n, k, bits, e) for n, k in ((i, h), (i, h), (h, i)))
        st["packed"] = [(ops.moe_pack(w, bits=bits), s, b) for w, s, b in (st["gate"], st["up"], st["down"])]
        st["x"] = _randn(g, m, h)
        st["logits"] = _randn(g, m, e)
    elif kind == "prompt":
        w, s, b = _quantized(g, case["n"], case["k"], case["bits"])
        st["lin"] = QuantizedLinear(w, s, b, _randn(g, case["n"], scale=0.02) if case["bias"] else None,
                                    bits=case["bits"])
        st["x"] = _randn(g, 1, m, case["k"])
    else:
        st["target"] = _target(case, seed)
        context = case.get("context", 0)
        st["cache"] = st["target"].make_cache(context + m)
        for c in st["cache"]:                              # the KV of the positions before this call
            if context:
                kv = [_randn(g, 1, case["hk"], context, case["d"]) for _ in range(2)]
                c.update_and_fetch(*kv)
        st["ids"] = torch.randint(0, case["vocab"], (1, m), generator=g, device=DEV)
    return st


# ------------------------------------------------------------------ one pass


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["packed"]:
            return ops.quantized_matmul_packed(st["x"], st["packed"])
        return skinny_qmm.qmm(st["x"], *st["w"], case["bits"])
    if kind == "mlp":
        return ops.quantized_matmul_packed(ops.quantized_swiglu_packed(st["x"], st["pair"]), st["packed_down"])
    if kind == "attn":
        scale = case["d"] ** -0.5
        if case["kv_bits"] != 16:
            return ops.verify_attention_quantized(st["q"], st["k"], st["v"], scale=scale, causal=True,
                                                  bits=case["kv_bits"])
        return ops.verify_attention(st["q"], st["k"], st["v"], scale=scale, causal=True)
    if kind == "moe":
        out, inds, scores = ops.moe_switch_glu(st["x"], st["logits"], *st["packed"], k=case["top_k"], bits=case["bits"])
        return {"out": out, "experts": inds, "scores": scores}
    if kind == "prompt":
        with torch.no_grad(), wide_gemm.wide_matmul(wide_gemm.SAFE_MIN_ROWS):
            return st["lin"](st["x"])
    if kind == "attn_prefill":
        with torch.no_grad():
            return fast.scaled_dot_product_attention(st["q"], st["k"], st["v"], scale=case["d"] ** -0.5, mask="causal")
    target, cache = st["target"], st["cache"]
    if kind == "step":                                     # a round whose drafts are all rejected
        logits, fused = target.verify(st["ids"], cache, tap=(0, case["layers"] - 1))
        target.rollback(cache, case["m"])
        return {"logits": logits, "fused": fused}
    for c in cache:
        c.trim(c.offset)
    with torch.no_grad(), wide_gemm.wide_matmul(wide_gemm.SAFE_MIN_ROWS):
        logits, fused = target.prefill(st["ids"], cache, tap=(case["layers"] - 1,), want_logits=True)
    return {"logits": logits, "fused": fused, "kv": [t for c in cache for t in c.fetch()]}


# ------------------------------------------------------------------ what a pass cannot do without


def _wbytes(n, k, bits):
    return n * k * bits / 8 + 4 * n * (k // GROUP)


def _seen(m, keys):
    """(query, key) pairs a causal call of m rows at the end of ``keys`` positions computes."""
    return m * (keys - m) + m * (m + 1) // 2


def _layer_work(case, m, keys):
    h, i, hq, hk, d = case["hidden"], case["inter"], case["hq"], case["hk"], case["d"]
    mats = ((hq * d, h), (hk * d, h), (hk * d, h), (h, hq * d), (i, h), (i, h), (h, i))
    kv_row = 2 * hk * ({0: 2 * d, 8: d + 4 * d // GROUP, 4: d / 2 + 4 * d // GROUP}[case.get("kv_bits", 0)])
    return (sum(_wbytes(n, k, case["bits"]) for n, k in mats) + kv_row * keys,
            sum(2.0 * m * n * k for n, k in mats) + 4.0 * hq * d * _seen(m, keys))


def work(case):
    kind, m = case["kind"], case["m"]
    if kind in ("linear", "prompt"):
        n, k = case["n"], case["k"]
        return {"bytes": _wbytes(n, k, case["bits"]) + 2 * m * (n + k), "flops": 2.0 * m * n * k}
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"bytes": 3 * _wbytes(i, h, case["bits"]) + 4 * m * h, "flops": 6.0 * m * h * i}
    if kind in ("attn", "attn_prefill"):
        hq, hk, d, keys = case["hq"], case["hk"], case["d"], case["keys"]
        bits = case.get("kv_bits", 16)
        row = 2 * d if bits == 16 else d * bits / 8 + 4 * (d // GROUP)
        return {"bytes": 2 * hk * keys * row + 4 * hq * m * d, "flops": 4.0 * hq * d * _seen(m, keys)}
    if kind == "moe":
        e, k, h, i = case["experts"], case["top_k"], case["hidden"], case["inter"]
        live = e * (1 - (1 - k / e) ** m)                  # experts that some token selects
        return {"bytes": live * 3 * _wbytes(i, h, case["bits"]) + 4 * m * h + 2 * m * e + 6 * m * k,
                "flops": 6.0 * m * k * h * i}
    keys = case.get("context", 0) + m
    by, fl = _layer_work(case, m, keys)
    rows = m if kind == "step" else 1
    h, vocab = case["hidden"], case["vocab"]
    return {"bytes": case["layers"] * by + _wbytes(vocab, h, 8) + 2 * rows * vocab,
            "flops": case["layers"] * fl + 2.0 * rows * vocab * h}


def tolerance(case):
    return {"linear": {"rel": 4e-3}, "prompt": {"rel": 4e-3}, "mlp": {"rel": 1e-2}, "attn": {"rel": 6e-3},
            "attn_prefill": {"rel": 6e-3}, "moe": {"rel": 1e-2}, "step": {"rel": 2.5e-2, "max": 0.3},
            "prefill": {"rel": 2.5e-2, "max": 0.5}}[case["kind"]]


# ------------------------------------------------------------------ the same in 64 bits


def _deq64(w, s, b, bits):
    f = 32 // bits
    sh = torch.arange(f, device=w.device, dtype=torch.int32) * bits
    q = ((w.unsqueeze(-1) >> sh) & ((1 << bits) - 1)).double()
    q = q.reshape(*w.shape[:-1], -1, GROUP)
    return (q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(*w.shape[:-1], -1)


def _mm64(x, triple, bits):
    return x @ _deq64(*triple, bits).t()


def _silu64(g):
    return g * torch.sigmoid(g)


def _attn64(q, k, v, scale):
    """[Hq, m, D] over [Hk, L, D], causal from the bottom right; one query head at a time."""
    hq, m, _ = q.shape
    hk, L = k.shape[0], k.shape[1]
    seen = torch.arange(L, device=q.device)[None, :] <= (L - m + torch.arange(m, device=q.device))[:, None]
    out = []
    for h in range(hq):
        kk, vv = k[h * hk // hq], v[h * hk // hq]
        s = (q[h] @ kk.t().contiguous() * scale).masked_fill(~seen, float("-inf"))
        out.append(torch.softmax(s, -1) @ vv)
    return torch.stack(out)


def _kv64(kv, bits):
    """[1, Hk, L, D] of a plain or quantized cache's fetched view, in 64 bits."""
    return kv.double()[0] if bits in (0, 16) else _deq64(*(t.contiguous() for t in kv), bits)[0]


def _norm64(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos0, base):
    d = x.shape[-1]
    freq = base ** (-2.0 * torch.arange(d // 2, device=x.device, dtype=torch.float64) / d)
    ang = torch.arange(pos0, pos0 + x.shape[-2], device=x.device, dtype=torch.float64)[:, None] * freq
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1)


def _model64(case, st):
    model, m, bits = st["target"].model, case["m"], case["bits"]
    hq, hk, d, base = case["hq"], case["hk"], case["d"], model.args.rope_theta
    tri = lambda lin: (lin.weight, lin.scales, lin.biases)  # noqa: E731
    pos0 = case.get("context", 0)
    h = model.embed_tokens[st["ids"][0]].double()
    streams, kv = [], []
    for layer, c in zip(model.layers, st["cache"]):
        at, mlp = layer.self_attn, layer.mlp
        x = _norm64(h, layer.input_layernorm)
        heads = lambda lin, n: _mm64(x, tri(lin), bits).reshape(m, n, d).transpose(0, 1)  # noqa: E731
        q = _rope64(_norm64(heads(at.q_proj, hq), at.q_norm), pos0, base)
        k = _rope64(_norm64(heads(at.k_proj, hk), at.k_norm), pos0, base)
        v = heads(at.v_proj, hk)
        kv += [k[None], v[None]]
        if pos0:
            old = [_kv64(t, case["kv_bits"]) for t in c.fetch()]
            k, v = torch.cat([old[0], k], 1), torch.cat([old[1], v], 1)
        a = _attn64(q, k, v, d ** -0.5).transpose(0, 1).reshape(m, hq * d)
        h = h + _mm64(a, tri(at.o_proj), bits)
        x = _norm64(h, layer.post_attention_layernorm)
        x = _silu64(_mm64(x, tri(mlp.gate_proj), bits)) * _mm64(x, tri(mlp.up_proj), bits)
        h = h + _mm64(x, tri(mlp.down_proj), bits)
        streams.append(h)
    last = _norm64(h, model.norm)
    return last, streams, kv, tri(model.lm_head)


def exact(case, seed):
    st = prepare(case, seed)
    kind, bits = case["kind"], case.get("bits")
    if kind == "linear":
        return _mm64(st["x"].double(), st["w"], bits)
    if kind == "prompt":
        lin = st["lin"]
        y = _mm64(st["x"][0].double(), (lin.weight, lin.scales, lin.biases), bits)
        return (y if lin.bias is None else y + lin.bias.double())[None]
    if kind == "mlp":
        x = st["x"].double()
        return _mm64(_silu64(_mm64(x, st["gate"], bits)) * _mm64(x, st["up"], bits), st["down"], bits)
    if kind in ("attn", "attn_prefill"):
        kvb = case.get("kv_bits", 16)
        return _attn64(st["q"][0].double(), _kv64(st["k"], kvb), _kv64(st["v"], kvb), case["d"] ** -0.5)[None]
    if kind == "moe":
        x, k = st["x"].double(), case["top_k"]
        gates = torch.softmax(st["logits"].double(), -1)
        order = torch.sort(st["logits"].float(), dim=-1, descending=True, stable=True)[1][:, :k]
        p = torch.gather(gates, 1, order)
        p = p / p.sum(-1, keepdim=True)
        out = torch.zeros_like(x)
        for e in range(case["experts"]):
            t, slot = (order == e).nonzero(as_tuple=True)
            if t.numel():
                xe = x[t]
                mats = [tuple(a[e] for a in st[n]) for n in ("gate", "up", "down")]
                y = _mm64(_silu64(_mm64(xe, mats[0], bits)) * _mm64(xe, mats[1], bits), mats[2], bits)
                out.index_add_(0, t, y * p[t, slot].unsqueeze(-1))
        return {"out": out, "experts": None, "scores": p}
    last, streams, kv, head = _model64(case, st)
    if kind == "step":
        taps = sorted({0, case["layers"] - 1})
        return {"logits": _mm64(last, head, 8)[None], "fused": torch.cat([streams[i] for i in taps], -1)[None]}
    return {"logits": _mm64(last[-1:], head, 8)[None], "fused": streams[-1][None], "kv": kv}
