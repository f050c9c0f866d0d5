"""The host side of the native verify step: what it passes on, and what it leaves to the single
launches. It is given bare pointers and strides, so it has to leave alone every cache and norm weight
that is not what the kernels take it for; the single launches refuse those. Host only: no kernel
runs."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from dspark_rocm import _lib, ops
from dspark_rocm.kv_cache import KVCache, QuantizedKVCache
from dspark_rocm.model import DenseModel, ModelArgs, VerifyEngine

HK, D = 2, 64


def _engine(width=512):
    args = ModelArgs(hidden_size=width, num_hidden_layers=2, intermediate_size=width, num_attention_heads=width // D,
                     num_key_value_heads=HK, head_dim=D, vocab_size=64, bits=8)
    model = DenseModel.random(args, device="cpu", seed=1)
    e = VerifyEngine(model, packed=False)

    def pack(mod):
        n, words = mod.weight.shape
        return SimpleNamespace(n=n, k=words * 32 // mod.bits, bits=mod.bits, buf=mod.weight)

    for layer in model.layers:
        at, mlp = layer.self_attn, layer.mlp
        e._packed.update({id(m): pack(m) for m in (at.q_proj, at.k_proj, at.v_proj, at.o_proj, mlp.down_proj)})
        e._swiglu[id(mlp)] = pack(mlp.gate_proj)
    e._packed[id(model.lm_head)] = pack(model.lm_head)
    return e


@pytest.fixture
def calls(monkeypatch):
    out = []
    monkeypatch.setattr(_lib, "call", lambda *a: out.append(a))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: SimpleNamespace(cuda_stream=0))
    return out


@pytest.mark.parametrize("width,needs", [(512, False), (2048, True)])
def test_workspace_is_passed_where_there_is_one(calls, width, needs):
    """Matrices of one K slice need no workspace, and the engine then holds none."""
    e = _engine(width)
    assert (e.qmm_ws is not None) == needs
    cache = [KVCache(1, HK, D, device="cpu", capacity=32) for _ in range(2)]
    assert e._native_step(4, cache, 0)
    (name, args, *_), = calls
    assert name == "dspark_verify_step"
    assert (args.qmm_ws, args.qmm_ws_bytes) == ((e.qmm_ws.data_ptr(), e.qmm_ws.numel()) if needs else (None, 0))


def _caches(kv_bits, batch=1, heads=HK, dim=D, device="cpu", **kw):
    make = (lambda: QuantizedKVCache(batch, heads, dim, bits=kv_bits, device=device, capacity=32, **kw)) if kv_bits \
        else (lambda: KVCache(batch, heads, dim, device=device, capacity=32, **kw))
    return [make(), make()]


@pytest.mark.parametrize("kv_bits", [0, 8, 4])
def test_caches_the_native_step_refuses(kv_bits):
    e = _engine()
    good = _caches(kv_bits)
    assert e._native_layers(4, good, 0) and e._native_layers(4, good, 252)
    assert e._native_layers(4, good, 253) is None                              # no room
    bad = {"another device": _caches(kv_bits, device="meta"), "batch 2": _caches(kv_bits, batch=2),
           "fewer heads": _caches(kv_bits, heads=1), "more heads": _caches(kv_bits, heads=4),
           "wider heads": _caches(kv_bits, dim=128), "fp16": _caches(kv_bits, dtype=torch.float16)}
    if not kv_bits:
        bad["narrower heads"] = _caches(0, dim=32)
    for what, c in bad.items():
        assert e._native_layers(4, c, 0) is None, what
        assert e._native_layers(4, [good[0], c[1]], 0) is None, what          # every layer's, not the first's
    mixed = _caches(kv_bits)
    if kv_bits:
        w, s, b = mixed[1].values
        mixed[1].values = (w[:, :, :2], s, b)
        assert e._native_layers(4, mixed, 0) is None                           # one tensor too short
        mixed[1].values = (w.float(), s, b)
        assert e._native_layers(4, mixed, 0) is None
        mixed[1].values, mixed[1].group_size = (w, s, b), 32
        assert e._native_layers(4, mixed, 0) is None
    else:
        v = mixed[1].values
        mixed[1].values = v[:, :, :2]
        assert e._native_layers(4, mixed, 0) is None
        mixed[1].values = v.transpose(2, 3).contiguous().transpose(2, 3)       # no unit last stride
        assert e._native_layers(4, mixed, 0) is None
        mixed[1].values = v.half()                                             # not the type it claims
        assert e._native_layers(4, mixed, 0) is None


@pytest.mark.parametrize("owner,name", [("layer", "input_layernorm"), ("layer", "post_attention_layernorm"),
                                        ("attn", "q_norm"), ("attn", "k_norm"), ("model", "norm")])
def test_norm_weights_the_native_step_refuses(calls, owner, name):
    e = _engine()
    cache = _caches(0)
    assert e._native_step(4, cache, 0) and [c[0] for c in calls] == ["dspark_verify_step"]
    mod = {"layer": e.model.layers[1], "attn": e.model.layers[1].self_attn, "model": e.model}[owner]
    w = getattr(mod, name)
    for bad in (w.float(), w[:-8], w.repeat(2)[::2], w.to("meta")):
        setattr(mod, name, bad)
        assert not e._native_step(4, cache, 0)
    assert len(calls) == 1


def test_the_single_launches_refuse_caches_too_small(calls, monkeypatch):
    """Fewer heads or narrower rows than the kernel will write are refused before it is launched."""
    monkeypatch.setattr(ops, "_require_cuda", lambda *ts: None)
    monkeypatch.setattr(ops, "_stream", lambda t: 0)
    q, k, w = torch.zeros(3, 4 * D).bfloat16(), torch.zeros(3, HK * D).bfloat16(), torch.ones(D).bfloat16()
    kw = dict(heads=4, kv_heads=HK, head_dim=D, eps=1e-6, rope_base=1e4, pos0=0, q_out=torch.zeros(4, 3, D).bfloat16())

    def plain(heads, dim):
        c = torch.zeros(heads, 8, dim).bfloat16()
        ops.qk_norm_rope_kv(q, k, k, w, w, k_cache=c, v_cache=c, **kw)

    def quantized(heads, dim):
        sb = torch.zeros(heads, 8, max(dim // 64, 1)).bfloat16()
        c = (torch.zeros(heads, 8, dim // 4, dtype=torch.int32), sb, sb)
        ops.qk_norm_rope_kv_quantized(q, k, k, w, w, k_cache=c, v_cache=c, bits=8, **kw)

    for f in (plain, quantized):
        f(HK, D)
        done = len(calls)
        for heads, dim in ((HK - 1, D), (HK, D // 2)):
            with pytest.raises(ValueError):
                f(heads, dim)
        assert len(calls) == done
    assert len(calls) == 2
