"""The host side of the native verify step: what it passes on, and what it leaves to the single
launches. Host only: no kernel runs."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from dspark_rocm import _lib
from dspark_rocm.kv_cache import KVCache
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
