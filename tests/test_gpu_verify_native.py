"""GPU: the verify step enqueued from native code against the same launches made one by one: the
same kernels on the same operands, so logits, taps and caches agree to the bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _target(dev, d, bits, kv_bits):
    from dspark_rocm.model import DenseModel, ModelArgs, Target

    args = ModelArgs(hidden_size=512, num_hidden_layers=3, intermediate_size=1024, num_attention_heads=512 // d,
                     num_key_value_heads=2, head_dim=d, vocab_size=1000, bits=bits)
    return Target(DenseModel.random(args, device=dev, seed=3), kv_bits=kv_bits)


def _rounds(tgt, tap):
    cache = tgt.make_cache(8)
    g = torch.Generator().manual_seed(0)
    out = []
    for m, reject in ((16, 3), (1, 0), (5, 5), (16, 0), (2, 1)):
        logits, fused = tgt.verify(torch.randint(0, 1000, (1, m), generator=g), cache, tap)
        out += [logits.clone()] + ([] if fused is None else [fused.clone()])
        tgt.rollback(cache, reject)
    for c in cache:
        for part in c.fetch():
            out += list(part) if isinstance(part, tuple) else [part]
    return out


@pytest.mark.parametrize("tap", [None, (0, 2), (1,)])
@pytest.mark.parametrize("d,bits,kv_bits", [(128, 8, None), (64, 4, 8), (256, 8, 4)])
def test_native_step_is_the_launch_sequence(dev, monkeypatch, d, bits, kv_bits, tap):
    from dspark_rocm.model import VerifyEngine

    tgt = _target(dev, d, bits, kv_bits)
    took, native = [], VerifyEngine._native_step
    monkeypatch.setattr(VerifyEngine, "_native_step", lambda self, *a: took.append(native(self, *a)) or took[-1])
    got = _rounds(tgt, tap)
    assert took and all(took)
    monkeypatch.setattr(VerifyEngine, "_native_step", lambda self, *a: False)
    want = _rounds(tgt, tap)
    assert len(got) == len(want) and all(torch.equal(g, w) for g, w in zip(got, want))


def test_steps_it_leaves_alone(dev):
    """Unpacked projections and another cache class are enqueued launch by launch; a cache without
    room is refused as before."""
    from dspark_rocm.kv_cache import KVCache
    from dspark_rocm.model import Target

    class Other(KVCache):
        pass

    tgt = _target(dev, 128, 8, None)
    plain = Target(tgt.model, packed=False)
    cache = tgt.make_cache(32)
    assert tgt.engine._native_layers(4, cache, 0) and tgt.engine._native_layers(4, cache, cache[0].capacity) is None
    assert plain.engine._native_layers(4, cache, 0) is None
    other = [Other(1, 2, 128, device=dev, capacity=32) for _ in cache]
    assert tgt.engine._native_layers(4, other, 0) is None
    ids = torch.arange(4)[None]
    want = tgt.verify(ids, cache)[0].clone()
    assert torch.equal(tgt.verify(ids, other)[0], want)
    with pytest.raises(ValueError):
        tgt.engine.step(4, cache, cache[0].capacity)


def test_step_without_a_qmm_workspace(dev, monkeypatch):
    """A target whose matrices are all one K slice holds no qmm workspace; its steps are native too."""
    from dspark_rocm.model import DenseModel, ModelArgs, Target, VerifyEngine

    args = ModelArgs(hidden_size=512, num_hidden_layers=2, intermediate_size=512, num_attention_heads=4,
                     num_key_value_heads=2, head_dim=128, vocab_size=1000, bits=8)
    tgt = Target(DenseModel.random(args, device=dev, seed=3))
    assert tgt.engine.qmm_ws is None and tgt.engine._native_layers(4, tgt.make_cache(8), 0)
    got = _rounds(tgt, None)
    monkeypatch.setattr(VerifyEngine, "_native_step", lambda self, *a: False)
    assert all(torch.equal(g, w) for g, w in zip(got, _rounds(tgt, None)))
