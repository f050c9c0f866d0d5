"""GPU: the module path's fused row kernels at prefill widths against its torch ops.

Both round at the same points; they differ where an fp32 sum or a sine lands on the other side of a
bf16 rounding, so layer by layer by isolated half units (2^-8 of a value), which a random-weight
stack carries on: two layers stay within 2^-6 in the 2-norm.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _target(dev, d=128, hq=4, hk=2, kv_bits=None, seed=0):
    from dspark_rocm.model import DenseModel, ModelArgs, Target

    args = ModelArgs(hidden_size=512, num_hidden_layers=2, intermediate_size=768, num_attention_heads=hq,
                     num_key_value_heads=hk, head_dim=d, vocab_size=640, bits=8)
    return Target(DenseModel.random(args, device=dev, seed=seed), kv_bits=kv_bits)


def _chunks(tgt, ids, sizes):
    cache = tgt.make_cache(8)                    # grows under the chunks
    out, at = [], 0
    for n in sizes:
        logits, fused = tgt.prefill(ids[:, at:at + n], cache, tap=(0, 1), want_logits=True)
        out += [logits, fused]
        at += n
    return out + [t for c in cache for t in c.fetch()]


@pytest.mark.parametrize("d,hq,hk,sizes", [(128, 4, 2, (17,)), (64, 8, 2, (40, 300)), (256, 2, 1, (33, 16, 18)),
                                           (96, 2, 2, (20,))])
def test_fused_rows_match_the_torch_ops(dev, monkeypatch, d, hq, hk, sizes):
    from dspark_rocm import model as mod

    tgt = _target(dev, d, hq, hk)
    ids = torch.randint(0, 640, (1, sum(sizes)), generator=torch.Generator().manual_seed(1))
    got = _chunks(tgt, ids, sizes)
    calls = []
    monkeypatch.setattr(mod, "_fused", lambda rows, *ts: calls.append(rows) and False)
    want = _chunks(tgt, ids, sizes)
    assert calls
    for g, w in zip(got, want):
        assert g.shape == w.shape and g.dtype == w.dtype
        rel = float((g.double() - w.double()).norm() / w.double().norm())
        assert rel <= 2.0 ** -6, rel


def test_what_keeps_the_torch_ops(dev):
    """Verify widths, a quantized cache, rows autograd follows."""
    from dspark_rocm import model as mod

    x = torch.randn(17, 64, device=dev).to(torch.bfloat16)
    assert mod._fused(17, x) and not mod._fused(16, x) and not mod._fused(17, x.float())
    assert not mod._fused(17, x[:, :32]) and not mod._fused(17, x.clone().requires_grad_())
    tgt = _target(dev, kv_bits=8)
    out = _chunks(tgt, torch.arange(20)[None], (20,))
    assert bool(torch.isfinite(out[0].float()).all())
    layer = tgt.model.layers[0]
    h = torch.randn(1, 20, 512, device=dev).to(torch.bfloat16).requires_grad_()
    layer.mlp(mod.add_rms_norm(h, None, layer.post_attention_layernorm, 1e-6)[1]).float().sum().backward()
    assert h.grad is not None and bool(torch.isfinite(h.grad).all())
