"""GPU: the module path's fused row kernels at prefill widths against its torch ops.

Both round at the same points; they differ where an fp32 sum or a sine lands on the other side of a
bf16 rounding, so op by op in few values and by few units (a unit is at most 2^-7 of a value). A
random-weight stack carries that on: two layers stay within 2^-6 in the 2-norm.
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


def _few_units(got, want, scale, units):
    """Every value within ``units`` bf16 units of ``scale``, and equal but for one in fifty: an fp32
    sum of n terms is off by up to n 2^-24 of itself, which crosses a bf16 rounding for at most n 2^-16
    of the values (1 in 128 at 512 terms); an angle of up to 300 by 300 2^-24, half that."""
    assert got.shape == want.shape and got.dtype == want.dtype == torch.bfloat16
    d = (got.double() - want.double()).abs()
    assert float((d - units * 2.0 ** -7 * scale).max()) <= 0
    assert float((d > 0).double().mean()) <= 0.02


@pytest.mark.parametrize("d,hq,hk,rows", [(128, 4, 2, 17), (64, 8, 2, 300), (256, 2, 1, 33), (96, 2, 2, 20)])
def test_each_fused_op_matches_its_torch_ops(dev, monkeypatch, d, hq, hk, rows):
    from dspark_rocm import model as mod

    tgt = _target(dev, d, hq, hk)
    layer = tgt.model.layers[0]
    layer.mlp.down_proj = torch.nn.Identity()
    g = torch.Generator(device=dev).manual_seed(rows)
    x, r = (torch.randn((1, rows, 512), generator=g, device=dev).to(torch.bfloat16) for _ in range(2))
    w = (1 + 0.1 * torch.randn(512, generator=g, device=dev)).to(torch.bfloat16)
    real = mod.fast.scaled_dot_product_attention

    def run():
        qs = []
        monkeypatch.setattr(mod.fast, "scaled_dot_product_attention", lambda q, *a, **k: qs.append(q) or real(q, *a, **k))
        cache = tgt.make_cache(rows)[0]
        layer.self_attn(x, cache)
        return (*mod.add_rms_norm(x, r, w, 1e-6), *mod.add_rms_norm(x, None, w, 1e-6)[1:], layer.mlp(x), qs[0],
                *cache.fetch())

    with torch.no_grad():
        got = run()
        calls = []
        monkeypatch.setattr(mod, "_fused", lambda n, *ts: calls.append(n) and False)
        want = run()
    assert len(calls) == 4
    h, y, y1, mlp, q, k, v = zip(got, want)
    assert torch.equal(*h) and torch.equal(*v)
    for a, b in (y, y1):            # two roundings: of the normalised value and of its product with w
        _few_units(a, b, b.double().abs(), 2)
    _few_units(*mlp, mlp[1].double().abs(), 3)      # of the sigmoid, times g, times u
    for a, b in (q, k):             # the norm's two, then a rotation: |x1| + |x2| <= sqrt(2) of the pair's length
        pair = torch.hypot(b.double(), b.double().roll(d // 2, -1))
        _few_units(a, b, 2 ** 0.5 * pair, 3)


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
