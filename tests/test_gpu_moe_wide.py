"""GPU: the fused MoE block over a prompt chunk (large buckets, the grouped prefill product).

Against float64 of the dequantized experts with the block's own roundings left out. Bound per output:
the down product of a pair rounds h (bf16, three roundings of silu(gate) * up, each input to it
rounded once: 5 half units of 2^-8 in all), its own sum, its score (bf16, renormalised: 3 roundings),
the scored value and the sum: 10 half units of sum_j score_j * (|h| . |w_down|), and the fp32 sums
under one more. Sizes sit at the edges of the row tiles (32, 64), the 128 / 256-column strips,
the scale chunks (K / 64 a multiple of 8 or not) and the rule that picks this path.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _experts(dev, e, n, k, bits, g):
    from dspark_rocm import quant

    w, s, b = quant.random_quantized(n * e, k, bits, generator=g, device=dev)
    return tuple(t.reshape(e, n, -1) for t in (w, s, b))


def _block(dev, m, e, h, i, bits, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn((m, h), generator=g, device=dev).to(torch.bfloat16)
    logits = torch.randn((m, e), generator=g, device=dev).to(torch.bfloat16)
    return x, logits, [_experts(dev, e, n, k, bits, g) for n, k in ((i, h), (i, h), (h, i))]


def _deq(w, s, b, bits):
    f = 32 // bits
    sh = torch.arange(f, device=w.device, dtype=torch.int32) * bits
    q = ((w.unsqueeze(-1) >> sh) & ((1 << bits) - 1)).double().reshape(w.shape[0], -1, 64)
    wide = q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)
    return wide.reshape(w.shape[0], -1).t().contiguous()


def _check(out, x, inds, scores, mats, bits, what=""):
    ref = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    mag = torch.zeros_like(ref)
    xd = x.double()
    for e in range(mats[0][0].shape[0]):
        t, j = (inds == e).nonzero(as_tuple=True)
        if t.numel():
            gate, up, down = (_deq(*(a[e] for a in m), bits) for m in mats)
            g = xd[t] @ gate
            hh = g * torch.sigmoid(g) * (xd[t] @ up)
            sc = scores[t, j].double().unsqueeze(-1)
            # a half unit of gate moves silu by at most 1.1 |gate| half units
            hm = torch.maximum(hh.abs(), 1.1 * g.abs() * (xd[t] @ up).abs())
            ref.index_add_(0, t, sc * (hh @ down))
            mag.index_add_(0, t, sc * (hm @ down.abs()))
    worst = float(((out.double() - ref).abs() - 10 * 2.0 ** -8 * mag).max())
    assert worst <= 0, f"{what}: error exceeds its bound by {worst}"


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,e,k,h,i", [(17, 2, 1, 128, 128), (80, 8, 1, 256, 128), (100, 4, 2, 512, 384),
                                       (65, 1, 1, 640, 256), (130, 3, 3, 1024, 384), (500, 32, 4, 512, 128),
                                       (257, 2, 2, 192, 64), (1000, 64, 8, 256, 256)])
def test_prompt_chunks_match_float64(dev, bits, m, e, k, h, i):
    from dspark_rocm import ops

    x, logits, mats = _block(dev, m, e, h, i, bits, seed=m + e)
    out, inds, scores = ops.moe_switch_glu(x, logits, *mats, k=k, bits=bits)
    _check(out, x, inds, scores, mats, bits, f"{m}x{e}x{k}x{h}x{i}")
    parts = [ops.moe_switch_glu(x[j:j + 16], logits[j:j + 16], *mats, k=k, bits=bits)[1:] for j in range(0, m, 16)]
    assert torch.equal(inds, torch.cat([p[0] for p in parts])) and torch.equal(scores, torch.cat([p[1] for p in parts]))
    if h % 128 == 0 and i % 128 == 0:            # the packed experts give the same bits
        packed = [(ops.moe_pack(w, bits=bits), s, b) for w, s, b in mats]
        assert torch.equal(ops.moe_switch_glu(x, logits, *packed, k=k, bits=bits)[0], out)


def _row_tiles(m, e, k, h, i, bits):
    """Whether the block of this shape runs the grouped prefill product."""
    from dspark_rocm import ops

    plan = ops.moe_packed_plan(m, h, i, e, k, bits)
    assert (plan["gate_up"] == "row tiles") == (plan["down"] == "row tiles")
    return plan["gate_up"] == "row tiles"


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,e,k,h,i", [(512, 2, 1, 128, 128), (520, 8, 1, 256, 128), (301, 4, 2, 512, 384),
                                       (1030, 1, 1, 640, 256), (345, 3, 3, 1024, 384), (515, 2, 2, 192, 64),
                                       (65, 64, 8, 1024, 384), (97, 128, 8, 512, 256), (33, 16, 8, 2560, 640)])
def test_row_tiles_match_float64(dev, bits, m, e, k, h, i):
    """Sizes the rule sends to the grouped product, at the edges of its tiles, strips and chunks."""
    assert _row_tiles(m, e, k, h, i, bits) or (h > 2048 and bits == 4)
    test_prompt_chunks_match_float64(dev, bits, m, e, k, h, i)


@pytest.mark.parametrize("m", [16, 17, 255, 256, 257])
def test_both_sides_of_the_rule(dev, m):
    """16 small experts, one each: from 256 tokens on."""
    from dspark_rocm import ops

    assert _row_tiles(m, 16, 1, 256, 192, 4) == (m >= 256)
    x, logits, mats = _block(dev, m, 16, 256, 192, 4, seed=m)
    out, inds, scores = ops.moe_switch_glu(x, logits, *mats, k=1, bits=4)
    _check(out, x, inds, scores, mats, 4, f"{m} rows")


@pytest.mark.parametrize("bits", [4, 8])
def test_one_bucket_holds_every_token(dev, bits):
    """Every token on the same experts: their buckets take many row tiles, the others none."""
    from dspark_rocm import ops

    assert _row_tiles(300, 32, 2, 256, 128, bits)
    x, logits, mats = _block(dev, 300, 32, 256, 128, bits)
    logits[:, 3] = 9.0
    logits[:, 30] = 8.0
    out, inds, scores = ops.moe_switch_glu(x, logits, *mats, k=2, bits=bits)
    assert bool((inds == torch.tensor([3, 30], device=dev)).all())
    _check(out, x, inds, scores, mats, bits)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("bits", [4, 8])
def test_an_infinite_input_is_the_plain_product(dev, bits, packed):
    """The outputs of a row that holds an infinity are those of the dequantized product (an infinity
    or a NaN, never a finite value), and the other rows keep their bits."""
    from dspark_rocm import ops

    assert _row_tiles(320, 4, 1, 256, 128, bits)
    x, logits, mats = _block(dev, 320, 4, 256, 128, bits)
    arg = [(ops.moe_pack(w, bits=bits), s, b) for w, s, b in mats] if packed else mats
    want, inds, scores = ops.moe_switch_glu(x, logits, *arg, k=1, bits=bits)
    x2 = x.clone()
    x2[5, 70] = float("inf")
    out = ops.moe_switch_glu(x2, logits, *arg, k=1, bits=bits)[0]
    keep = torch.arange(320, device=dev) != 5
    assert torch.equal(out[keep], want[keep])
    e = int(inds[5, 0])
    gate, up, down = (_deq(*(a[e] for a in m), bits) for m in mats)
    g, u = x2[5].double() @ gate, x2[5].double() @ up
    h = g * torch.sigmoid(g) * u                 # -inf * 0 is a NaN in both
    ref = h @ down
    assert not bool(torch.isfinite(ref).any()) and not bool(torch.isfinite(out[5]).any())
    assert torch.equal(torch.isnan(out[5]), torch.isnan(ref))


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("bits", [4, 8])
def test_an_infinite_weight_beside_an_infinite_row(dev, bits, packed):
    """A gate of inf * 1 + 2 * -inf is a NaN, not an infinity, and so is the sum of its columns."""
    from dspark_rocm import ops

    x, logits, mats = _block(dev, 320, 4, 256, 128, bits)
    inds = ops.moe_switch_glu(x, logits, *mats, k=1, bits=bits)[1]
    e = int(inds[5, 0])
    (_, gs, gb), (_, us, ub), (_, ds, db) = mats
    gs[e, :, 0], gb[e, :, 0], gs[e, :, 1], gb[e, :, 1] = 0, 1, 0, -float("inf")
    us[e], ub[e], ds[e], db[e] = 0, 0, 0, 1
    ub[e, :, 2] = 1
    x[:, 64:128], x[5, 3], x[5, 128:192] = 2 / 64, float("inf"), 1
    arg = [(ops.moe_pack(w, bits=bits), s, b) for w, s, b in mats] if packed else mats
    g = x[5].double() @ _deq(*(a[e] for a in mats[0]), bits)
    assert bool(torch.isnan(g).all())
    assert bool(torch.isnan(ops.moe_switch_glu(x, logits, *arg, k=1, bits=bits)[0][5]).all())


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("bits", [4, 8])
def test_infinite_rows_cost_no_more_than_their_terms(dev, bits, packed):
    """An infinity in every row: the call stays within 20 times one without (about 3 measured; a whole
    product per output took 480), and no output is finite."""
    from dspark_rocm import ops

    assert _row_tiles(300, 8, 4, 1024, 512, bits)
    x, logits, mats = _block(dev, 300, 8, 1024, 512, bits)
    arg = [(ops.moe_pack(w, bits=bits), s, b) for w, s, b in mats] if packed else mats
    x2 = x.clone()
    x2[:, 3] = float("inf")

    def us(x):
        best = float("inf")
        for _ in range(4):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            ops.moe_switch_glu(x, logits, *arg, k=4, bits=bits)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3)
        return best

    assert not bool(torch.isfinite(ops.moe_switch_glu(x2, logits, *arg, k=4, bits=bits)[0]).any())
    assert us(x2) <= 20 * us(x) + 100
