"""GPU: attention over many query rows (``dspark_prefill_attention``) behind the stock entry point.

Against float64 attention of the same inputs. Bound per output: half a unit of the output type, plus
the errors of the fp32 path: a score is off by at most (D + 2) units of 2^-24 of scale * sum |q k|
and its exponent's argument by as much again of its size, a probability by that and the units of its
exponential, the two sums over L keys by L / 16 units (16 keys a lane are added in turn, 16 or more in
the matrix core); numerator and denominator both, over sum p |v|.
Sizes sit at the edges of the 32-row waves, 128-row workgroups, 64-key tiles and key splits.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _inputs(dev, b, hq, hk, m, L, d, dtype, seed=0, qscale=2.0):
    g = torch.Generator(device=dev).manual_seed(seed)
    mk = lambda h, n, s: (torch.randn((b, h, n, d), generator=g, device=dev) * s).to(dtype)  # noqa: E731
    return mk(hq, m, qscale), mk(hk, L, 1.0), mk(hk, L, 1.0)


def _reference(q, k, v, scale, causal):
    """(float64 attention, sum p |v|, largest scale * sum |q k| of a row)"""
    hq, m, L = q.shape[1], q.shape[2], k.shape[2]
    rep = hq // k.shape[1]
    kk, vv = (t.double().repeat_interleave(rep, dim=1) for t in (k, v))
    kt = kk.transpose(-1, -2).contiguous()
    s = torch.matmul(q.double(), kt) * scale
    mag = torch.matmul(q.double().abs(), kt.abs()) * scale
    if causal:
        i, j = torch.arange(m, device=q.device)[:, None], torch.arange(L, device=q.device)[None]
        s = s.masked_fill(j > L - m + i, float("-inf"))
    p = torch.softmax(s, -1)
    return torch.matmul(p, vv), torch.matmul(p, vv.abs()), mag.amax(-1, keepdim=True)


def _check(out, q, k, v, scale, causal, what=""):
    ref, pv, mag = _reference(q, k, v, scale, causal)
    amp = 2 * (2 * (q.shape[-1] + 2) * mag + 8 + k.shape[2] / 16) * 2.0 ** -24
    bound = UNIT[q.dtype] * (ref.abs() + amp * pv) + amp * pv + 2.0 ** -25
    worst = float(((out.double() - ref).abs() - bound).max())
    assert out.shape == ref.shape and out.dtype == q.dtype and out.is_contiguous()
    assert worst <= 0, f"{what}: error exceeds its bound by {worst}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,hq,hk,m,L", [(1, 1, 1, 17, 17), (1, 4, 1, 32, 33), (2, 6, 2, 43, 64), (1, 8, 8, 129, 129),
                                         (1, 8, 2, 33, 1500), (1, 5, 1, 100, 257), (1, 16, 1, 24, 31 + 24),
                                         (1, 32, 8, 300, 1301), (1, 64, 8, 65, 2048)])
def test_matches_float64_attention(dev, b, hq, hk, m, L, d, dtype):
    from dspark_rocm import fast

    q, k, v = _inputs(dev, b, hq, hk, m, L, d, dtype)
    for mask in ("causal", None):
        assert fast.prefill_kernel(q, k, v, d ** -0.5, mask, None)
        out = fast.scaled_dot_product_attention(q, k, v, scale=d ** -0.5, mask=mask)
        _check(out, q, k, v, d ** -0.5, mask == "causal", f"{b}x{hq}/{hk}x{m}x{L}x{d} {mask}")


def test_views_of_a_cache_and_of_projections(dev):
    """A cache's filled rows and [B, L, H, D] projections seen as [B, H, L, D] are read in place, to
    the bits of their contiguous copies."""
    from dspark_rocm import fast

    q, k, v = _inputs(dev, 2, 8, 2, 70, 190, 128, torch.bfloat16)
    want = fast.scaled_dot_product_attention(q, k, v, scale=0.1, mask="causal")
    _check(want, q, k, v, 0.1, True)
    big = torch.full((2, 2, 256, 128), float("nan"), dtype=k.dtype, device=dev)
    kc, vc = big.clone(), big.clone()
    kc[:, :, :190], vc[:, :, :190] = k, v
    qt = q.transpose(1, 2).contiguous().transpose(1, 2)
    kt = k.transpose(1, 2).contiguous().transpose(1, 2)
    for qq, kk, vv in ((q, kc[:, :, :190], vc[:, :, :190]), (qt, kt, v)):
        assert fast.prefill_kernel(qq, kk, vv, 0.1, "causal", None)
        got = fast.scaled_dot_product_attention(qq, kk, vv, scale=0.1, mask="causal")
        assert torch.equal(got, want)


def test_calls_that_keep_the_torch_ops(dev):
    from dspark_rocm import fast

    q, k, v = _inputs(dev, 1, 4, 2, 20, 40, 64, torch.bfloat16)
    ok = lambda q=q, k=k, v=v, scale=0.1, mask="causal", sinks=None: fast.prefill_kernel(  # noqa: E731
        q, k, v, scale, mask, sinks)
    assert ok()
    assert not ok(q=q[:, :, :16])
    assert not ok(q=q.float()) and not ok(q=q.half())
    assert not ok(mask=torch.ones(20, 40, dtype=torch.bool, device=dev))
    assert not ok(sinks=torch.zeros(4, device=dev))
    assert not ok(k=k[:, :, :19], v=v[:, :, :19]) and ok(k=k[:, :, :19], v=v[:, :, :19], mask=None)
    assert not ok(scale=0.0) and not ok(scale=-1.0) and not ok(scale=float("inf"))
    assert not ok(q=q[..., :40], k=k[..., :40], v=v[..., :40])
    assert not ok(k=k[:, :, :, ::1].transpose(2, 3).contiguous().transpose(2, 3))
    shifted = torch.zeros(q.numel() + 1, dtype=q.dtype, device=dev)[1:].view(q.shape)
    assert not ok(q=shifted)
    qg = q.clone().requires_grad_()
    assert not ok(q=qg)
    fast.scaled_dot_product_attention(qg, k, v, scale=0.1, mask="causal").float().sum().backward()
    assert qg.grad is not None and bool(torch.isfinite(qg.grad).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_large_scores_and_non_finite_values(dev, dtype):
    """Scores of any size keep the softmax exact at its maximum; a row whose scores hold an infinity
    or a NaN is NaN, as the torch ops have it, and the other rows are what they were."""
    from dspark_rocm import fast

    q, k, v = _inputs(dev, 1, 2, 1, 40, 700, 64, dtype)
    big = (q.float() * 200).to(dtype), (k.float() * 200).to(dtype)
    ref, _, _ = _reference(*big, v, 50.0, True)
    out = fast.scaled_dot_product_attention(*big, v, scale=50.0, mask="causal")
    assert float((out.double() - ref).abs().max()) <= UNIT[dtype] * float(ref.abs().max())
    want = fast.scaled_dot_product_attention(q, k, v, scale=0.125, mask="causal")
    q2 = q.clone()
    q2[0, 1, 7, 3] = float("inf")
    q2[0, 0, 9, 5] = float("nan")
    out = fast.scaled_dot_product_attention(q2, k, v, scale=0.125, mask="causal")
    hit = torch.zeros((2, 40), dtype=torch.bool, device=dev)
    hit[1, 7] = hit[0, 9] = True
    assert bool(torch.isnan(out[0][hit]).all()) and torch.equal(out[0][~hit], want[0][~hit])


def test_capture_replays_on_new_inputs(dev):
    from dspark_rocm import fast

    q, k, v = _inputs(dev, 1, 8, 2, 64, 900, 128, torch.bfloat16)   # splits the keys
    run = lambda: fast.scaled_dot_product_attention(q, k, v, scale=0.1, mask="causal")  # noqa: E731
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for seed in (1, 2, 3):
        for t, n in zip((q, k, v), _inputs(dev, 1, 8, 2, 64, 900, 128, torch.bfloat16, seed=seed)):
            t.copy_(n)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, run())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,L", [(64, 33), (128, 90), (256, 90), (64, 1200), (128, 1200), (256, 1200)])
def test_small_probabilities_keep_fp32_precision(dev, dtype, d, L):
    """The largest weight of every row falls on a key whose value is zero, so probabilities of e^-gap
    of it make up the output. All are equal, so what their pieces lose does not average out. The
    scores are exact; the bound is half a unit of the output type, the fp32 errors of the exponent's
    argument (3 units of its size, gap) and the units of the two sums."""
    from dspark_rocm import fast

    g = torch.Generator(device=dev).manual_seed(3)
    for gap in (9.625, 13.25, 17.25, 18.875, 20.125, 22.75):
        q = torch.zeros((1, 4, 24, d), dtype=dtype, device=dev)
        q[..., 0] = 1
        k = torch.zeros((1, 2, L, d), dtype=dtype, device=dev)
        k[:, :, 5, 0] = gap
        v = (torch.rand((1, 2, L, d), generator=g, device=dev) * 3e4 + 3e4).to(dtype)
        v[:, :, 5] = 0
        for mask in (None, "causal") if L > 33 else (None,):
            assert fast.prefill_kernel(q, k, v, 1.0, mask, None)
            out = fast.scaled_dot_product_attention(q, k, v, scale=1.0, mask=mask)
            ref = _reference(q, k, v, 1.0, mask == "causal")[0]
            bound = (UNIT[dtype] + (3 * gap + 8 + L / 16) * 2.0 ** -24) * ref.abs() + 2.0 ** -25
            worst = float(((out.double() - ref).abs() / bound).max())
            assert worst <= 1, f"gap {gap} {mask}: {worst} of the bound"


@pytest.mark.parametrize("b,hq,hk,m,d", [(1, 8, 2, 2048, 64), (1, 8, 2, 1000, 64), (1, 4, 1, 700, 128),
                                         (1, 2, 1, 400, 256)])
def test_key_splits_without_keys(dev, b, hq, hk, m, d):
    """Few KV heads over as many rows as keys split the keys, and the first row tiles see fewer key
    tiles than there are splits: a split without any has nothing to add."""
    from dspark_rocm import _lib, fast

    assert _lib.load().dspark_prefill_attention_workspace(b, hq, hk, m, m, d) > 0
    q, k, v = _inputs(dev, b, hq, hk, m, m, d, torch.bfloat16)
    out = fast.scaled_dot_product_attention(q, k, v, scale=d ** -0.5, mask="causal")
    _check(out, q, k, v, d ** -0.5, True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hk,m,L,d", [(1, 4, 2, 70, 150, 64), (2, 6, 2, 43, 64, 128), (1, 2, 1, 40, 90, 256),
                                           (1, 8, 2, 33, 1500, 64), (1, 8, 2, 33, 1500, 128), (1, 5, 1, 19, 1300, 256)])
def test_values_that_are_not_finite(dev, dtype, b, hq, hk, m, L, d):
    """An infinite value makes its column infinite in the rows that see its key, a NaN or both signs
    make it NaN. Rows masked from it keep theirs or, in its tile, are NaN (zero times infinity, as a
    product over all keys has it); every other output is what it was, to the bit."""
    from dspark_rocm import fast

    inf, nan = float("inf"), float("nan")
    q, k, v = _inputs(dev, b, hq, hk, m, L, d, dtype, qscale=0.5)
    rep, scale, j = hq // hk, d ** -0.5, L - m + 9        # rows 9.. see key j
    v2 = v.clone()
    v2[:, 0, j, 0], v2[:, 0, j, 1], v2[:, -1, j, d - 1] = inf, -inf, nan
    v2[:, 0, 3, 2], v2[:, 0, 4, 2] = inf, -inf
    v2[:, 0, 2, 4] = -inf
    for mask in ("causal", None):
        clean = fast.scaled_dot_product_attention(q, k, v, scale=scale, mask=mask)
        got = fast.scaled_dot_product_attention(q, k, v2, scale=scale, mask=mask)
        first = 9 if mask else 0
        for heads, row, col, value in ((slice(0, rep), first, 0, inf), (slice(0, rep), first, 1, -inf),
                                       (slice(0, rep), 0, 2, nan), (slice(0, rep), 0, 4, -inf),
                                       (slice(hq - rep, hq), first, d - 1, nan)):
            hit, before = got[:, heads, row:, col], got[:, heads, :row, col]
            assert bool((hit.isnan() if value != value else hit == value).all()), f"column {col} {mask}"
            assert bool((before.isnan() | (before == clean[:, heads, :row, col])).all())
            got[:, heads, :, col] = clean[:, heads, :, col]
        assert torch.equal(got, clean)


@pytest.mark.parametrize("d,L", [(64, 100), (128, 1500)])
def test_values_at_the_end_of_the_range(dev, d, L):
    """Values whose unnormalised sum passes the largest fp32 number: the mean of them does not."""
    from dspark_rocm import fast

    q, k, v = _inputs(dev, 1, 4, 2, 20, L, d, torch.bfloat16)
    v = (v.float().clamp(-3, 3) * 2.0 ** 125).to(torch.bfloat16)
    v[..., : d // 2] = v[..., : d // 2].abs()
    out = fast.scaled_dot_product_attention(q, k, v, scale=0.01, mask="causal")
    _check(out, q, k, v, 0.01, True)


def test_function_transforms_keep_the_torch_ops(dev):
    """vmap, grad and jvp over the stock entry point, whose tensors have no data pointer."""
    from dspark_rocm import fast

    q, k, v = _inputs(dev, 3, 4, 2, 20, 40, 64, torch.bfloat16)
    f = lambda q, k, v: fast.scaled_dot_product_attention(q, k, v, scale=0.1, mask="causal")  # noqa: E731
    out = torch.vmap(f)(*(t.unsqueeze(1) for t in (q, k, v)))
    _check(out.squeeze(1).contiguous(), q, k, v, 0.1, True)
    qg = q.clone().requires_grad_()
    want, = torch.autograd.grad(f(qg, k, v).float().sum(), qg)
    assert torch.equal(torch.func.grad(lambda q: f(q, k, v).float().sum())(q), want)
    primal, tangent = torch.func.jvp(lambda q: f(q, k, v), (q,), (q,))
    _check(primal, q, k, v, 0.1, True)
    assert bool(torch.isfinite(tangent).all()) and float(tangent.float().abs().max()) > 0
