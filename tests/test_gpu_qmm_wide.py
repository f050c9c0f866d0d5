"""GPU: the many-row quantized product (``dspark_qmm_wide``) behind QuantizedLinear's stock path.

Against the float64 product of the dequantized weight. Bound per output: one bf16 rounding (8
significant bits: half a unit is at most 2^-8 of the value; twice with a bias), plus fp32 sums of
at most 64 + 7 G terms over sum |x| (|s| (q + 16) + |b|), the factored terms' magnitude (q + 16:
the 4-bit field offset).
Sizes sit at the edges of the tiles (16-row steps, 128/256-column workgroups), of the scale chunks
(G % 8), of the K slices and of the 32-group bias steps.
"""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _mats(dev, n, k, bits, seed=0):
    from dspark_rocm import quant

    g = torch.Generator(device=dev).manual_seed(seed)
    return quant.random_quantized(n, k, bits, generator=g, device=dev)


def _x(dev, m, k, seed=1):
    g = torch.Generator(device=dev).manual_seed(seed)
    return torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)


def _reference(x, w, s, b, bits):
    """(float64 product, sum of the magnitudes of the factored terms)"""
    f = 32 // bits
    sh = torch.arange(f, device=w.device, dtype=torch.int32) * bits
    q = ((w.unsqueeze(-1) >> sh) & ((1 << bits) - 1)).double().reshape(w.shape[0], -1, 64)
    s, b = s.double().unsqueeze(-1), b.double().unsqueeze(-1)
    wide = lambda t: t.reshape(w.shape[0], -1).t().contiguous()  # noqa: E731
    return x.double() @ wide(q * s + b), x.double().abs() @ wide((q + 16) * s.abs() + b.abs())


def _check(y, x, w, s, b, bits, bias=None, what=""):
    ref, mag = _reference(x.reshape(-1, x.shape[-1]), w, s, b, bits)
    n_terms = 64 + 7 * s.shape[1]
    sums = n_terms * 2.0 ** -24 * mag
    bound = 2.0 ** -8 * (ref.abs() + sums) + sums
    if bias is not None:
        ref = ref + bias.double()
        bound = bound + 2.0 ** -8 * (ref.abs() + bound)
    err = (y.reshape(ref.shape).double() - ref).abs()
    worst = float((err - bound).max())
    assert worst <= 0, f"{what}: error exceeds its bound by {worst}"


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(1, 515, 1088), (16, 130, 4096), (17, 1, 64), (32, 64, 128), (33, 130, 512), (65, 257, 576), (96, 128, 1088),
                                   (97, 300, 2112), (129, 1000, 4096), (256, 4096, 1024), (300, 515, 8256)])
def test_matches_the_float64_product(dev, m, n, k, bits):
    from dspark_rocm import ops

    w, s, b = _mats(dev, n, k, bits)
    x = _x(dev, m, k)
    _check(ops.quantized_matmul_wide(x, w, s, b, bits=bits), x, w, s, b, bits, what=f"{m}x{n}x{k}")


@pytest.mark.parametrize("bits", [4, 8])
def test_forms_the_stock_path_accepts(dev, bits):
    """Leading dims, row strides, misaligned views, a module bias: all against the same bound, and
    the rows of one call equal to the bit whatever the view they came from."""
    from dspark_rocm.nn import QuantizedLinear

    n, k, m = 200, 640, 40
    w, s, b = _mats(dev, n, k, bits)
    bias = (torch.randn(n, device=dev) * 0.02).to(torch.bfloat16)
    base = _x(dev, m, k)
    padded = torch.zeros((m, k + 8), device=dev, dtype=torch.bfloat16)
    padded[:, :k] = base
    shifted = torch.zeros((m, k + 3), device=dev, dtype=torch.bfloat16)
    shifted[:, 3:] = base
    views = {"plain": base, "leading dims": base.reshape(2, 20, k), "row stride": padded[:, :k],
             "misaligned": shifted[:, 3:], "transposed": base.t().contiguous().t()}
    for bb in (None, bias):
        lin = QuantizedLinear(w, s, b, bb, bits=bits)
        want = None
        for name, v in views.items():
            assert lin.wide_kernel(v), name
            y = lin(v)
            assert y.shape == (*v.shape[:-1], n) and y.dtype == torch.bfloat16
            _check(y, base, w, s, b, bits, bb, name)
            want = y.reshape(m, n) if want is None else want
            assert torch.equal(y.reshape(m, n), want), name


def test_calls_that_keep_the_torch_product(dev):
    """Other dtypes and anything autograd or a transform has to see."""
    from dspark_rocm.nn import QuantizedLinear

    w, s, b = _mats(dev, 64, 128, 8)
    lin = QuantizedLinear(w, s, b, bits=8)
    x = _x(dev, 32, 128)
    assert lin.wide_kernel(x) and lin.wide_kernel(x[:1]) and not lin.wide_kernel(x[:0])
    assert not lin.wide_kernel(x.half())
    assert not lin.wide_kernel(x.cpu()) and not lin.wide_kernel(x[:, :64])
    assert not QuantizedLinear(w, s.half(), b.half(), bits=8).wide_kernel(x)
    xg = x.clone().requires_grad_(True)
    assert not lin.wide_kernel(xg)
    lin(xg).float().sum().backward()
    assert xg.grad is not None and bool(torch.isfinite(xg.grad).all())
    with torch.no_grad():
        assert lin.wide_kernel(xg)
    with torch.autograd.forward_ad.dual_level():
        assert not lin.wide_kernel(x)
    y = torch.func.vmap(lin)(x.reshape(2, 16, 128))      # a transform sees 16 rows of a batched tensor
    assert y.shape == (2, 16, 64)
    with pytest.raises(RuntimeError):
        lin(x[:, :64])                                    # a wrong K is refused as before


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(40, 200, 192), (96, 640, 2048)])   # one slice, K slices
def test_infinities_and_nans_follow_the_dequantized_product(dev, m, n, k, bits):
    from dspark_rocm import ops, quant

    w, s, b = _mats(dev, n, k, bits)
    s[5] = 0
    b[5:7] = 0
    x = _x(dev, m, k)
    inf = float("inf")
    x[3, 5], x[7, 9], x[9, 1], x[11, 0], x[11, 64] = inf, -inf, float("nan"), inf, -inf
    got = ops.quantized_matmul_wide(x, w, s, b, bits=bits).float()
    want = (x.float() @ quant.dequantize(w, s, b, 64, bits).t()).to(torch.bfloat16).float()
    odd = ~torch.isfinite(want)
    assert bool(odd[[3, 7, 9, 11]].any(-1).all()) and torch.equal(~torch.isfinite(got), odd)
    assert torch.equal(torch.nan_to_num(got[odd], nan=7.0), torch.nan_to_num(want[odd], nan=7.0))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(40, 200, 192), (96, 640, 2048)])
def test_infinite_weights_beside_infinite_rows(dev, m, n, k, bits):
    """A weight that is infinite too meets the row's finite values: an infinity of either sign, or a NaN."""
    from dspark_rocm import ops, quant

    w, s, b = _mats(dev, n, k, bits)
    inf = float("inf")
    b[8, 1], b[9, 1], s[130, 0] = -inf, inf, inf
    s[8:10, 0], b[8:10, 0] = 0, 1
    x = _x(dev, m, k)
    x[2:8, 64:128] = x[2:8, 64:128].abs()
    x[3, 5], x[7, 9], x[5, 70] = inf, -inf, inf
    got = ops.quantized_matmul_wide(x, w, s, b, bits=bits).float()
    want = (x.float() @ quant.dequantize(w, s, b, 64, bits).t()).to(torch.bfloat16).float()
    odd = ~torch.isfinite(want)
    assert bool(want[2, 8] == -inf) and bool(want[2, 9] == inf) and bool(want[3, 8].isnan())
    assert torch.equal(~torch.isfinite(got), odd)
    assert torch.equal(torch.nan_to_num(got[odd], nan=7.0), torch.nan_to_num(want[odd], nan=7.0))


def test_capture_and_replay(dev):
    """A captured product replays on new inputs (its workspace is the graph's own)."""
    from dspark_rocm.nn import QuantizedLinear

    w, s, b = _mats(dev, 512, 2048, 4)
    lin = QuantizedLinear(w, s, b, bits=4)
    x = _x(dev, 100, 2048)
    lin(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = lin(x)
    for seed in (5, 6, 7):
        x.copy_(_x(dev, 100, 2048, seed))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, lin(x))


def test_function_transforms_keep_the_torch_product(dev):
    """A map over several weights, whose tensors have no data pointer, and one over rows."""
    from dspark_rocm.nn import QuantizedLinear

    mats = [_mats(dev, 96, 128, 8, seed=i) for i in range(2)]
    lin = QuantizedLinear(*mats[0], bits=8)
    x = _x(dev, 20, 128)
    w = torch.stack([m[0] for m in mats])
    out = torch.vmap(lambda w: torch.func.functional_call(lin, {"weight": w}, (x,)))(w)
    for i in range(2):
        _check(out[i], x, w[i], *mats[0][1:], 8)
    _check(torch.vmap(lin)(x), x, *mats[0], 8)


def _us(f):
    f()
    best = float("inf")
    for _ in range(3):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3)
    return best


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(70, 300, 1088), (96, 5120, 2048), (300, 8192, 1024)])   # also one slice, K slices
def test_infinite_rows_cost_no_more_than_their_terms(dev, m, n, k, bits):
    """An infinity in every row: each output is its term (a NaN where the weight is zero), and the call
    stays within 20 times one without (about 1.3 measured; a whole product per output took 1000)."""
    from dspark_rocm import ops, quant

    w, s, b = _mats(dev, n, k, bits)
    s[5], b[5] = 0, 0
    x = _x(dev, m, k)
    at = torch.arange(m, device=dev) * 7 % k
    x2 = x.clone()
    x2[torch.arange(m, device=dev), at] = float("inf")
    call = lambda x: ops.quantized_matmul_wide(x, w, s, b, bits=bits)  # noqa: E731
    got, deq = call(x2).float(), quant.dequantize(w, s, b, 64, bits)
    want = float("inf") * deq[:, at].t()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
    assert _us(lambda: call(x2)) <= 20 * _us(lambda: call(x)) + 100


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(40, 200, 192), (96, 640, 2048)])
def test_factored_sums_that_overflow_are_the_plain_product(dev, m, n, k, bits):
    """Inputs near the end of the range, whose products with whole fields overflow."""
    from dspark_rocm import ops

    w, s, b = _mats(dev, n, k, bits)
    x = _x(dev, m, k)
    x[3, 5], x[9, 17], x[9, 18] = 2.0 ** 125, 2.0 ** 124, -(2.0 ** 124)
    ref, _ = _reference(x, w, s, b, bits)
    assert float(ref.abs().max()) < 2.0 ** 127
    got = ops.quantized_matmul_wide(x, w, s, b, bits=bits)
    big = [3, 9]
    deq = (x[big].double().abs() @ (_reference(torch.eye(k, device=dev), w, s, b, bits)[0]).abs())
    assert bool(((got[big].double() - ref[big]).abs() <= 2.0 ** -8 * ref[big].abs() + k * 2.0 ** -23 * deq).all())
    keep = torch.ones(m, dtype=torch.bool, device=dev)
    keep[big] = False
    _check(got[keep], x[keep], w, s, b, bits)


def test_rows_beyond_one_launch_keep_the_torch_product(dev):
    from dspark_rocm.nn import QuantizedLinear

    lin = QuantizedLinear(*_mats(dev, 8, 64, 8), bits=8)
    x = _x(dev, 1, 64)
    assert lin.wide_kernel(x.expand(1 << 23, 64)) and not lin.wide_kernel(x.expand((1 << 23) + 1, 64))
