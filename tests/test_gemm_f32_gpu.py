"""fp32 projections of many rows by `nsa_gemm_f32` (operands split in three bf16 numbers) against float64.

Bound: a product loses at most 2^-22 of its magnitude, a sum at most 2^-24 of the magnitudes added up per rounding, of which there are
k / 16 in the leading sums (and as many within the sixteen, generously): (k / 8 + 8) 2^-24 sum |x w|."""
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _r(*s, seed=0, scale=1.):
    return (torch.randn(*s, generator=torch.Generator().manual_seed(seed + s[-1])) * scale).to(DEV)


def _check(y, x, w, b=None, act=None):
    k = x.shape[-1]
    want, size = F.linear(x.double(), w.double()), F.linear(x.double().abs(), w.double().abs())
    if b is not None:
        want, size = want + b.double(), size + b.double().abs()
    if act == "relu":
        want = want.relu()
    bad = (y.double() - want).abs() > (k / 8 + 8) * 2 ** -24 * size
    assert not bad.any(), (int(bad.sum()), bad.nonzero()[:4].tolist())


@pytest.mark.parametrize("m,n,k,act,bias", [
    (1, 1, 4, None, False),               # a tile of one element, less than one step
    (129, 127, 16, "relu", True),         # a row past a tile, one step
    (128, 257, 36, None, True),           # a column past two tiles, steps 2 and a quarter
    (200, 130, 2048, "relu", False),
    (33, 65, 500, None, True),
])
def test_against_float64(m, n, k, act, bias):
    from native_sparse_attention_pytorch_amd import ops
    x, w, b = _r(m, k), _r(n, k, seed=1, scale=k ** -0.5), _r(n, seed=2) if bias else None
    _check(ops._gemm_f32(x, w, b, act), x, w, b, act)
    x2, w2, b2 = _r(m, k, seed=3), _r(n, k, seed=4, scale=k ** -0.5), _r(n, seed=5) if bias else None
    y, y2 = ops._gemm_f32(x, w, b, act, (x2, w2, b2))
    _check(y, x, w, b, act)
    _check(y2, x2, w2, b2, act)


@pytest.mark.parametrize("spread", [0., 4.])       # the second: magnitudes from 1e-7 to 1e7
def test_no_larger_error_than_the_library(spread):
    from native_sparse_attention_pytorch_amd import ops
    x, w = _r(600, 1024) * (spread * _r(600, 1024, seed=1)).exp(), _r(300, 1024, seed=2)
    want = F.linear(x.double(), w.double())
    error = lambda y: float((y.double() - want).norm() / want.norm())
    assert error(ops._gemm_f32(x, w, None)) <= error(F.linear(x, w))


def test_what_is_not_finite_or_overflows():
    """As the library has it: row 3 infinite, row 7 NaN; the largest numbers of fp32 do not round up to infinity."""
    from native_sparse_attention_pytorch_amd import ops
    big = torch.finfo(torch.float32).max
    x, w = _r(64, 64), _r(64, 64, seed=1) * 0.01
    x[3, 5], x[7, 9], x[11], x[12, 2] = math.inf, math.nan, big, -big
    x[13, 0], w[5, 0] = 1e30, 1e30
    got, want = ops._gemm_f32(x, w, None), F.linear(x.double(), w.double())
    want = torch.where(want.abs() > big, want.sign() * math.inf, want)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    # (64 products, at most 2^-24 of the magnitudes for each of 16 roundings)
    size = F.linear(x.double().abs(), w.double().abs())
    assert ((got.double() - want).abs()[fine] <= 16 * 2 ** -24 * size[fine]).all()
    assert torch.equal(got[want.isinf()].sign().double(), want[want.isinf()].sign())


def test_which_projections_take_it(monkeypatch):
    from native_sparse_attention_pytorch_amd import ops
    taken = []
    kernel = ops._gemm_f32
    monkeypatch.setattr(ops, "_gemm_f32", lambda *a: taken.append(1) or kernel(*a))
    x, w = _r(2049, 64), _r(2048, 64, seed=1)                 # 17 x 16 tiles
    b = _r(2048, seed=2)

    def served(f):
        taken.clear()
        y = f()
        return bool(taken), y

    with torch.no_grad():
        hit, y = served(lambda: ops.linear(x[None], w, b))
        assert hit and y.shape == (1, 2049, 2048)
        _check(y[0], x, w, b)
        for xx, ww, bb in ((x[:1900], w, b), (x[:, :62], w[:, :62], b), (x.bfloat16(), w.bfloat16(), b.bfloat16()), (x.t().contiguous().t(), w, b),
                           (x, w.t().contiguous().t(), b), (x, w, b[:1]), (_r(1 + 2049 * 64)[1:].view(2049, 64), w, b)):
            hit, y = served(lambda: ops.linear(xx, ww, bb))
            assert not hit and torch.equal(y, F.linear(xx, ww, bb))
        with torch.autocast("cuda", torch.bfloat16):
            assert not served(lambda: ops.linear(x, w, b))[0]
        assert not served(lambda: torch.vmap(lambda t: ops.linear(t, w, b))(x[None]))[0]
        for bad in (_r(2048, 60), _r(2048, 64).bfloat16()):
            with pytest.raises(RuntimeError):
                ops.linear(x, bad)
    # under autograd: the value by the kernel, the gradients as ever, a second derivative too
    xg, wg = x.clone().requires_grad_(), w.clone().requires_grad_()
    hit, y = served(lambda: ops.linear(xg, wg, b))
    assert hit
    (gx,) = torch.autograd.grad(y.square().sum(), xg, create_graph=True)
    (gw,) = torch.autograd.grad(gx.sum(), wg)
    xr, wr = x.double().requires_grad_(), w.double().requires_grad_()
    (rx,) = torch.autograd.grad(F.linear(xr, wr, b.double()).square().sum(), xr, create_graph=True)
    (rw,) = torch.autograd.grad(rx.sum(), wr)
    for a, r in ((gx, rx), (gw, rw)):
        assert float(((a - r).norm() / r.norm()).detach()) < 1e-5


def test_both_compression_networks_in_one_launch(monkeypatch):
    from native_sparse_attention_pytorch_amd import SparseAttention, ops
    torch.manual_seed(0)
    layer = SparseAttention(dim=256, dim_head=64, heads=8, kv_heads=8, causal=True, sliding_window_size=32, compress_block_size=16,
                            compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2).to(DEV)
    kw, vw = _r(2, 8, 128, 16, 64), _r(2, 8, 128, 16, 64, seed=1)      # 2048 windows x 1024: 128 tiles each
    with torch.no_grad():
        pair = layer._compress_both(kw, vw)
        alone = layer.k_compress(kw), layer.v_compress(vw)
    for a, b in zip(pair, alone):
        assert float((a - b).norm() / b.norm()) < 1e-6
    seen = []
    handle = layer.v_compress[2].register_forward_hook(lambda *a: seen.append(1))
    with torch.no_grad():
        layer._compress_both(kw, vw)
    handle.remove()
    assert seen


def test_operands_of_another_device(monkeypatch):
    """Where the current device is another one (told to the rules only), the library makes the products: a launch by address would go to a
    stream of the wrong device."""
    from native_sparse_attention_pytorch_amd import _lib, ops
    x, w, few = _r(2049, 64), _r(2048, 64, seed=1), _r(4, 64)
    h = lambda *s: _r(*s).bfloat16().requires_grad_()
    net = h(256, 128), h(256), h(128, 256), h(128)
    y, dy = h(700, 128), h(700, 64).detach()
    with torch.no_grad():
        assert ops.gemm_f32_supported(x, w) and ops.linear_f32_supported(few, w[:64]) and ops._wgrad_supported(dy, y, y.dtype)
    assert ops.mlp_supported("relu", [y], [net])
    other = torch.cuda.current_device() + 1
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: other)
    monkeypatch.setattr(_lib, "lib", lambda: pytest.fail("launched"))
    assert not ops.mlp_supported("relu", [y], [net])
    with torch.no_grad():
        assert not ops._wgrad_supported(dy, y, y.dtype)
        for t, v in ((x, w), (few, w[:64])):
            assert torch.equal(ops.linear(t, v), F.linear(t, v))
