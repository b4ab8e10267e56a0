"""nsa_skinny_linear (projections of a decode step, norm in front) against float64, at the edges of its tiles: rows around the groups
of 16, fewer K steps than waves, a K slice that is not a whole number of read-ahead rounds, features that are no multiple of 16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows,k,n,bias,norm", [
    (1, 32, 5, True, True), (1, 4096, 100, False, True), (2, 512, 16, False, True), (3, 6400, 33, True, True), (4, 1024, 17, False, False),
    (5, 96, 48, True, False), (8, 2080, 64, False, True), (16, 4064, 16, True, True), (17, 64, 31, False, True), (32, 2016, 40, True, True),
])
def test_skinny_linear(rows, k, n, bias, norm):
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(rows * k + n)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    wide, w = r(rows, k + 8), r(n, k) * k ** -0.5
    x = wide[:, :k]                                            # a strided row
    b, nw = (r(n) if bias else None), (r(k) if norm else None)
    assert ops.skinny_linear_supported(x.to(DEV), w.to(DEV))
    dev = lambda t: None if t is None else t.to(DEV)
    got = ops.skinny_linear(wide.to(DEV)[:, :k], dev(w), dev(b), dev(nw), 1e-6)
    torch.cuda.synchronize()
    xd = x.double()
    if norm:
        xd = (xd * (xd.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * nw.double()).to(torch.bfloat16).double()
    want = xd @ w.double().t() + (b.double() if bias else 0.)
    mag = xd.abs() @ w.double().abs().t()
    # the result's rounding 2^-9 |y|; a normed input may round the other way: 2^-8 of single products, at most 2^-8 / sqrt(k) x 8 of
    # their sum for independent ones; fp32 accumulation k 2^-24 of the sum of magnitudes
    tol = 2 ** -8 * want.abs() + (2 ** -5 * k ** -0.5 * want.abs().max() if norm else 0.) + k * 2 ** -24 * mag + 1e-6
    err = (got.double().cpu() - want).abs()
    assert (err <= tol).all(), (err - tol).max().item()


def test_skinny_limits():
    from native_sparse_attention_pytorch_amd import ops
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    assert not ops.skinny_linear_supported(z(33, 64), z(8, 64))
    assert not ops.skinny_linear_supported(z(1, 40), z(8, 40))
    assert not ops.skinny_linear_supported(z(16, 4096), z(8, 4096))
    with pytest.raises(RuntimeError):
        ops.skinny_linear(z(33, 64), z(8, 64))


@pytest.mark.parametrize("rows,k,n,act,res", [(1, 64, 40, "gelu", False), (7, 512, 33, "gelu", True), (20, 128, 16, "relu", True), (32, 64, 100, None, True)])
def test_skinny_epilogue(rows, k, n, act, res):
    """Activation and residual: as the layers they replace, each result rounded to bf16."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(rows + k + n)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    x, w, b, add = r(rows, 1, k), r(n, k) * k ** -0.5, r(n), r(rows, 1, n)
    got = ops.skinny_linear(x.to(DEV), w.to(DEV), b.to(DEV), act=act, residual=add.to(DEV) if res else None)
    torch.cuda.synchronize()
    y = x.double() @ w.double().t() + b.double()
    fn = {"gelu": torch.nn.functional.gelu, "relu": torch.relu, None: lambda t: t}[act]
    want = fn(y) + (add.double() if res else 0.)
    # the linear's rounding through a function of slope <= 1.13, the activation's own, the sum's
    tol = 2 ** -8 * (1.13 * y.abs() + fn(y).abs() + want.abs()) + 1e-6
    err = (got.double().cpu() - want).abs()
    assert got.shape == (rows, 1, n) and (err <= tol).all(), (err - tol).max().item()


@pytest.mark.parametrize("dtype, act", [(torch.bfloat16, None), (torch.bfloat16, "relu"), (torch.bfloat16, "gelu"), (torch.float32, None), (torch.float32, "relu")])
def test_what_is_not_finite_passes_the_epilogue(dtype, act):
    """NaN and infinities through the activations as the layers hand them on (relu(NaN) is NaN)."""
    from native_sparse_attention_pytorch_amd import ops
    fn = ops.skinny_linear if dtype == torch.bfloat16 else ops.linear_f32
    bias = torch.tensor([float("nan"), float("inf"), float("-inf"), 1., -1.])
    want = {None: lambda t: t, "relu": torch.relu, "gelu": torch.nn.functional.gelu}[act](bias.to(DEV, dtype)).expand(3, 5)
    got = fn(torch.zeros(3, 64, device=DEV, dtype=dtype), torch.zeros(5, 64, device=DEV, dtype=dtype), bias.to(DEV, dtype), act=act)
    torch.cuda.synchronize()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


def test_decode_layer_fills_the_newest_rows_and_reports_the_selection():
    """The whole-layer call: rows of the caches and of the open window, the selection's views, against the general path."""
    from native_sparse_attention_pytorch_amd import SparseAttention, ops
    torch.manual_seed(3)
    m = SparseAttention(dim=96, dim_head=64, heads=4, kv_heads=2, sliding_window_size=20, compress_block_size=8, compress_block_sliding_stride=4,
                        selection_block_size=8, num_selected_blocks=3, causal=True).to(DEV).bfloat16()
    x = torch.randn(2, 41, 96, device=DEV, dtype=torch.bfloat16)
    seen = []
    orig = ops.decode_step
    def spy(*a, **kw):
        r = orig(*a, **kw)
        seen.append((r[1].clone(), r[2].clone(), kw.get("layer") is not None))
        return r
    with torch.no_grad():
        _, cache = m(x[:, :40], return_cache=True)
        ops.decode_step = spy
        try:
            a, ca = m(x[:, 40:], cache=cache, return_cache=True)
            m._decode_whole = lambda *args, **kw: None
            b_, cb = m(x[:, 40:], cache=cache, return_cache=True)
        finally:
            ops.decode_step = orig
    torch.cuda.synchronize()
    assert seen[0][2] and not seen[1][2]
    assert torch.equal(seen[0][0], seen[1][0]) and torch.equal(seen[0][1], seen[1][1])
    flat = lambda c: [t for pair in (c[0], c[1][0], c[1][1]) for t in pair]
    assert torch.equal(a, b_) and all(torch.equal(s, t) for s, t in zip(flat(ca), flat(cb)))
