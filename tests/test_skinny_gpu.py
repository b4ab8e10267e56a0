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
