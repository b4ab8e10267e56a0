"""fp32 products on the bf16 matrix instructions (operands split in three) are no further from float64 than fp32 multiplications and
fused multiply-adds are, also where few of them are summed."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _normal(*s, seed=0):
    return torch.randn(*s, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)


def _few(x, nonzero, seed=9):
    """x with `nonzero` values of each row left, anywhere in it."""
    return x * (torch.rand(x.shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).argsort(-1) < nonzero)


@pytest.mark.parametrize("k,nonzero", [(4, 4), (64, 1), (64, 2), (36, 4), (64, 8), (256, 256)])
def test_projections(k, nonzero):
    """One product: the rounding of an fp32 number, 2^-24, and those of the small sums, 2^-31 of it each; more: no more in the mean than
    the library's fused multiply-adds."""
    from native_sparse_attention_pytorch_amd import ops
    x, w = _few(_normal(512, k), nonzero), _normal(768, k, seed=1)
    want, size = F.linear(x.double(), w.double()), F.linear(x.double().abs(), w.double().abs())
    error = lambda y: ((y.double() - want) / size).nan_to_num(0.)
    got, library = error(ops._gemm_f32(x, w, None)), error(F.linear(x, w))
    if nonzero == 1:
        assert got.abs().max().item() <= 2 ** -24 + 2 ** -29
    assert got.norm() <= library.norm() * (1.01 if nonzero == 1 else 1.)


@pytest.mark.parametrize("hq,hk,d", [(16, 4, 64), (32, 8, 128)])
def test_scores(hq, hk, d):
    """A window of the query's own key: the log-sum-exp is the score, with one feature in the query a single product; at d = 128 times a
    scale that is no power of two: its own rounding, half of one at most, and the result's."""
    from native_sparse_attention_pytorch_amd import ops
    n = 2048
    q, k, v = _few(_normal(2, hq, n, d), 1), _normal(2, hk, n, d, seed=1), _normal(2, hk, n, d, seed=2)
    out, lse = ops.dense_attend_f32(q, k, v, 0, True, 0)
    want = (q.double() * k.double().repeat_interleave(hq // hk, 1)).sum(-1) * d ** -0.5
    bound = (2 ** -24 + 2 ** -29) * (1 if d == 64 else 2.5)
    assert ((lse.double() - want).abs() <= bound * want.abs()).all()
    assert torch.equal(out, v.repeat_interleave(hq // hk, 1))


@pytest.mark.parametrize("hq,hk,d", [(16, 4, 64), (32, 8, 128)])
def test_log_sum_exp(hq, hk, d):
    """Of a window of 512 keys: its own rounding and that of the logarithm in it, numbers of 4 to 8, are 2.0e-7 in the mean; fp32
    products and exponentials (v_mfma_f32, expf) were 2.8e-7 and 2.9e-7 off."""
    from native_sparse_attention_pytorch_amd import ops
    n = 2048
    q, k, v = _normal(2, hq, n, d), _normal(2, hk, n, d, seed=1), _normal(2, hk, n, d, seed=2)
    _, lse = ops.dense_attend_f32(q, k, v, 0, True, 512)
    i, j = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    sim = q.double() @ k.double().repeat_interleave(hq // hk, 1).transpose(-1, -2).contiguous() * d ** -0.5
    want = sim.masked_fill_((j > i) | (i - j > 512), -torch.inf).logsumexp(-1)
    assert (lse.double() - want).square().mean().sqrt() <= 2.95e-7


@pytest.mark.parametrize("d", [64, 128])
def test_values_near_the_largest(d):
    """A value of 3e38 behind a score that is the largest of its row by 2^7 in weight: no weight of a sum is above 1."""
    from native_sparse_attention_pytorch_amd import ops
    b, hq, hk, n, B = 4, 8, 4, 320, 64
    q, k, v = torch.zeros(b, hq, n, d, device=DEV), torch.zeros(b, hk, n, d, device=DEV), torch.zeros(b, hk, n, d, device=DEV)
    q[..., 0] = d ** 0.5
    k[:, :, 40, 0], v[:, :, 40, 3] = 5., 3e38
    idx = torch.zeros(b, hk, n, 1, dtype=torch.int32, device=DEV)
    msk = (torch.arange(n, device=DEV) >= B)[None, None, :, None].expand(b, hk, n, 1).contiguous()
    i, j = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    weight = (j == 40) * torch.exp(torch.tensor(5., dtype=torch.double, device=DEV)) + (j != 40)
    for got, seen in ((ops.dense_attend_f32(q, k, v, 0, True, n)[0], j <= i),
                      (ops.native_sparse_attend_f32(q, k, v, B, idx, msk), (j <= i) & ((j // B == i // B) | (j < B)))):
        w = weight * seen
        want = torch.zeros(n, d, dtype=torch.double, device=DEV)
        want[:, 3] = (w / w.sum(-1, keepdim=True))[:, 40] * v[0, 0, 40, 3].double()
        assert ((got.double() - want).abs() <= 1e-5 * want).all()
