"""The launches an fp32 layer on a few tokens shares (norm + two projections, two networks, gate + output projection, compressed branch +
window, importance scores + top-k) against the operators and kernels they replace.

Bounds: sums of k products in another order, (k / 2 + 8) 2^-24 of the magnitudes added up (fp32 matrix instructions: one rounding per
two products, eight partial sums); attention 1e-5 + 1e-5 |value| as everywhere."""
import math

import pytest
import torch
import torch.nn.functional as F

from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _r(*s, seed=0, scale=1.):
    return (torch.randn(*s, generator=torch.Generator().manual_seed(seed + s[-1])) * scale).to(DEV)


def _close(y, x, w, b, act=None):
    k = x.shape[-1]
    want, size = F.linear(x.double(), w.double(), None if b is None else b.double()), F.linear(x.double().abs(), w.double().abs())
    size = size + (0 if b is None else b.double().abs())
    want = want.relu() if act else want
    assert ((y.double() - want).abs() <= (k / 2 + 8) * 2 ** -24 * size).all()


@pytest.mark.parametrize("norm", ["none", "ones", "weight"])
@pytest.mark.parametrize("lead,k,n,n2", [((2, 31), 512, 1536, 24), ((33,), 8, 1, 40), ((1, 256), 256, 200, 33), ((1,), 512, 64, 64)])
def test_two_projections(lead, k, n, n2, norm):
    from native_sparse_attention_pytorch_amd import ops
    x, nw = _r(*lead, k), _r(k, seed=5) if norm == "weight" else None
    first, second = (_r(n, k, seed=1, scale=k ** -0.5), None), (_r(n2, k, seed=2, scale=k ** -0.5), _r(n2, seed=3))
    eps = None if norm == "none" else 1e-3
    got = ops.linear_pair_f32(x, first, second, nw, eps)
    xn = x.double()
    if eps is not None:
        xn = F.rms_norm(xn, (k,), None if nw is None else nw.double(), eps)
    for y, (w, b) in zip(got, (first, second)):
        assert y.shape == (*lead, w.shape[0])
        _close(y, xn, w, b)
    x2 = _r(*lead, k, seed=7)
    got = ops.linear_pair_f32(x, first, second, x2=x2, act="relu")
    _close(got[0], x, *first, act="relu")
    _close(got[1], x2, *second, act="relu")


def test_norms_that_overflow_or_are_not_finite():
    """As the layers: a row whose squares overflow is zero after its norm, one with an infinity or NaN is NaN."""
    from native_sparse_attention_pytorch_amd import ops
    x, w = _r(40, 64), _r(16, 64, seed=1)
    x[3], x[4, 5], x[5, 6], x[6] = 1e37, math.inf, math.nan, 0.
    w[:] = w.abs()
    got = ops.linear_pair_f32(x, (w, None), (w, None), None, 1e-6)[0]
    want = F.linear(F.rms_norm(x, (64,), None, 1e-6), w)
    assert torch.equal(got.isnan(), want.isnan())
    assert_close(got.nan_to_num(0.), want.nan_to_num(0.), 1e-5, 1e-5, "rows")


def test_projections_a_pair_does_not_take():
    from native_sparse_attention_pytorch_amd import ops
    x, w, b = _r(40, 64), _r(16, 64, seed=1), _r(16, seed=2)
    ok = (w, b)
    assert ops.linear_pair_f32(x, ok, ok) is not None
    for other in ((w.bfloat16(), b.bfloat16()), (w.t().contiguous().t(), b), (w, b[:1]), (_r(16, 32), b), (w.cpu(), b.cpu()), (_r(9000, 64), None)):
        assert ops.linear_pair_f32(x, ok, other) is None and ops.linear_pair_f32(x, other, ok) is None
    assert ops.linear_pair_f32(_r(300, 64), ok, ok) is None
    assert ops.linear_pair_f32(x, ok, ok, x2=_r(39, 64)) is None
    assert ops.linear_pair_f32(x, ok, ok, _r(32), 1e-6) is None
    assert ops.linear_pair_f32(_r(1 + 40 * 64)[1:].view(40, 64), ok, ok) is None


@pytest.mark.parametrize("b,h,n,d,out", [(2, 8, 31, 64, 512), (1, 2, 33, 20, 7), (3, 4, 1, 128, 200)])
def test_gate_and_output_projection(b, h, n, d, out):
    from native_sparse_attention_pytorch_amd import ops
    logits, w, bias = _r(b, n, 3 * h), _r(out, h * d, seed=1, scale=(h * d) ** -0.5), _r(out, seed=2)
    c, s = _r(b, h, n, d, seed=3), _r(b, h, n, d, seed=4)
    f = _r(b, n, h, d, seed=5).transpose(1, 2)                    # (token-major)
    got = ops.gate_linear_f32(logits, c, f, s, w, bias)
    g = logits.double().sigmoid().view(b, n, h, 3).permute(0, 2, 1, 3)
    merged = sum(g[..., t:t + 1] * x.double() for t, x in enumerate((c, f, s))).permute(0, 2, 1, 3).reshape(b, n, h * d)
    _close(got, merged, w, bias)


@pytest.mark.parametrize("b,hq,hk,n,d,stride,mem,window,causal", [
    (2, 8, 8, 31, 64, 2, 1, 2, False), (1, 8, 4, 130, 64, 8, 2, 64, True), (1, 6, 2, 3, 100, 4, 1, 16, True), (2, 16, 2, 300, 128, 16, 1, 40, True),
    (8, 8, 8, 200, 64, 8, 1, 32, True),                           # many queries: the tile kernel, a launch each
])
def test_compressed_branch_and_window(b, hq, hk, n, d, stride, mem, window, causal):
    from native_sparse_attention_pytorch_amd import ops
    q, rq, k, v = _r(b, hq, n, d), _r(b, hq, n, d, seed=1), _r(b, hk, n, d, seed=2), _r(b, hk, n, d, seed=3)
    ck, cv, m = _r(b, hk, n // stride, d, seed=4), _r(b, hk, n // stride, d, seed=5), _r(2, hk, mem, d, seed=6)
    c_out, s_out = ops.compress_window_f32(q, ck, cv, m, stride, rq, k, v, window, causal)
    assert torch.equal(c_out, ops.compress_attend_f32(q, ck, cv, m, stride, causal))
    assert torch.equal(s_out, ops.dense_attend_f32(rq, k, v, 0, causal, window)[0])


@pytest.mark.parametrize("share", [True, False])
@pytest.mark.parametrize("b,hq,hk,n,d,stride,B,k,causal,own", [
    (2, 8, 8, 31, 64, 2, 4, 2, False, True), (1, 16, 4, 1030, 64, 16, 64, 16, True, True), (2, 12, 4, 70, 20, 4, 4, 17, True, True),
    (3, 4, 1, 1, 128, 8, 16, 5, False, False), (1, 4, 2, 520, 100, 8, 8, 64, True, True),     # 64 and 65 blocks
    (1, 4, 2, 528, 64, 8, 8, 9, True, True),
])
def test_importance_and_selection(b, hq, hk, n, d, stride, B, k, causal, own, share):
    """The selection equals the one from float64 scores but where two blocks' probabilities agree to 1e-5."""
    from native_sparse_attention_pytorch_amd import ops
    nc = max(n, 40 * B) // stride if n == 1 else n // stride
    q, ck = _r(b, n, hq, d).transpose(1, 2), _r(b, hk, nc, d, seed=1)
    k = min(k, nc // (B // stride))
    vals, idx, fm = ops.importance_select_f32(q, ck, stride, B, share, causal, k, mask_own=own)
    logits = ops.importance_logits_f32(q.double(), ck.double(), stride, B, share, causal, mask_own=own)
    p = torch.cat((logits.new_full((*logits.shape[:-1], 1), -1e3), logits), dim=-1).softmax(-1)[..., 1:]
    want, at = p.topk(k, dim=-1)
    assert_close(vals, want, 1e-6, 1e-5, "values")
    assert_close(p.gather(-1, idx.long()), want, 1e-6, 1e-5, "chosen")
    assert (idx.sort(-1).values.diff(dim=-1) > 0).all()
    assert torch.equal(fm, vals > 1e-10)
    dead = want == 0                                              # nothing left to choose: the lowest blocks in order
    assert torch.equal(dead, vals == 0)


@pytest.mark.parametrize("b,n,share", [(6, 1024, True), (3, 1024, False), (2, 2049, True)])
def test_importance_of_many_queries(b, n, share):
    """Above the lines the products are the library's."""
    from native_sparse_attention_pytorch_amd import ops
    q, ck = _r(b, 8, n, 64), _r(b, 4, n // 8, 64, seed=1)
    for x, y in zip(ops.importance_select_f32(q, ck, 8, 32, share, True, 4), ops.importance_topk_f32(q, ck, 8, 32, share, True, 4)):
        assert torch.equal(x, y)


def test_importance_of_many_queries_of_a_waiting_host():
    """The kernel's line where the host's time counts, against the GEMM's scores; and above it."""
    from native_sparse_attention_pytorch_amd import ops
    for b, same in ((8, False), (9, True)):
        q, ck = _r(b, 8, 1024, 64), _r(b, 4, 128, 64, seed=1)
        args = (q, ck, 8, 16, True, True, 4)
        got, want = ops.importance_select_f32(*args, host_bound=True), ops.importance_topk_f32(*args)
        assert_close(got[0], want[0], 1e-6, 1e-5, "values")
        assert (not same) or all(torch.equal(x, y) for x, y in zip(got, want))


def test_scores_that_are_not_numbers():
    from native_sparse_attention_pytorch_amd import ops
    q, ck = _r(1, 4, 50, 64), _r(1, 2, 25, 64, seed=1)
    q[0, 1, 7] = math.nan
    vals, idx, fm = ops.importance_select_f32(q, ck, 2, 4, True, True, 3)
    assert vals[0, 0, 7].isnan().all() and not fm[0, 0, 7].any() and idx[0, 0, 7].tolist() == [0, 1, 2]
    assert not vals[0, 1].isnan().any() and not vals[0, 0, 8:].isnan().any()


@pytest.mark.parametrize("kw", [
    dict(heads=8, sliding_window_size=2, compress_block_size=4, compress_block_sliding_stride=2, selection_block_size=4, num_selected_blocks=2),
    dict(heads=8, kv_heads=4, causal=True, sliding_window_size=8, compress_block_size=8, compress_block_sliding_stride=4, selection_block_size=8,
         num_selected_blocks=3, num_compressed_mem_kv=2),
    dict(heads=8, kv_heads=2, causal=True, sliding_window_size=8, compress_block_size=8, compress_block_sliding_stride=8, selection_block_size=8,
         num_selected_blocks=0, query_heads_share_selected_kv=False),
])
@pytest.mark.parametrize("n", [1, 31, 70])
def test_layer(kw, n):
    """The layer against itself with a hook on every part, which sends it through the layers one by one."""
    from native_sparse_attention_pytorch_amd import SparseAttention
    torch.manual_seed(n)
    m = SparseAttention(dim=256, dim_head=64, **kw).to(DEV)
    with torch.no_grad():
        for p in m.parameters():
            p += 0.05 * torch.randn_like(p)
        x = _r(2, n, 256)
        causal = kw.get("causal", False)
        got = m(x, return_cache=causal)
        calls = []
        handles = [layer.register_forward_hook(lambda *a: calls.append(1)) for layer in (m.norm, m.to_qkv, m.combine_heads, m.to_strategy_combine[0],
                                                                                         m.k_compress[1], m.v_compress[1])]
        want = m(x, return_cache=causal)
        for h in handles:
            h.remove()
    assert len(calls) == 6
    flat = lambda t: [t] if torch.is_tensor(t) else [u for s in t for u in flat(s)]
    for a, b in zip(flat(got), flat(want)):
        assert_close(a, b, 1e-5, 1e-5, "layer")
