"""The selection and sliding branches as one node whose backward sums their gradients in the kernels (nsa_dense_bwd_accumulate), against the
two branches by themselves."""

import pytest
import torch

from tests.util import causal_random_selection

pytestmark = pytest.mark.gpu
DEV = "cuda"


# ragged lengths, one tile, both head widths, groups of 1 and 8, a window longer than the sequence
@pytest.mark.parametrize("b,hq,hk,n,d,B,S,window,gated", [(2, 4, 2, 200, 64, 16, 3, 7, False), (1, 8, 1, 333, 128, 64, 2, 64, True), (1, 2, 2, 64, 64, 32, 1, 500, True),
                                                         (2, 8, 4, 1030, 64, 16, 4, 64, False), (1, 4, 2, 1, 128, 16, 1, 3, False)])
def test_gradients_are_the_sum_of_the_branches(b, hq, hk, n, d, B, S, window, gated):
    """The separate branches' gradients are each rounded to bf16 and added in bf16, the node's are one of them rounded plus the other in
    fp32 with one rounding: they differ by at most the other's rounding and those of the two sums, 2^-9 of each value's magnitude."""
    from native_sparse_attention_pytorch_amd import ops
    print(b, hq, hk, n, d, B, S, window, flush=True)
    g = torch.Generator().manual_seed(n)
    r = lambda h: (torch.randn(b, h, n, d, generator=g) * d ** -0.25).to(DEV, torch.bfloat16)
    q, k, v = (t.requires_grad_() for t in (r(hq), r(hk), r(hk)))
    douts = [r(hq), r(hq)]
    idx, live = (t.to(DEV) for t in causal_random_selection(b, hk, n, B, S, seed=5))
    gates = torch.ones(idx.shape, device=DEV, requires_grad=True) if gated else None
    leaves = [q, k, v] + ([gates] if gated else [])
    both = ops.select_and_slide(q, k, v, B, idx, live, gates, window)
    alone = ops.native_sparse_attend(q, k, v, B, idx, live, sel_scale=gates), ops.sliding_attend(q, k, v, window)
    assert all(torch.equal(x, y) for x, y in zip(both, alone))
    first = torch.autograd.grad(alone[0], leaves, douts[0], retain_graph=True)
    second = torch.autograd.grad(alone[1], leaves[:3], douts[1], retain_graph=True)
    got = torch.autograd.grad(both, leaves, douts, retain_graph=True)
    for x, s, t in zip(got, first, second):
        s, t = s.float(), t.float()
        assert ((x.float() - (s + t)).abs() <= 2 ** -8 * ((s + t).abs() + t.abs()) + 1e-30).all()
    if gated:
        assert torch.equal(got[3], first[3])
    # either branch by itself
    assert all(torch.equal(x, y) for x, y in zip(torch.autograd.grad(both[0], leaves, douts[0], retain_graph=True), first))
    assert all(torch.equal(x, y) for x, y in zip(torch.autograd.grad(both[1], leaves[:3], douts[1]), second))


def test_what_the_node_does_not_take():
    from native_sparse_attention_pytorch_amd import ops
    z = lambda h, d=64: torch.zeros(1, h, 32, d, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    idx = torch.zeros(1, 2, 32, 1, device=DEV, dtype=torch.int64)
    call = lambda q, k, B=16, i=idx: ops.select_and_slide(q, k, k, B, i, i.bool(), None, 8)
    assert call(z(4), z(2)) is not None
    assert call(z(6), z(2)) is None and call(z(4, 32), z(2, 32)) is None and call(z(4), z(2), B=128) is None
    assert call(z(4), z(2), i=idx.repeat_interleave(2, 1)) is None and call(z(4).float(), z(2).float()) is None
    with torch.no_grad():
        assert call(z(4), z(2)) is None


def test_gradients_of_gradients_are_refused():
    """The backward kernels' results are no functions of their operands to autograd: differentiating them again raises, where it would leave
    out what depends on them - also where only the inputs and not the incoming gradients ask for it."""
    from native_sparse_attention_pytorch_amd import ops
    b, hq, hk, n, B, S, window = 1, 4, 2, 100, 16, 2, 9
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(b, h, n, 64, generator=g).to(DEV, torch.bfloat16).requires_grad_() for h in (hq, hk, hk))
    idx, live = (t.to(DEV) for t in causal_random_selection(b, hk, n, B, S, seed=5))
    for name, f in (("node", lambda: sum(ops.select_and_slide(q, k, v, B, idx, live, None, window))),
                    ("selection", lambda: ops.native_sparse_attend(q, k, v, B, idx, live)),
                    ("window", lambda: ops.sliding_attend(q, k, v, window)),
                    ("compressed", lambda: ops.compress_attend(q, k[:, :, :8], v[:, :, :8], 2, 16, True)[0]),
                    ("in fp32", lambda: ops.fp32_value_bf16_grad(lambda *t: ops.dense_attend_f32(*(x.float() for x in t), 0, True, window)[0],
                                                                 lambda *t: ops.sliding_attend(*t, window), q, k, v))):
        plain = torch.autograd.grad(f().sum(), (q, k, v))
        first = torch.autograd.grad(f().sum(), (q, k, v), create_graph=True)
        assert all(torch.equal(x, y) for x, y in zip(plain, first)), name
        with pytest.raises(RuntimeError, match="cannot be differentiated again"):
            torch.autograd.grad(sum(t.float().square().sum() for t in (*first, q)), q)


def test_importance_scores_have_a_second_derivative():
    """They are linear in queries and compressed keys, and their gradient is made of matrix products: against float64."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(1)
    q, ck, cv = (torch.randn(1, h, m, 64, generator=g).to(DEV, torch.bfloat16).requires_grad_() for h, m in ((4, 100), (2, 7), (2, 7)))
    res = []
    for t, c in ((q, ck), (q.detach().double().requires_grad_(), ck.detach().double().requires_grad_())):
        if t.dtype == torch.bfloat16:
            logits = ops.compress_attend(t, c, cv, 1, 16, True, 16)[1]
        else:
            logits = ops.importance_logits_f32(t, c[:, :, 1:], 16, 16, True, True)
        seen = logits.masked_fill(logits.isinf(), 0.)
        dq, = torch.autograd.grad(seen.square().sum(), t, create_graph=True)
        res.append(torch.autograd.grad(dq.square().sum(), (t, c)))
    for x, y in zip(*res):
        assert ((x.double() - y).norm() <= 2 ** -6 * y.norm()).item()      # (operands, scores and results in bf16)
