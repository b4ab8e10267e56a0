"""The backward walk with one wave per tile (33 .. 64 keys a block, 128 features, four heads a group or more): where its tiles, units,
work-groups and heads begin and end, against the CPU oracle and against the walks that a call with gate gradients takes."""

import pytest
import torch

from tests.test_select_gpu import test_select_fwd_bwd_matches_oracle as check
from tests.util import causal_random_selection

pytestmark = pytest.mark.gpu


# batch, heads, kv heads, tokens, d, block, slots
@pytest.mark.parametrize("b,hq,hk,n,d,B,S", [
    (1, 4, 1, 1, 128, 64, 1),             # one row
    (1, 4, 1, 65, 128, 64, 1),            # a block of one key, tiles of one pair
    (1, 32, 1, 150, 128, 33, 5),          # 32 heads a group: a pair is a tile
    (2, 8, 2, 333, 128, 48, 3),           # blocks of 48 keys
    (1, 16, 2, 700, 128, 64, 12),         # units of 64 and 128 pairs, several to a block
    (35, 8, 2, 100, 128, 64, 2),          # 70 kv heads: more than a wave looks through at once
    (1, 8, 2, 4097, 128, 64, 4),
])
def test_against_the_oracle(b, hq, hk, n, d, B, S):
    check(b, hq, hk, n, d, B, S)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("layout", ["heads", "tokens", "sliced"])
@pytest.mark.parametrize("b,hq,hk,n,B,S", [(2, 16, 2, 509, 64, 4), (1, 4, 1, 1300, 40, 15)])
def test_against_the_other_walks(b, hq, hk, n, B, S, layout, causal):
    """Same blocks, same sums: what differs is the order of fp32 additions, which moves a bf16 result (or partial, or dS) by an ulp where it
    lies near the middle of two: 2^-8 of the few it does that to."""
    from native_sparse_attention_pytorch_amd import native_sparse_attend
    print(f"case {b} {hq} {hk} {n} {B} {S} {layout} {causal}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + S)

    def make(h):
        if layout == "tokens":
            t = torch.randn(b, n, h, 128, generator=g, device="cuda").transpose(1, 2)
        elif layout == "sliced":      # rows that start 16 bytes into wider ones
            t = torch.randn(b, h, n, 144, generator=g, device="cuda")
        else:
            t = torch.randn(b, h, n, 128, generator=g, device="cuda")
        t = (t * 128 ** -0.25).bfloat16()
        return t[..., 8:136] if layout == "sliced" else t

    q, k, v, do = make(hq), make(hk), make(hk), make(hq)
    idx, live = causal_random_selection(b, hk, n, B, S, seed=5)
    idx, live = idx.cuda(), live.cuda()
    grads = []
    for gates in (None, torch.ones(idx.shape, device="cuda", requires_grad=True)):
        leaves = [t.detach().requires_grad_() for t in (q, k, v)]
        out, lse = native_sparse_attend(*leaves, B, idx, live, sel_scale=gates, include_block_causal=causal, return_lse=True)
        dead = torch.isinf(lse)                                     # (not causal: queries that select nothing)
        ((out.float() * do.float()).sum() + (0.1 * lse.masked_fill(dead, 0.)).sum()).backward()
        grads.append([t.grad.float() for t in leaves])
    torch.cuda.synchronize()
    for name, x, y, tol in zip("qkv", *grads, (2 ** -8, 2 ** -9, 2 ** -9)):
        assert torch.isfinite(x).all(), name
        err = ((x - y).norm() / y.norm()).item()
        assert err < tol, (name, err)


@pytest.mark.parametrize("hq,hk,n,S", [(32, 8, 1024, 16), (16, 2, 4100, 15), (8, 2, 1500, 4)])
def test_both_backwards_of_one_index(hq, hk, n, S):
    """The walks with and without gate gradients have unit tables of their own in an index: either reads its own, whichever ran before.
    (Tolerance: test_against_the_other_walks.)"""
    from native_sparse_attention_pytorch_amd import ops
    print(f"case {hq} {hk} {n} {S}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k, v, do = ((torch.randn(1, h, n, 128, generator=g, device="cuda") * 128 ** -0.25).bfloat16() for h in (hq, hk, hk, hq))
    idx, live = (t.cuda() for t in causal_random_selection(1, hk, n, 64, S, seed=7))
    out, lse, index = ops.select_fwd(q, k, v, idx, live, None, 64, True, 128 ** -0.5)
    runs = [ops.select_bwd(q, k, v, out, do, lse, idx, live, index, 64, True, 128 ** -0.5, gated)[:3] for gated in (True, False, True)]
    torch.cuda.synchronize()
    for name, x, y, z, tol in zip("qkv", *runs, (2 ** -8, 2 ** -9, 2 ** -9)):
        assert torch.equal(x, z), name
        err = ((y.float() - x.float()).norm() / x.float().norm()).item()
        assert err < tol, (name, err)
