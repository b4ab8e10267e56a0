"""The fp32 forward kernels at the edges of their tiles, against float64: the kernel for many queries (32 rows x 32 keys) and the
kernel for one query per wave or per work-group (64 gathered keys), groups of every size, head dimensions that are no multiple of
a tile, key counts one off a tile, more slots than a wave has lanes, padding keys, decode offsets.

Bound: 1e-5 + 1e-5 |value|, the reference's own fp32 tolerance (tests/test_sparse_attn.py:86).  A logit is a sum of d <= 128
products, an output a weighted mean: their fp32 errors are below (d + 2) 2^-24 |q||k| / sqrt(d) ~ 1e-5 for unit normal inputs at
the very worst and ~1e-6 in practice."""
import math

import pytest
import torch

from oracle import nsa_oracle as O
from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("b,hq,hk,n,d,mode,causal,win,st,mem,qoff", [
    (1, 8, 1, 33, 64, 0, True, 31, 1, 0, 0),          # few queries: a work-group per query, window + 1 = half a tile
    (1, 5, 1, 1, 20, 0, True, 512, 1, 0, 700),        # a decode step: one query, 513 keys = 8 tiles + 1
    (2, 6, 2, 3, 128, 1, True, 0, 4, 64, 600),        # 64 memory slots: the first tile holds nothing else
    (2, 3, 3, 700, 64, 0, True, 63, 1, 0, 0),         # 4200 (query, kv head) pairs: the tile kernel, groups of 1
    (1, 20, 4, 1100, 100, 0, False, 40, 1, 0, 0),     # groups of 5: rows of a wave end inside a query
    (3, 16, 8, 181, 128, 1, True, 0, 16, 1, 0),       # 4344 pairs, strided prefixes that begin empty, d = 128
    (1, 8, 8, 513, 36, 1, False, 0, 5, 31, 0),        # 32-key tiles that end on a memory slot + 102 keys
])
def test_interval_masks(b, hq, hk, n, d, mode, causal, win, st, mem, qoff):
    from native_sparse_attention_pytorch_amd.ops import dense_attend_f32
    total = n + qoff
    keys = total if mode == 0 else total // st
    q, k, v = _rand((b, hq, n, d), n), _rand((b, hk, mem + keys, d), d), _rand((b, hk, mem + keys, d), 7)
    i, j = torch.arange(n)[:, None] + qoff, torch.arange(keys)[None, :]
    if mode == 0:
        see = (j <= i) & (i - j <= win) if causal else (i - j).abs() <= win
    else:
        see = torch.cat((torch.ones(n, mem, dtype=torch.bool), (j + 1) * st <= i if causal else torch.ones(n, keys, dtype=torch.bool)), dim=1)
    g = hq // hk
    kd, vd = k.double().repeat_interleave(g, 1), v.double().repeat_interleave(g, 1)
    sim = (q.double() @ kd.transpose(-1, -2) * d ** -0.5).masked_fill(~see, float("-inf"))
    got, lse = dense_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), mode, causal, win, st, mem, q_offset=qoff)
    torch.cuda.synchronize()
    assert_close(got, sim.softmax(-1) @ vd, 1e-5, 1e-5, "out")
    assert_close(lse, sim.logsumexp(-1), 1e-5, 1e-5, "lse")


@pytest.mark.parametrize("b,hq,hk,n,d,B,S,causal,qoff", [
    (1, 4, 1, 65, 64, 1, 3, True, 0),                 # blocks of one key
    (1, 7, 1, 64, 60, 5, 70, True, 0),                # more slots than lanes, blocks that straddle tiles, groups of 7
    (2, 2, 2, 1100, 128, 64, 2, True, 0),             # 4400 queries: a query per wave, groups of 1
    (1, 12, 4, 530, 64, 48, 4, False, 0),             # padding keys: the last block has 2 rows; groups of 3
    (1, 4, 2, 2, 128, 100, 3, True, 998),             # decode steps, blocks above a tile
    (1, 4, 2, 40, 64, 16, 0, True, 0),                # no slots: the own block only
])
def test_selection(b, hq, hk, n, d, B, S, causal, qoff):
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    total = n + qoff
    q, k, v = _rand((b, hq, n, d), n), _rand((b, hk, total, d), d), _rand((b, hk, total, d), 7)
    g = torch.Generator().manual_seed(B)
    W = math.ceil(total / B)
    idx = torch.randint(0, W, (b, hk, n, S), generator=g)
    msk = torch.rand(b, hk, n, S, generator=g) > 0.3
    if S and not causal:
        msk[..., 0] = True                            # (a query with no live slot at all has its own test)
        idx[..., 0] = W - 1                           # the block that reaches past the end
    want, want_lse = O.select_attend(q.double(), k.double(), v.double(), idx, msk, B, causal=causal, return_lse=True, q_offset=qoff)
    got, lse = native_sparse_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), B, idx.to(DEV), msk.to(DEV), include_block_causal=causal, return_lse=True,
                                        q_offset=qoff)
    torch.cuda.synchronize()
    assert_close(got, want, 1e-5, 1e-5, "out")
    assert_close(lse, want_lse, 1e-5, 1e-5, "lse")


def _overflowing(shape, rows, seed):
    """Keys whose first `rows` rows score -inf in fp32 against queries with 1e20 as their first feature."""
    k = _rand(shape, seed)
    k[..., 0] = 0
    k[..., :rows, 0] = -1e30
    return k


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [300, 2100])                       # a work-group per query; a wave per query
def test_selected_blocks_that_score_minus_infinity(n, d):
    """The first tile of every query holds such a block alone: it weighs nothing and the blocks after it are attended as ever."""
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    q, k, v = _rand((1, 4, n, d), 1), _overflowing((1, 1, n, d), 64, 2), _rand((1, 1, n, d), 3)
    q[..., 0] = 1e20
    idx = torch.stack((torch.zeros(n, dtype=torch.long), 1 + torch.arange(n) % (n // 64)), -1)[None, None]
    msk = torch.ones_like(idx, dtype=torch.bool)
    want = O.select_attend(q.double(), k.double(), v.double(), idx, msk, 64, causal=True)
    got = native_sparse_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), 64, idx.to(DEV), msk.to(DEV))
    torch.cuda.synchronize()
    assert_close(got, want, 1e-5, 1e-5, "out")


@pytest.mark.parametrize("n,win", [(420, 130), (1400, 130), (4200, 40)])      # a work-group, a wave per query; 32-row tiles
def test_interval_keys_that_score_minus_infinity(n, win):
    from native_sparse_attention_pytorch_amd.ops import dense_attend_f32
    q, k, v = _rand((1, 2, n, 64), 1), _overflowing((1, 1, n, 64), 300, 2), _rand((1, 1, n, 64), 3)
    q[..., 0] = 1e20
    got = dense_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), 0, True, win)[0][:, :, 300:340]      # (queries with at least one other key)
    torch.cuda.synchronize()
    i, j = torch.arange(300, 340)[:, None], torch.arange(n)[None, :]
    sim = (q[:, :, 300:340].double() @ k.double().transpose(-1, -2) / 8).masked_fill((j > i) | (i - j > win), float("-inf"))
    assert_close(got, sim.softmax(-1) @ v.double(), 1e-5, 1e-5, "out")


@pytest.mark.parametrize("d", [64, 100, 128])
@pytest.mark.parametrize("mode,win,st", [(0, 70, 1), (1, 0, 8)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), "both"])
def test_values_a_query_does_not_see_stay_out_of_its_result(value, mode, win, st, d):
    """32-row tiles (4200 queries): a value row that is not finite reaches the queries that see its key and no others."""
    from native_sparse_attention_pytorch_amd.ops import dense_attend_f32
    n, mem = 4200, mode                                           # (the strided prefix stands behind a memory row)
    keys = n // st
    q, k, v = _rand((1, 2, n, d), 1), _rand((1, 1, mem + keys, d), 2), _rand((1, 1, mem + keys, d), 3)
    rows = [mem + keys // 2, mem + keys - 40]
    run = lambda: dense_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), mode, True, win, st, mem)[0].cpu()
    clean = run()
    v[:, :, rows[0], 3], v[:, :, rows[1], 3] = (float("inf"), float("-inf")) if value == "both" else (value, value)
    v[:, :, rows[0], d - 1] = v[:, :, rows[0], 3]
    got = run()
    i, j = torch.arange(n), torch.tensor(rows) - mem
    see = (j[:, None] <= i) & (i - j[:, None] <= win) if mode == 0 else (j[:, None] + 1) * st <= i           # [row, query]
    want = clean.clone()
    for r, first in enumerate(rows):
        for f in (3, d - 1) if r == 0 else (3,):
            want[:, :, see[r], f] += v[0, 0, first, f]
    assert torch.equal(got.isnan(), want.isnan())
    same = want.isnan() | (got == want)
    assert same.all(), (~same).nonzero()[:5]


def test_queries_without_a_live_slot_do_not_read_their_keys_scores():
    """They attend their slots' blocks uniformly (NSA.py:809-815), also where the keys are infinite."""
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    n = 130
    q, k, v = (_rand((1, 2, n, 64), i) for i in range(3))
    k, v = k[:, :1], v[:, :1]
    idx = torch.tensor([0, 3]).expand(1, 1, n, 2).contiguous()
    msk = torch.zeros_like(idx, dtype=torch.bool)
    args = lambda key: (q.to(DEV), key.to(DEV), v.to(DEV), 32, idx.to(DEV), msk.to(DEV), False)
    want = native_sparse_attend_f32(*args(k))
    k[:, :, :5] = float("inf")
    got = native_sparse_attend_f32(*args(k))
    torch.cuda.synchronize()
    mean = torch.cat((v[:, :, :32], v[:, :, 96:128]), 2).double().mean(2, keepdim=True).expand(1, 2, n, 64)
    assert torch.equal(got, want)
    assert_close(got, mean, 1e-5, 1e-5, "out")


def test_live_slots_that_name_no_block_attend_nothing():
    """Not causal, an index out of range under a live slot: the query is not one without live slots, and has nothing to attend."""
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    n = 128
    q, k, v = (_rand((1, 2, n, 64), i)[:, :h].to(DEV) for i, h in ((1, 2), (2, 1), (3, 1)))
    idx = torch.tensor([-1, 5]).expand(1, 1, n, 2).contiguous().to(DEV)
    out, lse = native_sparse_attend_f32(q, k, v, 32, idx, torch.ones_like(idx, dtype=torch.bool), False, return_lse=True)
    torch.cuda.synchronize()
    assert not out.any() and (lse == float("-inf")).all()


@pytest.mark.parametrize("rows,k,n,bias,act", [(1, 8, 1, True, None), (31, 264, 33, True, "relu"), (32, 512, 32, False, None), (33, 72, 100, True, None),
                                               (256, 512, 40, True, "relu")])
def test_linear_f32(rows, k, n, bias, act):
    """Against float64: a sum of k products, each partial sum exact to 2^-24 of the sum of magnitudes per addition."""
    from native_sparse_attention_pytorch_amd import ops
    wide, w, b = _rand((rows, k + 4), 1), _rand((n, k), 2) * k ** -0.5, _rand((n,), 3)
    x = wide[:, :k]
    assert ops.linear_f32_supported(x.to(DEV), w.to(DEV))
    got = ops.linear_f32(wide.to(DEV)[:, :k], w.to(DEV), b.to(DEV) if bias else None, act=act)
    torch.cuda.synchronize()
    want = x.double() @ w.double().t() + (b.double() if bias else 0.)
    tol = k * 2 ** -24 * (x.double().abs() @ w.double().abs().t()) + 2 ** -23 * want.abs() + 1e-12
    want = torch.relu(want) if act else want
    assert ((got.double().cpu() - want).abs() <= tol).all()


@pytest.mark.parametrize("b,hq,hk,n,nc,st,B,share,causal,own,S", [
    (2, 4, 2, 70, 35, 2, 8, True, True, True, 5),
    (1, 6, 2, 31, 15, 2, 4, True, False, True, 2),          # not causal: only the own block is hidden
    (1, 4, 4, 40, 40, 1, 1, False, False, True, 16),        # stride = block: nothing hidden
    (1, 4, 2, 600, 600, 1, 1, True, True, True, 17),        # k > 16: a row per wave
    (1, 2, 1, 1, 90, 4, 12, True, False, False, 7),         # a decode step
])
def test_importance_topk_f32(b, hq, hk, n, nc, st, B, share, causal, own, S):
    """Scale and masks inside the top-k kernel: bit for bit what the kernel gives on the scaled, masked logits."""
    from native_sparse_attention_pytorch_amd import ops
    q, ck = _rand((b, hq, n, 64), 1).to(DEV), _rand((b, hk, nc, 64), 2).to(DEV)
    vals, idx, fm = ops.importance_topk_f32(q, ck, st, B, share, causal, S, mask_own=own)
    wv, wi, wf = ops.importance_topk(ops.importance_logits_f32(q, ck, st, B, share, causal, mask_own=own).contiguous(), S)
    torch.cuda.synchronize()
    assert torch.equal(vals, wv) and torch.equal(idx, wi) and torch.equal(fm, wf)


@pytest.mark.parametrize("b,hk,g,n,nc,d,mem,causal,qoff", [(1, 2, 3, 40, 10, 64, 1, True, 0), (2, 4, 2, 600, 37, 36, 33, True, 0), (1, 1, 4, 7, 0, 128, 2, False, 0),
                                                           (1, 8, 1, 1, 70, 64, 5, False, 300)])
def test_compressed_f32_memory_rows_of_their_own(b, hk, g, n, nc, d, mem, causal, qoff):
    """Memory rows read from the parameter instead of from in front of the keys: the same bits, in both kernels."""
    from native_sparse_attention_pytorch_amd import ops
    q, ck, cv, m = (_rand(s, i).to(DEV) for i, s in enumerate(((b, hk * g, n, d), (b, hk, nc, d), (b, hk, nc, d), (2, hk, mem, d))))
    got = ops.compress_attend_f32(q, ck, cv, m, 4, causal, q_offset=qoff)
    cat = lambda i, t: torch.cat((m[i][None].expand(b, -1, -1, -1), t), dim=2)
    want, _ = ops.dense_attend_f32(q, cat(0, ck), cat(1, cv), 1, causal, 0, 4, mem, q_offset=qoff)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_compressed_f32_memory_rows_elsewhere():
    """A parameter that is a slice at an odd place, or of another type, gives the same rows; one of another shape is refused."""
    from native_sparse_attention_pytorch_amd import ops
    q, ck, cv, m = (_rand(s, i).to(DEV) for i, s in enumerate(((1, 4, 9, 64), (1, 2, 4, 64), (1, 2, 4, 64), (2, 2, 3, 64))))
    want = ops.compress_attend_f32(q, ck, cv, m.bfloat16().float(), 4, True)
    odd = torch.empty(m.numel() + 1, device=DEV)[1:].view(m.shape).copy_(m.bfloat16())
    assert odd.data_ptr() % 16
    for t in (odd, m.bfloat16()):
        assert torch.equal(ops.compress_attend_f32(q, ck, cv, t, 4, True), want)
    for t in (m[:, :1], m[..., :32], m[:1]):
        with pytest.raises(RuntimeError):
            ops.compress_attend_f32(q, ck, cv, t, 4, True)


def test_selection_of_dead_blocks_only():
    """Not causal, every slot of some queries dead: uniform over the dead slots' blocks, padding included (NSA.py:809-815)."""
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    b, hq, hk, n, d, B, S = 1, 4, 2, 50, 64, 16, 3
    q, k, v = _rand((b, hq, n, d), 1), _rand((b, hk, n, d), 2), _rand((b, hk, n, d), 3)
    idx = torch.randint(0, 4, (b, hk, n, S), generator=torch.Generator().manual_seed(0))
    msk = torch.ones(b, hk, n, S, dtype=torch.bool)
    msk[:, :, ::3] = False
    want = O.select_attend(q.double(), k.double(), v.double(), idx, msk, B, causal=False)
    got = native_sparse_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), B, idx.to(DEV), msk.to(DEV), include_block_causal=False)
    torch.cuda.synchronize()
    assert_close(got, want, 1e-5, 1e-5, "out")


@pytest.mark.parametrize("b,h,n,d", [(1, 1, 1, 4), (2, 3, 5, 128), (1, 5, 33, 60)])
def test_gate_f32(b, h, n, d):
    from native_sparse_attention_pytorch_amd import ops
    lg, c, f, s = _rand((b, n, 3 * h), 1), *(_rand((b, h, n, d), i) for i in (2, 3, 4))
    got = ops.gate_combine_f32(*(t.to(DEV) for t in (lg, c, f, s)))
    torch.cuda.synchronize()
    g = lg.double().sigmoid().view(b, n, h, 3).permute(0, 2, 1, 3)
    want = (g[..., 0:1] * c.double() + g[..., 1:2] * f.double() + g[..., 2:3] * s.double()).permute(0, 2, 1, 3).reshape(b, n, h * d)
    assert_close(got, want, 1e-6, 1e-6, "merged")


def test_gate_f32_refuses():
    from native_sparse_attention_pytorch_amd import ops
    z = lambda *s: torch.zeros(*s, device=DEV)
    t = z(1, 4, 5, 64)
    for lg, f in ((z(1, 5, 9), t), (z(1, 4, 12), t), (z(1, 5, 12).bfloat16(), t), (z(1, 5, 12), z(1, 4, 4, 64))):
        with pytest.raises(RuntimeError):
            ops.gate_combine_f32(lg, t, f, t)


def _grads(outs, leaves, douts, **kw):
    used = [(o, g) for o, g in zip(outs, douts) if g is not None]
    return torch.autograd.grad([o for o, _ in used], leaves, [g for _, g in used], **kw)


@pytest.mark.parametrize("b,h,n,d", [(1, 1, 1, 4), (2, 3, 5, 128), (1, 5, 33, 60)])
def test_gate_f32_gradients(b, h, n, d):
    """Against float64; also with a graph of the gradient, which takes other operators.  A sum of d products: d + 8 roundings of
    the magnitudes (the sigmoid and its products among them)."""
    from native_sparse_attention_pytorch_amd import ops
    host = [_rand((b, n, 3 * h), 1), *(_rand((b, h, n, d), i) for i in (2, 3, 4))]
    do = _rand((b, n, h * d), 5)

    def merged(lg, c, f, s):
        g = lg.sigmoid().view(b, n, h, 3).permute(0, 2, 1, 3)
        return (g[..., 0:1] * c + g[..., 1:2] * f + g[..., 2:3] * s).permute(0, 2, 1, 3).reshape(b, n, h * d)

    ref = [t.double().requires_grad_() for t in host]
    want = torch.autograd.grad(merged(*ref), ref, do.double())
    mags = [t.double().abs().requires_grad_() for t in host]
    big = torch.autograd.grad(merged(*mags), mags, do.double().abs())
    wide = torch.zeros(b, n, 3 * h * d).to(DEV)
    wide[..., 1:1 + h * d] = do.to(DEV)                    # a gradient that is neither contiguous nor aligned
    for graph in (False, True):
        leaves = [t.to(DEV).requires_grad_() for t in host]
        got = torch.autograd.grad(ops.gate_combine_f32(*leaves), leaves, wide[..., 1:1 + h * d], create_graph=graph)
        torch.cuda.synchronize()
        for w, g, m in zip(want, got, big):
            assert ((g.double().cpu() - w).abs() <= (d + 8) * 2 ** -24 * (m.abs() + w.abs() + m.abs().max()) + 1e-30).all()


@pytest.mark.parametrize("b,hq,hk,n,d,cbs,st,offset,missing", [
    (1, 4, 2, 1, 64, 4, 2, 0, ()),                  # fewer tokens than a stride: no window
    (2, 2, 1, 33, 64, 16, 8, 0, ()), (1, 3, 1, 70, 128, 6, 4, 5, ()), (1, 2, 2, 37, 128, 4, 4, 0, (0, 4)), (2, 8, 4, 130, 64, 5, 1, 0, (1, 2, 3)),
])
def test_qkv_prep_f32_gradients(b, hq, hk, n, d, cbs, st, offset, missing):
    """Against float64 of the operators it stands for, outputs and gradients, gradients left out among them, and with a graph of
    the gradient.  An angle is off by a rounding of its size (n + offset at most), a sum has at most 4 + cbs / st terms; the
    gradients of the positions sum b * windows of them."""
    from native_sparse_attention_pytorch_amd import ops
    qkv, kp, vp = _rand((b, n, (hq + 2 * hk) * d), 1), _rand((hk, cbs, d), 2), _rand((hk, cbs, d), 3)
    freqs = 1.0 / (10000 ** (torch.arange(0, d, 2).float() / d))
    douts = [None if i in missing else _rand((b, h, n, d), 4 + i) for i, h in enumerate((hq, hq, hk, hk))]
    douts += [None if i in missing else _rand((b, hk, n // st, cbs, d), 4 + i) for i in (4, 5)]

    def parts(z, kp, vp):
        q, k, v = (u.unflatten(-1, (-1, d)).transpose(1, 2) for u in z.split((hq * d, hk * d, hk * d), dim=-1))
        ang = torch.outer(torch.arange(offset, offset + n).double(), freqs.double())
        cos, sin = ang.cos().repeat_interleave(2, -1), ang.sin().repeat_interleave(2, -1)
        rot = lambda t: t * cos + torch.stack((-t[..., 1::2], t[..., 0::2]), -1).flatten(-2) * sin
        return q, rot(q), rot(k), v, ops.windows_of(k, kp, cbs, st), ops.windows_of(v, vp, cbs, st)

    ref = [t.double().requires_grad_() for t in (qkv, kp, vp)]
    outs = parts(*ref)
    want = _grads(outs, ref, [None if g is None else g.double() for g in douts], allow_unused=True)
    tol = 2 ** -24 * (2 * (n + offset) + 16) * 5 * (4 + -(-cbs // st))
    for graph in (False, True):
        leaves = [t.to(DEV).requires_grad_() for t in (qkv, kp, vp)]
        mine = ops.qkv_prep_f32(leaves[0], freqs.to(DEV), leaves[1], leaves[2], hq, hk, d, cbs, st, offset)
        got = _grads(mine, leaves, [None if g is None else g.to(DEV) for g in douts], allow_unused=True, create_graph=graph)
        torch.cuda.synchronize()
        for o, w in zip(mine, outs):
            assert o.shape == w.shape and ((o.detach().double().cpu() - w.detach()).abs() <= tol).all()
        for i, (g, w) in enumerate(zip(got, want)):
            assert (g is None) == (w is None)
            if g is not None:
                assert ((g.double().cpu() - w).abs() <= (tol if i == 0 else tol * b * max(1, n // st))).all()


@pytest.mark.parametrize("rows,nb,k", [(1, 1, 1), (5, 3, 3), (7, 64, 4), (33, 65, 17), (3, 2048, 64), (2, 2049, 3)])
def test_importance_topk_gradient(rows, nb, k):
    """Against float64 of softmax with the pad column; rows with nothing to select and masked entries among them.  A product of a
    probability (exp to 2 ulp, a sum of nb) and a difference of two sums of k terms."""
    from native_sparse_attention_pytorch_amd import ops
    x, dv = _rand((rows, nb), 1), _rand((rows, k), 2)
    x[torch.rand(rows, nb, generator=torch.Generator().manual_seed(3)) < 0.2] = -math.inf
    x[rows // 2] = -math.inf
    for graph in (False, True):
        leaf = x.to(DEV).requires_grad_()
        vals, idx, _ = ops.importance_topk(leaf, k)
        got, = torch.autograd.grad(vals, leaf, dv.to(DEV), create_graph=graph)
        torch.cuda.synchronize()
        p = torch.nn.functional.pad(x.double(), (1, 0), value=-1e3).softmax(-1)[:, 1:]
        full = torch.zeros(rows, nb, dtype=torch.float64).scatter_add_(-1, idx.cpu().long(), dv.double())
        dot = (p * full).sum(-1, keepdim=True)
        tol = 2 ** -24 * (nb + k + 16) * p * (full.abs() + (p * full.abs()).sum(-1, keepdim=True)) + 1e-30
        assert ((got.double().cpu() - p * (full - dot)).abs() <= tol).all()


@pytest.mark.parametrize("b,h,n,d,hrep,off,rrep,srows,base32", [(1, 1, 1, 8, 1, 0, 1, 1, False), (2, 4, 9, 64, 2, 0, 1, 9, False), (2, 6, 23, 128, 1, 2, 4, 5, True),
                                                                (1, 3, 37, 64, 3, 1, 3, 12, True)])
def test_add_repeated(b, h, n, d, hrep, off, rrep, srows, base32):
    """bf16(base + c * small), rounded once; in place where the base is bf16."""
    from native_sparse_attention_pytorch_amd import ops
    base = _rand((b, h, n, d), 1) if base32 else _rand((b, h, n, d), 1).bfloat16()
    small = _rand((b, h // hrep, srows, d), 2)
    want = base.double().clone()
    rep = small.double().repeat_interleave(hrep, 1).repeat_interleave(rrep, 2)
    want[:, :, off:off + srows * rrep] += 0.3 * rep
    dev = base.to(DEV)
    got = ops._add_repeated(dev, small.to(DEV), torch.empty_like(dev, dtype=torch.bfloat16) if base32 else dev, hrep, off, rrep, 0.3)
    torch.cuda.synchronize()
    assert ((got.double().cpu() - want).abs() <= want.abs() * (2 ** -8 + 2 ** -20) + 2 ** -20).all()
