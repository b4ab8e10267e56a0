"""Every (batch, kv head) pair's every tile of the fp32 tile kernel is some work-group's, whatever the number of pairs: on the host for all
launches whose order is turned round, and on the device against float64 with results that start as NaN.

Bound: 1e-5 + 1e-5 |value|, the reference's own fp32 tolerance (tests/test_sparse_attn.py:86)."""
import ctypes as C
import math

import pytest
import torch

from tests.util import assert_close

DEV = "cuda"


def _order(pairs, tiles, two=True):
    from native_sparse_attention_pytorch_amd import _lib
    out = (C.c_int32 * (pairs * tiles))()
    assert _lib.lib().nsa_selftest_f32_tiles(pairs, tiles, two, out) == 0
    return list(out)


@pytest.mark.parametrize("two", [True, False])
def test_each_tile_once(two):
    for pairs in range(1, 521):
        for tiles in range(1, 520 // pairs + 1):
            assert sorted(_order(pairs, tiles, two)) == list(range(pairs * tiles)), (pairs, tiles)


def test_longest_first_and_in_pairs():
    """The last tiles, whose key lists are the longest, come first; work-groups 256 apart share a CU, and the two together have as long a
    walk everywhere, to one tile.  Where a CU holds one, the order is not turned."""
    assert [t % 24 for t in _order(12, 24)[:24:12]] == [23, 22]
    assert {o % 32 + p % 32 for o, p in zip(_order(16, 32)[:256], _order(16, 32)[256:])} <= {30, 31, 32}
    assert [t % 32 for t in _order(16, 32, False)] == [31 - i // 16 for i in range(512)]
    assert [t % 60 for t in _order(10, 60)] == [59 - i // 10 for i in range(600)]


def _visible(mode, n, nk, mem, window, stride, causal):
    i, j = torch.arange(n, device=DEV)[:, None], torch.arange(nk + mem, device=DEV)[None]
    if mode == 0:
        return (i - j <= window) & (j <= i if causal else j - i <= window)
    return (j < mem) | ~torch.tensor(causal, device=DEV) | ((j - mem + 1) * stride <= i)


def _attention(q, k, v, weight):
    g = q.shape[1] // k.shape[1]
    sim = q.double() @ k.double().repeat_interleave(g, 1).transpose(-1, -2).contiguous() * q.shape[-1] ** -0.5 + weight.log()
    return sim.softmax(-1) @ v.double().repeat_interleave(g, 1), sim.logsumexp(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("b,hq,hk,n,d", [
    (3, 8, 2, 1500, 64),      # 6 pairs of 47 tiles
    (3, 16, 4, 1000, 64),     # 12 of 32
    (3, 8, 8, 1500, 64),      # 24 of 12
    (1, 12, 12, 2900, 64),    # 12 of 23
    (3, 32, 8, 500, 128),     # 24 of 16
    (3, 6, 2, 1000, 100),     # 6 of 24, groups of 3: 144 work-groups, none turned
])
def test_every_row_is_written(b, hq, hk, n, d, monkeypatch):
    from native_sparse_attention_pytorch_amd import ops
    print(b, hq, hk, n, d, flush=True)
    g = torch.Generator(device=DEV).manual_seed(n)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, v, rq = r(b, hq, n, d), r(b, hk, n, d), r(b, hk, n, d), r(b, hq, n, d)
    stride, mem, window, B, S = 16, 2, 100, 64, 8
    ck, cv, m = r(b, hk, n // stride, d), r(b, hk, n // stride, d), r(2, hk, mem, d)
    W, own = math.ceil(n / B), (torch.arange(n, device=DEV) // B)[:, None]
    val, idx = torch.rand(b, hk, n, W, generator=g, device=DEV).masked_fill_(torch.arange(W, device=DEV)[None] >= own, -1.).topk(min(S, W), dim=-1)
    idx, msk = idx.masked_fill(val < 0, 0).contiguous(), (val >= 0).contiguous()
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: empty(*a, **kw).fill_(math.nan))
    c_out, s_out = ops.compress_window_f32(q, ck, cv, m, stride, rq, k, v, window, True)
    c_alone = ops.compress_attend_f32(q, ck, cv, m, stride, True)
    w_out, w_lse = ops.dense_attend_f32(rq, k, v, 0, False, window)
    f_out, f_lse = ops.native_sparse_attend_f32(rq, k, v, B, idx, msk, return_lse=True)
    monkeypatch.undo()
    mk, mv = (torch.cat((t[None].expand(b, -1, -1, -1), c), dim=2) for t, c in zip(m, (ck, cv)))
    want, _ = _attention(q, mk, mv, _visible(1, n, n // stride, mem, 0, stride, True).double())
    assert_close(c_out, want, 1e-5, 1e-5, "compressed, beside the window")
    assert_close(c_alone, want, 1e-5, 1e-5, "compressed")
    assert_close(s_out, _attention(rq, k, v, _visible(0, n, n, 0, window, 1, True).double())[0], 1e-5, 1e-5, "window")
    for name, got, ref in zip(("out", "lse"), (w_out, w_lse), _attention(rq, k, v, _visible(0, n, n, 0, window, 1, False).double())):
        assert_close(got, ref, 1e-5, 1e-5, "window of both sides, " + name)
    i, j = torch.arange(n, device=DEV)[:, None], torch.arange(n, device=DEV)[None]
    seen = torch.zeros(b, hk, n, W, device=DEV, dtype=torch.double).scatter_add_(-1, idx, msk.double()).repeat_interleave(B, -1)[..., :n]
    seen = seen + ((j // B == i // B) & (j <= i)).double()
    for name, got, ref in zip(("out", "lse"), (f_out, f_lse), _attention(rq, k, v, seen.repeat_interleave(hq // hk, 1))):
        assert_close(got, ref, 1e-5, 1e-5, "selected blocks, " + name)


@pytest.mark.gpu
@pytest.mark.parametrize("b,hq,hk,n,window,causal", [(1, 8, 8, 127, 3, True), (1, 8, 8, 128, 2, True), (2, 16, 8, 128, 47, False), (1, 8, 8, 256, 48, True), (1, 8, 8, 257, 5, False)])
def test_narrow_windows_of_ungrouped_heads(b, hq, hk, n, window, causal):
    """Both sides of the lines between rows and tiles at 128 features."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator(device=DEV).manual_seed(n)
    q, k, v = (torch.randn(b, h, n, 128, generator=g, device=DEV) for h in (hq, hk, hk))
    for name, got, ref in zip(("out", "lse"), ops.dense_attend_f32(q, k, v, 0, causal, window),
                              _attention(q, k, v, _visible(0, n, n, 0, window, 1, causal).double())):
        assert_close(got, ref, 1e-5, 1e-5, name)
