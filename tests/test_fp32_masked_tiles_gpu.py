"""Block selection of fp32 modules as masked tiles (many queries that attend a fair share of at most 128 blocks) against float64,
and against the same call cut into pieces too small for that kernel.

Bound: 1e-5 + 1e-5 |value|, the reference's own fp32 tolerance (tests/test_sparse_attn.py:86); the errors measured are ~5e-6 of
the results' root mean square."""
import math

import pytest
import torch

from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _selection(b, hk, n, B, S, anything, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    W = math.ceil(n / B)
    if anything:      # blocks named twice, the own block, later ones, the one that reaches past the end, dead slots
        return (torch.randint(0, W, (b, hk, n, S), generator=g, device=DEV), torch.rand(b, hk, n, S, generator=g, device=DEV) > 0.3)
    own = (torch.arange(n, device=DEV) // B)[:, None]
    scores = torch.rand(b, hk, n, W, generator=g, device=DEV).masked_fill_(torch.arange(W, device=DEV)[None] >= own, -1.)
    val, idx = scores.topk(min(S, W), dim=-1)
    return idx.masked_fill(val < 0, 0).contiguous(), (val >= 0).contiguous()


def _weights(idx, msk, n, B):
    """How often each key counts for each query: once per live slot that names its block, once more in the own block up to the query."""
    W = math.ceil(n / B)
    times = torch.zeros(*idx.shape[:3], W, device=DEV, dtype=torch.double).scatter_add_(-1, idx.long(), msk.double())
    i, j = torch.arange(n, device=DEV)[:, None], torch.arange(W * B, device=DEV)[None]
    return times.repeat_interleave(B, -1) + ((j // B == i // B) & (j <= i)).double()


def _inputs(b, hq, hk, n, d, seed):
    """Queries, keys and values as views of one projection 'b n (h d)'."""
    x = torch.randn(b, n, (hq + 2 * hk) * d, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV)
    return (t.unflatten(-1, (-1, d)).transpose(1, 2) for t in x.split((hq * d, hk * d, hk * d), dim=-1))


@pytest.mark.parametrize("anything", [False, True])
@pytest.mark.parametrize("b,hq,hk,n,d,B,S", [
    (8, 4, 2, 300, 64, 64, 4),           # the last block has 44 keys
    (11, 4, 4, 128, 64, 4, 3),           # eight blocks to a tile; groups of 1
    (8, 12, 4, 130, 100, 32, 5),         # groups of 3: rows of a wave end inside a query; 100 features
    (1, 8, 8, 2041, 64, 16, 24),         # 128 blocks, two to a tile
    (1, 32, 2, 577, 128, 64, 9),         # d = 128; a tenth block of one key
    (3, 10, 2, 700, 60, 128, 4),         # blocks of four tiles
])
def test_against_float64(b, hq, hk, n, d, B, S, anything):
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    q, k, v = _inputs(b, hq, hk, n, d, n)
    idx, msk = _selection(b, hk, n, B, S, anything, B)
    got, lse = native_sparse_attend_f32(q, k, v, B, idx.int() if d == 64 else idx, msk, return_lse=True)
    g, pad = hq // hk, math.ceil(n / B) * B - n
    wide = lambda t: torch.nn.functional.pad(t.double(), (0, 0, 0, pad)).repeat_interleave(g, 1)
    sim = q.double() @ wide(k).transpose(-1, -2) * d ** -0.5 + _weights(idx, msk, n, B).log().repeat_interleave(g, 1)
    assert_close(got, sim.softmax(-1) @ wide(v), 1e-5, 1e-5, "out")
    assert_close(lse, sim.logsumexp(-1), 1e-5, 1e-5, "lse")
    parts = torch.cat([native_sparse_attend_f32(q[:1, h * g:h * g + g], k[:1, h:h + 1], v[:1, h:h + 1], B, idx[:1, h:h + 1], msk[:1, h:h + 1])
                       for h in range(min(hk, 2))], dim=1)
    assert_close(got[:1, :parts.shape[1]], parts, 1e-5, 1e-5, "pieces")


@pytest.mark.parametrize("d", [64, 128])
def test_what_is_not_finite_stays_with_the_queries_that_see_it(d):
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    b, n, B = 8, 600, 64
    q, k, v = (t.clone() for t in _inputs(b, 4, 2, n, d, 1))
    idx, msk = _selection(b, 2, n, B, 3, False, 2)
    run = lambda: native_sparse_attend_f32(q, k, v, B, idx, msk)
    clean = run()
    see = _weights(idx, msk, n, B)[..., :n].repeat_interleave(2, 1)
    v[:, :, 70, 3], v[:, :, 330, 3], v[:, :, 331, d - 1] = math.inf, -math.inf, math.nan
    got, want = run(), clean.clone()
    for key, f in ((70, 3), (330, 3), (331, d - 1)):
        want[..., f] = torch.where(see[..., key] > 0, want[..., f] + v[0, 0, key, f], want[..., f])
    assert torch.equal(got.isnan(), want.isnan())
    assert_close(got[want.isfinite()], want[want.isfinite()], 1e-6, 1e-6, "finite")
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    # keys of scores that overflow to minus infinity weigh nothing, keys that are not finite reach those that see them
    v.nan_to_num_(0., 0., 0.)
    q[..., 0], k[..., 0] = q[..., 0].abs() + 1e20, 0.
    k[:, :, 64:128, 0] = -1e30
    got, msk2 = run(), msk & (idx != 1)
    assert_close(got[:, :, 128:], native_sparse_attend_f32(q, k, v, B, idx, msk2)[:, :, 128:], 1e-5, 1e-5, "overflow")
    k[:, :, 64:128, 0], k[:, :, 100, 1] = 0., math.nan
    assert torch.equal(run().isnan().any(-1), see[..., 100] > 0)


def test_a_scale_of_any_sign():
    """Through the C entry: attention under scale 0 is the mean of what is seen, under -s that of negated queries under s."""
    import ctypes as C
    from native_sparse_attention_pytorch_amd import _lib
    from native_sparse_attention_pytorch_amd.ops import _ptr, _select_desc, _stream
    b, hk, n, d, B, S = 8, 2, 300, 64, 64, 3
    q, k, v = (t.contiguous() for t in _inputs(b, 4, hk, n, d, 3))
    idx, msk = _selection(b, hk, n, B, S, False, 4)
    idx, fm = idx.int(), msk.view(torch.uint8)

    def run(q, scale):
        out = torch.empty_like(q)
        dsc = _select_desc(q, k, v, out, S, B, True, scale, False)
        _lib.check(_lib.lib().nsa_select_fwd_f32(C.byref(dsc), _ptr(q), _ptr(k), _ptr(v), _ptr(idx), _ptr(fm), _ptr(out), None, n, 0, _stream()), "select")
        return out

    w = _weights(idx, msk, n, B)[..., :n].repeat_interleave(2, 1)
    assert_close(run(q, 0.), (w / w.sum(-1, keepdim=True)) @ v.double().repeat_interleave(2, 1), 1e-5, 1e-5, "scale 0")
    assert torch.equal(run(-q, -0.125), run(q, 0.125))
