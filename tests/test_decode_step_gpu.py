"""The decode step's three launches (window + new token, compressed keys with pooled logits; selection + selected blocks; merge)
against the same step through the separate entry points, at the sizes where they can go wrong: a newest key that is alone in its
tile, spare cache rows full of NaN, every pooling ratio, selections with ties, with many equal entries and with their
winners in few lanes, rows of up to 2048 blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF16 = torch.bfloat16


def _step(b, hq, hk, d, pos, nc, npf, B, S, share, window, mem, ck=None, seed=0, q=None):
    """The fused step and the step from its parts: (merged, idx, fmask, keys, vals, run rows) each, and the pooled probabilities."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).to(BF16).to(DEV)
    q = r(b, hq, 1, d) if q is None else q
    k, v = r(b, hk, 1, d), r(b, hk, 1, d)
    cap = pos + 70
    def cache():
        t = torch.full((b, hk, cap, d), float("nan"), dtype=BF16, device=DEV)
        return t
    keys, vals = cache(), cache()
    keys[:, :, :pos], vals[:, :, :pos] = r(b, hk, pos, d), r(b, hk, pos, d)
    ck = r(b, hk, nc, d) if ck is None else ck
    cv = r(b, hk, nc, d)
    mk, mv = r(hk, mem, d), r(hk, mem, d)
    gl = r(b, 1, 3 * hq)
    freqs = (1.0 / (10000 ** (torch.arange(0, d, 2).float() / d))).to(DEV)
    run = [torch.zeros(b, hk, 1, d, dtype=BF16, device=DEV) for _ in range(4)]
    k1, v1, k2, v2 = keys.clone(), vals.clone(), keys.clone(), vals.clone()
    merged, idx, fm = ops.decode_step(q, k, v, freqs, pos, k1, v1, ck if nc else None, cv if nc else None, mk, mv, run[0], run[1], gl, per_block=npf,
                                      block=B, num_sel=S, share=share, window=window)
    rq = ops.decode_prep(q, k, v, freqs, pos, k2[:, :, pos:pos + 1], v2[:, :, pos:pos + 1], run[2], run[3])
    kk = min(S, nc // npf)
    c = None
    want_i, want_m, probs = idx[..., :0], fm[..., :0], None
    if nc:
        c, logits = ops.decode_range_attend(q, ck, cv, 0, nc, mk, mv, return_logits=True, merge=False)
        if kk:
            _, want_i, want_m = ops.decode_importance_topk(logits, hk, npf, share, kk)
            nb = nc // npf
            p = logits[..., :nb * npf].reshape(b, hk, hq // hk, nb, npf).mean(-1)
            probs = (p.mean(2, keepdim=True) if share else p.reshape(b, hq, 1, nb)).softmax(-1)
    f = ops.decode_select_attend(rq, k2, v2, pos + 1, B, want_i.int(), want_m, merge=False)
    w = min(pos + 1, window + 1)
    s = ops.decode_range_attend(rq, k2, v2, pos + 1 - w, w, merge=False)
    want = ops.decode_combine(gl, c, f, s)
    torch.cuda.synchronize()
    return (merged, idx, fm, k1, v1, run[0], run[1]), (want, want_i, want_m, k2, v2, run[2], run[3]), probs


def _check(got, want, probs, exact):
    for a, b_, what in zip(got[3:], want[3:], ("keys", "values", "window key", "window value")):
        assert torch.equal(a.view(torch.int16), b_.view(torch.int16)), what
    assert got[1].shape == want[1].shape
    same = (got[1].long() == want[1].long()).all(-1).flatten()
    if exact:
        assert same.all() and torch.equal(got[2], want[2])
    elif probs is not None:
        # the pooled sums are taken in another order: an order of two blocks may change where their probabilities agree to 1e-5
        pg, pw = probs.gather(-1, got[1].long()), probs.gather(-1, want[1].long())
        assert torch.allclose(pg, pw, rtol=1e-5, atol=0)
    rows = same.view(got[0].shape[0], -1).all(-1)
    assert torch.isfinite(got[0]).all()
    err = (got[0][rows].float() - want[0][rows].float()).abs()
    # bf16 results of the same partial sums merged in another order: at most one rounding of the three branches and of the sum
    assert (err <= 2 ** -7 * want[0][rows].float().abs() + 2 ** -7).all(), err.max().item()


@pytest.mark.parametrize("b,hq,hk,d,pos,nc,npf,B,S,share,window,mem", [
    (2, 8, 2, 64, 96, 24, 4, 16, 3, True, 96, 1),       # window of 97 keys: the newest alone in the last tile
    (1, 4, 4, 128, 0, 0, 1, 16, 4, True, 16, 1),        # the first token of a sequence: nothing cached
    (1, 8, 1, 128, 64, 40, 1, 8, 5, True, 0, 2),        # a block per compressed key, window of the newest key alone, groups of 8
    (3, 6, 2, 64, 333, 166, 2, 4, 6, True, 50, 1),      # groups of 3 heads
    (1, 8, 4, 64, 500, 250, 8, 16, 7, False, 64, 40),   # selection per head; two tiles of memory slots
    (1, 4, 2, 128, 700, 175, 16, 64, 9, True, 128, 1),
    (2, 4, 2, 64, 900, 900, 32, 32, 20, False, 32, 1),
    (1, 4, 2, 64, 300, 75, 5, 20, 4, True, 31, 1),      # 5 compressed keys per block: pooled by the top-k kernel
    (1, 4, 1, 64, 100, 3, 4, 16, 4, True, 31, 1),       # compressed keys but no whole block yet
])
def test_step_equals_its_parts(b, hq, hk, d, pos, nc, npf, B, S, share, window, mem):
    got, want, probs = _step(b, hq, hk, d, pos, nc, npf, B, S, share, window, mem)
    _check(got, want, probs, exact=False)


@pytest.mark.parametrize("nb,k,scores", [
    (200, 16, "equal"),           # every block alike: the lowest indices, found by the exact search with ties
    (2048, 64, "equal"),          # the longest row, the most slots
    (640, 16, "column"),          # the winners in one lane: more than 64 entries beyond its maximum
    (64, 64, "rising"),           # as many slots as blocks
    (70, 5, "pairs"),             # equal pairs across the boundary of the selection
    (1000, 16, "falling"),
    (300, 16, "spike"),           # one block with all the probability: the others' slots are dead
])
def test_selection_order(nb, k, scores):
    """Exact logits (multiples of 1/8 of equal vectors): indices, their order and the mask equal the top-k kernel's bit for bit."""
    j = torch.arange(nb).float()
    a = {"equal": j * 0 + 1, "column": (j % 64 == 5).float() * (2 + (j // 64) / 8), "rising": j / 8, "pairs": (j // 2) / 8, "falling": (nb - j) / 64,
         "spike": (j == 17).float() * 240}[scores]
    d, hq, hk = 64, 4, 2
    ck = (a[:, None] * torch.full((d,), 0.125)).to(BF16).expand(1, hk, nb, d).contiguous().to(DEV)
    q = torch.ones(1, hq, 1, d, dtype=BF16, device=DEV)
    got, want, probs = _step(1, hq, hk, d, 4 * nb, nb, 1, 4, k, True, 16, 1, ck=ck, q=q)
    _check(got, want, probs, exact=True)


@pytest.mark.parametrize("wrong", ["batch", "heads"])
def test_caches_of_another_shape_are_refused(wrong):
    from native_sparse_attention_pytorch_amd import ops
    z = lambda *s: torch.zeros(*s, dtype=BF16, device=DEV)
    b, hk = (1, 2) if wrong == "batch" else (2, 1)
    q, k, gl, freqs = z(2, 4, 1, 64), z(2, 2, 1, 64), z(2, 1, 12), torch.zeros(32, device=DEV)
    with pytest.raises(RuntimeError, match="batch, heads"):
        ops.decode_step(q, k, k, freqs, 8, z(b, hk, 9, 64), z(b, hk, 9, 64), None, None, None, None, None, None, gl, per_block=2, block=16, num_sel=2,
                        share=True, window=16)


def test_caches_of_more_sequences_or_heads_are_read_from_their_start():
    """Buffers larger than the step (more sequences, more heads): the step takes their first ones."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g).to(BF16).to(DEV)
    q, k, v, gl, freqs = r(2, 4, 1, 64), r(2, 2, 1, 64), r(2, 2, 1, 64), r(2, 1, 12), torch.ones(32, device=DEV)
    big = [r(3, 3, n, 64) for n in (41, 41, 10, 10)]
    first = [t[:2, :2].clone() for t in big]
    run = lambda c: ops.decode_step(q, k, v, freqs, 40, *c, None, None, None, None, gl, per_block=2, block=16, num_sel=2, share=True, window=16)[0]
    rest = [t.clone() for t in big]
    got, want = run(big), run(first)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and all(torch.equal(a[:2, :2], b) for a, b in zip(big, first))
    for a, b in zip(big, rest):
        b[:2, :2] = a[:2, :2]
        assert torch.equal(a, b)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_branch_whose_sum_is_no_number_adds_nothing(value, d):
    """Keys that are not finite in the window: the branch is left out whole, as when it is merged on its own; the others stand."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(d)
    r = lambda *s: torch.randn(*s, generator=g).to(BF16).to(DEV)
    b, hq, hk, n = 2, 4, 2, 130
    rq, ks, vs, gl = r(b, hq, 1, d), r(b, hk, n, d), r(b, hk, n, d), r(b, 1, 3 * hq)
    ks[:, :, 70] = value
    idx = torch.zeros(b, hk, 1, 1, dtype=torch.int32, device=DEV)
    f = ops.decode_select_attend(rq, ks, vs, 64, 32, idx, torch.ones_like(idx, dtype=torch.bool), merge=False)      # the first 64 keys: finite
    s = ops.decode_range_attend(rq, ks, vs, n - 65, 65, merge=False)
    alone = ops.decode_range_attend(rq, ks, vs, n - 65, 65)
    got, want = ops.decode_combine(gl, None, f, s), ops.decode_combine(gl, None, f, ops.decode_range_attend(rq, ks, torch.zeros_like(vs), 0, 64, merge=False))
    torch.cuda.synchronize()
    assert not alone.any() and torch.isfinite(got).all() and torch.equal(got, want)
