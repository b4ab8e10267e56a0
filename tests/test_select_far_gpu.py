"""Block selection in layouts and scales that the walks by 32-bit offsets refuse - rows of Q, of out and d_out, or tokens of K and V beyond their
reach, a scale that is not positive - against the same attention in float64, through the C entry points (the operators make out and d_out
contiguous)."""

import ctypes as C

import pytest
import torch

from tests.util import causal_random_selection

pytestmark = pytest.mark.gpu
B, S = 64, 5


def spread(x, stride):
    """x [1, h, n, d] with its tokens `stride` elements apart."""
    _, h, n, d = x.shape
    return torch.empty((n - 1) * stride + h * d, dtype=x.dtype, device=x.device).as_strided((1, h, n, d), (n * stride, d, stride, 1)).copy_(x)


def reference(q, k, v, do, idx, live, scale):
    q, k, v, do = (t[0].double() for t in (q, k, v, do))
    hk, n = k.shape[:2]
    g = q.shape[0] // hk
    W = -(-n // B)
    sel = torch.zeros(hk, n, W + 1, dtype=torch.bool, device=q.device).scatter_(2, torch.where(live[0], idx[0].long(), W), True)[..., :W]
    i = torch.arange(n, device=q.device)
    m = sel.repeat_interleave(B, 2)[..., :n] | ((i[:, None] // B == i // B) & (i <= i[:, None]))
    m, k, v = (t.repeat_interleave(g, 0) for t in (m, k, v))
    s = (q @ k.transpose(1, 2).contiguous() * scale).masked_fill(~m, -torch.inf)
    lse = s.logsumexp(-1)
    p = (s - lse[..., None]).exp()
    dp = do @ v.transpose(1, 2).contiguous()
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
    per_kv = lambda t: t.unflatten(0, (hk, g)).sum(1)
    return p @ v, lse, ds @ k, per_kv(ds.transpose(1, 2).contiguous() @ q), per_kv(p.transpose(1, 2).contiguous() @ do)


# far: which rows; a token stride of 2^21 elements takes 1100 tokens beyond 4 GB, 2^24 is the first of K / V that is refused
@pytest.mark.parametrize("hq,hk,d", [(8, 2, 128), (8, 8, 128), (8, 2, 64)])
@pytest.mark.parametrize("far,gated,scale", [("q", False, 1.0), ("q", True, 1.0), ("out", False, 1.0), ("kv", False, 1.0), ("none", False, -1.0)])
def test_against_float64(hq, hk, d, far, gated, scale):
    """p and dS are rounded to bf16, and so are a slot's partial results and the sums of them: 2^-9 each."""
    from native_sparse_attention_pytorch_amd import _lib, ops
    print(f"case {hq} {hk} {d} {far} {gated} {scale}", flush=True)
    n, scale = 130 if far == "kv" else 1100, scale * d ** -0.5
    g = torch.Generator(device="cuda").manual_seed(n + d)
    q, k, v, do = (torch.randn(1, h, n, d, generator=g, device="cuda").mul_(d ** -0.25).bfloat16() for h in (hq, hk, hk, hq))
    idx, live = (t.cuda() for t in causal_random_selection(1, hk, n, B, S, seed=3))
    want = reference(q, k, v, do, idx, live, scale)
    if far == "q":
        q = spread(q, 1 << 21)
    if far == "kv":
        k, v = spread(k, 1 << 24), spread(v, 1 << 24)
    out = torch.empty_like(do)
    if far == "out":
        do, out = spread(do, 1 << 21), spread(out, 1 << 21)
    lse = torch.empty(1, hq, n, device="cuda")
    grads = [torch.empty(1, h, n, d, dtype=torch.bfloat16, device="cuda") for h in (hq, hk, hk)]
    dsel = torch.empty(idx.shape, device="cuda")
    dsc = ops._select_desc(q, k, v, out, S, B, True, scale, idx.dtype == torch.int64)
    L, st, mask = _lib.lib(), torch.cuda.current_stream().cuda_stream, live.view(torch.uint8)
    at = lambda t: t.data_ptr()
    ib, fb, wb = ops._ws_sizes(dsc)
    index, fws, bws = (torch.empty(x, dtype=torch.uint8, device="cuda") for x in (ib, fb, wb))
    assert L.nsa_select_build_index(C.byref(dsc), at(idx), at(mask), at(index), ib, st) == 0
    if scale > 0:
        assert L.nsa_select_fwd(C.byref(dsc), at(q), at(k), at(v), at(idx), at(mask), at(index), at(fws), fb, at(out), at(lse), st) == 0
    else:      # the forward takes the maximum of a row before it scales: positive scales only
        out.copy_(want[0][None])
        lse.copy_(want[1][None])
    assert L.nsa_select_bwd(C.byref(dsc), at(q), at(k), at(v), at(out), at(do), None, at(lse), at(idx), at(mask), at(index), at(bws), wb,
                            *map(at, grads), at(dsel) if gated else None, st) == 0
    torch.cuda.synchronize()
    assert (lse[0].double() - want[1]).abs().max().item() < 1e-5
    for name, x, y, tol in zip(("out", "dq", "dk", "dv"), (out, *grads), (want[0], *want[2:]), (2 ** -8, 2 ** -7, 2 ** -7, 2 ** -8)):
        assert torch.isfinite(x).all(), name
        err = ((x[0].double() - y).norm() / y.norm()).item()
        assert err < tol, (name, err)
