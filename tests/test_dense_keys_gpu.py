"""dK / dV of interval-masked attention at 128 features (one wave per tile of 32 rows, four per 64 keys): where its tiles, chunks, waves and
heads begin and end, in the layouts that callers have, against the same attention in float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def visible(mode, n, nkeys, mem, window, stride, causal):
    i, c = torch.arange(n, device="cuda")[:, None], torch.arange(nkeys, device="cuda")[None]
    if mode == 0:
        return (c <= i if causal else c - i <= window) & (i - c <= window)
    m = (c + 1) * stride <= i if causal else torch.ones(n, nkeys, dtype=torch.bool, device="cuda")
    return torch.cat((torch.ones(n, mem, dtype=torch.bool, device="cuda"), m), dim=1)


def reference(q, k, v, do, m, scale):
    q, k, v, do = (t.double() for t in (q, k, v, do))
    b, hq, n, d = q.shape
    hk = k.shape[1]
    q, do = (t.reshape(b, hk, hq // hk, n, d) for t in (q, do))
    s = (q @ k.transpose(-1, -2).contiguous()[:, :, None]).mul(scale).masked_fill(~m, -torch.inf)
    p = s.softmax(-1)
    dp = do @ v.transpose(-1, -2).contiguous()[:, :, None]
    ds = p * (dp - (p * dp).sum(-1, keepdim=True)) * scale
    dq = (ds @ k[:, :, None]).reshape(b, hq, n, d)
    dk = (ds.transpose(-1, -2).contiguous() @ q).sum(2)
    dv = (p.transpose(-1, -2).contiguous() @ do).sum(2)
    return dq, dk, dv


def make(b, h, n, layout, g):
    if layout == "tokens":
        return torch.randn(b, n, h, 128, generator=g, device="cuda").bfloat16().transpose(1, 2)
    if layout == "sliced":      # rows that start 16 bytes into wider ones
        return torch.randn(b, h, n, 144, generator=g, device="cuda").bfloat16()[..., 8:136]
    if layout == "far":         # rows 2 MB apart: beyond the 32-bit offsets of all but the general walk
        t = torch.empty(b, n, 2 ** 20, dtype=torch.bfloat16, device="cuda")[..., :128 * h].unflatten(2, (h, 128)).transpose(1, 2)
        return t.copy_(torch.randn(b, h, n, 128, generator=g, device="cuda"))
    return torch.randn(b, h, n, 128, generator=g, device="cuda").bfloat16()


# mode, batch, heads, kv heads, tokens, window | stride, memory slots, causal
CASES = [
    (0, 1, 32, 1, 20, 5, 0, True),            # 32 heads a group: a query is a tile; one work-group
    (0, 1, 16, 1, 65, 0, 0, True),            # a last tile of one key, rows that see themselves alone
    (0, 2, 16, 2, 203, 37, 0, True),
    (0, 1, 3, 3, 1001, 600, 0, True),         # heads not grouped: tiles of 32 queries
    (0, 1, 8, 2, 333, 200, 0, False),
    (0, 2, 8, 8, 300, 40, 0, True),           # few rows a tile: the pipelined walk
    (1, 1, 4, 1, 7, 16, 2, True),             # memory slots alone
    (1, 2, 4, 4, 37, 4, 1, True),
    (1, 2, 8, 2, 515, 8, 3, True),            # 67 rows of k / v: a last tile of three
    (1, 1, 32, 1, 130, 16, 1, True),
    (1, 1, 16, 4, 1111, 5, 0, False),         # a stride that is no power of two
    (1, 1, 8, 1, 4100, 16, 2, True),          # several chunks
]


@pytest.mark.parametrize("mode,b,hq,hk,n,ws,mem,causal,layout", [(*c, layout) for c in CASES for layout in ("heads", "tokens", "sliced")] + [
    (0, 1, 4, 1, 1100, 300, 0, True, "far"),
    (1, 1, 4, 2, 1100, 8, 1, True, "far"),
])
def test_against_float64(mode, b, hq, hk, n, ws, mem, causal, layout):
    """p and dS are rounded to bf16 and so are the results, 2^-9 each; out, which delta is taken from, adds as much to dS."""
    from native_sparse_attention_pytorch_amd import ops
    print(f"case {mode} {b} {hq} {hk} {n} {ws} {mem} {causal} {layout}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + hq)
    window, stride = (ws, 1) if mode == 0 else (0, ws)
    nkeys = n if mode == 0 else n // stride
    q, do = make(b, hq, n, layout, g), make(b, hq, n, layout, g)
    rows = "heads" if layout == "far" else layout
    k, v = make(b, hk, nkeys + mem, rows, g), make(b, hk, nkeys + mem, rows, g)
    scale = 128 ** -0.5
    out, lse, _ = ops.dense_fwd(q, k, v, mode, causal, window, stride, mem, 0, 1, True, scale)
    grads = ops.dense_bwd(q, k, v, out, do, lse, mode, causal, window, stride, mem, scale)
    torch.cuda.synchronize()
    m = visible(mode, n, nkeys, mem, window, stride, causal)
    for name, x, y, tol in zip("qkv", grads, reference(q, k, v, do, m, scale), (2 ** -7, 2 ** -7, 2 ** -8)):
        assert torch.isfinite(x).all(), name
        err = ((x.double() - y).norm() / y.norm().clamp_min(1e-3 * x.numel() ** 0.5)).item()
        assert err < tol, (name, err)


@pytest.mark.parametrize("layout", ["heads", "tokens"])
@pytest.mark.parametrize("mode,n,ws", [(0, 333, 200), (1, 515, 8), (0, 1003, 64)])
def test_rows_behind_a_sequence_are_not_used(mode, n, ws, layout):
    """A last tile reaches behind the sequence: what stands there (another batch entry's rows) takes no part, NaN or not."""
    from native_sparse_attention_pytorch_amd import ops
    print(f"case {mode} {n} {ws} {layout}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    window, stride, mem = (ws, 1, 0) if mode == 0 else (0, ws, 1)
    nkeys = n if mode == 0 else n // stride
    q, do = make(2, 16, n, layout, g), make(2, 16, n, layout, g)
    k, v = make(2, 2, nkeys + mem, layout, g), make(2, 2, nkeys + mem, layout, g)
    res = []
    for bad in (False, True):
        if bad:
            q[1], do[1] = float("nan"), float("nan")
        out, lse, _ = ops.dense_fwd(q, k, v, mode, True, window, stride, mem, 0, 1, True, 128 ** -0.5)
        res.append([t[0].clone() for t in ops.dense_bwd(q, k, v, out, do, lse, mode, True, window, stride, mem, 128 ** -0.5)])
    torch.cuda.synchronize()
    for x, y in zip(*res):
        assert torch.equal(x, y)
