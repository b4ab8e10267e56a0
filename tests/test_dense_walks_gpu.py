"""The dK / dV walks of interval-masked attention at 128 features that take what the walk with one wave per tile refuses - a scale that is not
positive, tokens of K and V 32 MB apart - against the same attention in float64."""

import pytest
import torch

from tests.test_dense_keys_gpu import reference, visible

pytestmark = pytest.mark.gpu


# mode, heads, kv heads, tokens, window | stride, memory slots, causal
@pytest.mark.parametrize("mode,hq,hk,n,ws,mem,causal", [(0, 8, 2, 203, 170, 0, True), (0, 8, 2, 130, 60, 0, False), (1, 8, 2, 515, 8, 3, True),
                                                          (1, 4, 4, 700, 16, 1, True), (1, 16, 4, 333, 5, 0, False)])
@pytest.mark.parametrize("scale,spread", [(-0.1, False), (0.1, True)])
def test_against_float64(mode, hq, hk, n, ws, mem, causal, scale, spread):
    """p and dS are rounded to bf16 and so are the results, 2^-9 each; out, which delta is taken from, adds as much to dS."""
    from native_sparse_attention_pytorch_amd import ops
    print(f"case {mode} {hq} {hk} {n} {ws} {mem} {causal} {scale} {spread}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + hq)
    window, stride = (ws, 1) if mode == 0 else (0, ws)
    nkeys = n if mode == 0 else n // stride
    make = lambda h, m: torch.randn(1, h, m, 128, generator=g, device="cuda").bfloat16()
    q, do, k, v = make(hq, n), make(hq, n), make(hk, nkeys + mem), make(hk, nkeys + mem)
    m = visible(mode, n, nkeys, mem, window, stride, causal)
    want = reference(q, k, v, do, m, scale)
    s = (q.double().unflatten(1, (hk, hq // hk)) @ k.double().transpose(-1, -2).contiguous()[:, :, None]).mul(scale).masked_fill(~m, -torch.inf)
    lse = s.logsumexp(-1)
    out = ((s - lse[..., None]).exp() @ v.double()[:, :, None]).flatten(1, 2).bfloat16()
    if spread:
        rows = lambda t: torch.empty(((t.shape[2] - 1) << 24) + hk * 128, dtype=t.dtype, device="cuda").as_strided(t.shape, (t.shape[2] << 24, 128, 1 << 24, 1)).copy_(t)
        k, v = rows(k), rows(v)
    grads = ops.dense_bwd(q, k, v, out, do, lse.flatten(1, 2).float(), mode, causal, window, stride, mem, scale)
    torch.cuda.synchronize()
    for name, x, y, tol in zip("qkv", grads, want, (2 ** -7, 2 ** -7, 2 ** -8)):
        assert torch.isfinite(x).all(), name
        err = ((x.double() - y).norm() / y.norm()).item()
        assert err < tol, (name, err)
