"""The two-layer networks of a bf16 module under autograd as one node (nsa_gemm_bf16, nsa_wgrad_bf16) against the same layers in float64."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _net(k, hidden, out, g):
    r = lambda *s: torch.randn(s, generator=g)
    return [t.to(DEV, torch.bfloat16).requires_grad_() for t in (r(hidden, k) * k ** -0.5, r(hidden) * 0.3, r(out, hidden) * hidden ** -0.5, r(out) * 0.3)]


def _layers(act, x, net, norm_w, residual):
    w1, b1, w2, b2 = net
    y = x if norm_w is None else F.rms_norm(x, norm_w.shape, norm_w, torch.finfo(torch.float32).eps)
    y = F.linear(getattr(F, act)(F.linear(y, w1, b1)), w2, b2)
    return y + x if residual else y


# a row, edges of the 64-row and 128-row tiles, more rows than one slice of the weight gradient, ragged token counts
@pytest.mark.parametrize("rows", (1, 63, 65, 130, 1000, 4100))
@pytest.mark.parametrize("act,k,hidden,out,nets,whole", [("gelu", 128, 384, 128, 1, True), ("relu", 256, 128, 64, 2, False), ("relu", 128, 128, 192, 1, False)])
def test_networks_as_one_node(rows, act, k, hidden, out, nets, whole):
    """Bounds from the roundings: a hidden value is rounded to 8 bits up to twice, so the output and each gradient carry the rounding of
    their own result (2^-9) and those of the values that go into its sums; relative to the norm of the whole tensor 2^-7 covers the four
    roundings of the longest chain (dx: norm, hidden slope, dh, result).  The slope of a ReLU is read from the rounded output: where that
    is 0 the exact value is within its rounding of 0, nothing in norm."""
    from native_sparse_attention_pytorch_amd import ops
    print(rows, act, k, hidden, out, nets, flush=True)
    g = torch.Generator().manual_seed(rows + k)
    xs = [torch.randn(1, rows, k, generator=g).to(DEV, torch.bfloat16).requires_grad_() for _ in range(nets)]
    ws = [_net(k, hidden, out, g) for _ in range(nets)]
    nw = (1 + 0.1 * torch.randn(k, generator=g)).to(DEV, torch.bfloat16).requires_grad_() if whole else None
    douts = [torch.randn(1, rows, out, generator=g).to(DEV, torch.bfloat16) for _ in range(nets)]
    assert ops.mlp_supported(act, xs, [tuple(w) for w in ws], nw)
    ys = ops.mlp(act, xs, [tuple(w) for w in ws], nw, None, residual=whole)
    ys = ys if nets > 1 else (ys,)
    leaves = [*xs, *(t for w in ws for t in w)] + ([nw] if whole else [])
    got = torch.autograd.grad(ys, leaves, douts)
    exact = {t: t.detach().double().requires_grad_() for t in leaves}
    ref = [_layers(act, exact[x], [exact[t] for t in w], exact[nw] if whole else None, whole) for x, w in zip(xs, ws)]
    want = torch.autograd.grad(ref, [exact[t] for t in leaves], [d.double() for d in douts])
    for name, a, b in [*((f"y{i}", a, b) for i, (a, b) in enumerate(zip(ys, ref))), *((f"grad {i}", a, b) for i, (a, b) in enumerate(zip(got, want)))]:
        assert a.shape == b.shape and a.dtype == torch.bfloat16, name
        err = ((a.double() - b).norm() / b.norm()).item()
        assert err < 2 ** -7, (name, err)


# products of 512 tiles of 128 rows and more take those instead of tiles of 64: a last tile of 1, 34, 64, 65 and 128 rows
@pytest.mark.parametrize("rows", (4097, 4130, 4160, 4161, 4224))
@pytest.mark.parametrize("act,k,hidden,out,nets,whole", [("gelu", 128, 2048, 128, 1, True), ("relu", 128, 1024, 64, 2, False), ("gelu", 2048, 128, 2048, 1, True)])
def test_tiles_of_128_rows(rows, act, k, hidden, out, nets, whole):
    """The wide side of each network; the bounds are those of the test above."""
    assert -(-rows // 128) * (max(k, hidden) // 128) * nets >= 512
    test_networks_as_one_node(rows, act, k, hidden, out, nets, whole)


def test_gradients_of_gradients_and_batches_of_them():
    """What the separate layers do beyond one backward pass, by the separate layers."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(3)
    x = torch.randn(2, 40, 128, generator=g).to(DEV, torch.bfloat16).requires_grad_()
    net = _net(128, 256, 128, g)
    nw = torch.ones(128, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    d = torch.randn(3, 2, 40, 128, generator=g).to(DEV, torch.bfloat16)
    run = {"node": lambda: ops.mlp("gelu", [x], [tuple(net)], nw, residual=True), "layers": lambda: _layers("gelu", x, net, nw, True)}
    res = {}
    for name, f in run.items():
        first = torch.autograd.grad(f(), [x, nw, *net], d[0], create_graph=True)
        second = torch.autograd.grad(sum((t.float() ** 2).sum() for t in first), [x, *net[:3]])
        batch = torch.autograd.grad(f(), [x, net[0], net[3]], d, is_grads_batched=True)
        res[name] = [*first, *second, *batch]
    for a, b in zip(res["node"], res["layers"]):
        assert a.shape == b.shape
        assert (a.float() - b.float()).norm() <= 2 ** -6 * b.float().norm()      # (both in bf16, second derivatives of sums of squares)


@pytest.mark.parametrize("act,residual", [("gelu", True), ("relu", False)])
def test_operands_off_a_16_byte_boundary(act, residual):
    """Inputs, norm weight and incoming gradients that are contiguous views at an odd offset."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(5)
    odd = lambda s: torch.randn(1 + s.numel(), generator=g).to(DEV, torch.bfloat16)[1:].view(s)
    shape = torch.Size((3, 50, 128))
    x, d, nw = odd(shape), odd(shape), odd(torch.Size((128,))) if residual else None
    net = _net(128, 256, 128, g)
    assert x.is_contiguous() and x.data_ptr() % 16 and d.data_ptr() % 16
    res = []
    for t, e, w in ((x, d, nw), (x.clone(), d.clone(), None if nw is None else nw.clone())):
        leaves = [t.requires_grad_(), *net] + ([w.requires_grad_()] if residual else [])
        assert ops.mlp_supported(act, [t], [tuple(net)], w)
        y = ops.mlp(act, [t], [tuple(net)], w, residual=residual)
        res.append([y, *torch.autograd.grad(y, leaves, e)])
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_what_the_node_does_not_take():
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(1)
    x = torch.randn(10, 128, generator=g).to(DEV, torch.bfloat16)
    net = tuple(_net(128, 128, 64, g))
    assert ops.mlp_supported("relu", [x], [net])
    assert not ops.mlp_supported("relu", [x.float()], [net]) and not ops.mlp_supported("relu", [x[:, :64]], [net])
    assert not ops.mlp_supported("relu", [x], [(net[0], None, *net[2:])]) and not ops.mlp_supported("relu", [x], [(net[0].t(), *net[1:])])
    assert not ops.mlp_supported("relu", [x, x[:5]], [net, net]) and not ops.mlp_supported("relu", [x[:0]], [net])
    with torch.no_grad():
        assert not ops.mlp_supported("relu", [x], [net])
    with torch.autocast("cuda", torch.bfloat16):
        assert not ops.mlp_supported("relu", [x], [net])


@pytest.mark.parametrize("rows,n_out,n_in,pad", [(1, 64, 128, 0), (200, 192, 128, 64), (4080, 64, 256, 0), (4097, 256, 384, 8)])
def test_weight_gradients(rows, n_out, n_in, pad):
    """bf16 roundings of exact sums: one rounding of the result, 2^-9 relative, and the fp32 sums' rounding below it."""
    from native_sparse_attention_pytorch_amd import ops
    g = torch.Generator().manual_seed(rows)
    dy = torch.randn(rows, n_out + pad, generator=g).to(DEV, torch.bfloat16)[:, :n_out]
    x = torch.randn(rows, n_in + pad, generator=g).to(DEV, torch.bfloat16)[:, pad:]
    with torch.no_grad():
        assert ops._wgrad_supported(dy, x, torch.bfloat16)
        (dw, db), = ops._wgrad_bf16([(dy, x)], True)
    for a, b in ((dw, dy.double().t() @ x.double()), (db, dy.double().sum(0))):
        assert ((a.double() - b).norm() <= 2 ** -8.5 * b.norm()).item()


def test_lines_of_the_rules(monkeypatch):
    """Either side of each line, by sizes alone (nothing is launched)."""
    from native_sparse_attention_pytorch_amd import ops
    z = lambda *s: torch.empty(s, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    net = lambda k, hidden, out: (z(hidden, k), z(hidden), z(out, hidden), z(out))
    block = lambda rows, k, hidden: ops.mlp_supported("gelu", [z(rows, k)], [net(k, hidden, k)])
    pair = lambda rows, k, out: ops.mlp_supported("relu", [z(rows, k)] * 2, [net(k, k, out)] * 2)
    assert block(3072, 1024, 4096) and not block(3073, 1024, 4096) and block(16384, 512, 2048) and block(8192, 1024, 2048) and not block(8192, 1024, 3072)
    assert pair(4080, 2048, 64) and not pair(1000, 4096, 128)

    def wgrad(rows, n_in, n_out, sums):
        with torch.no_grad():
            return ops._wgrad_supported(z(rows, n_out).detach(), z(rows, n_in).detach(), torch.bfloat16, sums)
    assert wgrad(2049, 2048, 1024, False) and not wgrad(2048, 2048, 1024, False) and not wgrad(2048, 2048, 1024, True)
    assert wgrad(600, 512, 512, False) and not wgrad(599, 512, 512, False) and wgrad(8, 512, 512, True)
    assert wgrad(8192, 512, 1024, False) and not wgrad(16384, 1024, 1024, True) and wgrad(16384, 1024, 64, False)
    monkeypatch.setattr(ops, "capturing", lambda: True)
    assert block(1000, 512, 2048) and not block(500, 512, 2048) and not block(2048, 1024, 4096) and not block(16384, 1024, 2048) and pair(64, 1024, 64)
    assert not wgrad(8192, 512, 1024, False) and wgrad(8192, 512, 1024, True) and wgrad(8192, 512, 512, False)
