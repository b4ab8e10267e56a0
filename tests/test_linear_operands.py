"""What the projection kernels for a few rows are handed (`ops.skinny_linear`, `ops.linear_f32` and the decode paths around them), with the
library replaced by a recorder: they read a weight as contiguous rows of the input's type in device memory, so everything else is
refused, copied or left to the layer, as F.linear would have it."""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from native_sparse_attention_pytorch_amd import SparseAttention, _lib, ops
from native_sparse_attention_pytorch_amd.transformer import FeedForward, Transformer

BF16, F32 = torch.bfloat16, torch.float32


class OnDevice(torch.Tensor):
    """A CPU tensor that says it lies on the GPU: with the library replaced nothing reads its address."""
    is_cuda = True


@pytest.fixture
def calls(monkeypatch):
    """(name, arguments) of every library call."""
    seen = []

    class Recorder:
        def __getattr__(self, name):
            return lambda *args: seen.append((name, args)) or 0

    monkeypatch.setattr(_lib, "lib", Recorder)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    return seen


def _dev(*shape, dtype=BF16):
    return torch.ones(shape, dtype=dtype).as_subclass(OnDevice)


KERNELS = [(ops.skinny_linear, BF16), (ops.linear_f32, F32)]


@pytest.mark.parametrize("fn, dtype", KERNELS)
def test_weights_and_inputs_the_kernel_cannot_read_are_refused(calls, fn, dtype):
    other = F32 if dtype == BF16 else BF16
    x = _dev(4, 64, dtype=dtype)
    for args in ((x, _dev(16, 64, dtype=other)), (x, torch.ones(16, 64, dtype=dtype, device="meta")), (torch.ones(4, 64, dtype=dtype), _dev(16, 64, dtype=dtype)),
                 (_dev(4, 64, dtype=other), _dev(16, 64, dtype=other)), (x, _dev(64, dtype=dtype))):
        with pytest.raises(RuntimeError):
            fn(*args)
    assert not calls


@pytest.mark.parametrize("fn, dtype", KERNELS)
def test_a_weight_that_is_not_contiguous_is_copied(calls, fn, dtype):
    w = _dev(64, 16, dtype=dtype).t()
    fn(_dev(4, 64, dtype=dtype), w)
    (_, args), = calls
    assert w.data_ptr() not in args


def _odd(linear, how):
    """`linear` with a weight the kernel must not be handed."""
    w = linear.weight.detach()
    if how == "fp32":
        linear.weight = nn.Parameter(w.float())
    elif how == "strided":
        linear.weight = nn.Parameter(w.t().contiguous().t())
    elif how == "offset":                                     # a slice of a flat buffer, off a 16-byte boundary
        flat = torch.zeros(w.numel() + 1, dtype=w.dtype)
        linear.weight = nn.Parameter(flat[1:].view(w.shape).copy_(w))
    return linear


@pytest.mark.parametrize("how", ["plain", "fp32", "strided", "offset"])
def test_second_projections_the_kernel_cannot_read_stay_with_the_layer(calls, monkeypatch, how):
    """The compression network's and the feed-forward block's second linear: its call is the layer's own (which refuses fp32)."""
    m = SparseAttention(dim=128, dim_head=64, heads=4, kv_heads=2, causal=True, sliding_window_size=16, compress_block_size=16,
                        compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2).to(BF16)
    ff = FeedForward(64).to(BF16)
    layers = []
    for down, run in ((m.k_compress[3], lambda: m._compress_rows(m.k_compress, _dev(2, 2, 16, 64))), (ff[3], lambda: Transformer._decode_feed_forward(ff, _dev(2, 1, 64)))):
        if how == "plain":
            with torch.no_grad():
                assert run().shape[-1] == down.out_features
            assert [name for name, _ in calls] == ["nsa_skinny_linear"] * 2
            calls.clear()
            continue
        w = _odd(down, how).weight
        with monkeypatch.context() as patch, torch.no_grad():
            patch.setattr(F, "linear", lambda x, w, b=None: layers.append(w) or torch.zeros(*x.shape[:-1], w.shape[0], dtype=BF16))
            assert run().shape[-1] == down.out_features
        assert not calls and any(u is w for u in layers)
        layers.clear()


def _off_boundary(t):
    flat = torch.zeros(t.numel() + 1, dtype=t.dtype)
    return flat[1:].view(t.shape).copy_(t)


def _decode_layer(norm_weight=None, out_bias=None):
    m = SparseAttention(dim=128, dim_head=64, heads=4, kv_heads=2, causal=True, sliding_window_size=16, compress_block_size=16,
                        compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2).to(BF16)
    if norm_weight is not None:
        m.norm.weight = nn.Parameter(norm_weight(m.norm.weight.detach()))
    if out_bias is not None:
        m.combine_heads.bias = nn.Parameter(out_bias)
    z = lambda rows: torch.zeros(2, 2, rows, 64, dtype=BF16)
    return m, ((z(40), z(40)), ((z(5), z(5)), (z(8), z(8))))


@pytest.mark.parametrize("vector", ["norm weight off a boundary", "bias of one element"])
def test_vectors_the_kernel_cannot_read_stay_with_the_layers(calls, monkeypatch, vector):
    """A decode step, a feed-forward block and the logits whose norm weight lies elsewhere or whose bias is broadcast."""
    norm_weight = _off_boundary if vector.startswith("norm") else None
    bias = None if norm_weight else torch.ones(1, dtype=BF16)
    m, cache = _decode_layer(norm_weight, bias)
    monkeypatch.setattr(ops, "decode_step", lambda q, *a, **kw: (_dev(2, 1, 256), None, None))
    with torch.no_grad():
        m.forward_inference(_dev(2, 1, 128), cache)
    assert "nsa_decode_layer" not in [n for n, _ in calls] and len(calls) == (1 if norm_weight else 2)       # output projection; qkv and gate logits
    calls.clear()

    model = Transformer(num_tokens=16, dim=64, depth=0).to(BF16)
    ff = FeedForward(64).to(BF16)
    if norm_weight:
        for norm in (ff[0], model.norm):
            norm.weight = nn.Parameter(_off_boundary(norm.weight.detach()))
    else:
        ff[1].bias, model.to_logits.bias = nn.Parameter(bias), nn.Parameter(bias)
    with torch.no_grad():
        assert Transformer._decode_feed_forward(ff, _dev(2, 1, 64)).shape == (2, 1, 64)
        assert model._decode_logits(_dev(2, 1, 64)).shape == (2, 1, 16)
    assert not calls


def test_inputs_off_a_boundary_are_copied(calls):
    x = _off_boundary(torch.ones(4, 64, dtype=BF16)).as_subclass(OnDevice)
    ops.skinny_linear(x, _dev(16, 64), norm_weight=_off_boundary(torch.ones(64, dtype=BF16)).as_subclass(OnDevice))
    (_, args), = calls
    assert x.data_ptr() not in args and args[3] % 16 == 0 and args[5] % 16 == 0


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("hook", ["register_forward_hook", "register_forward_pre_hook"])
def test_hooks_on_the_flatten_layer_run(calls, dtype, hook):
    """The compression network's first layer is its own call whenever something hangs on it."""
    m = SparseAttention(dim=128, dim_head=64, heads=4, kv_heads=2, causal=True, sliding_window_size=16, compress_block_size=8,
                        compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2).to(dtype)
    run = (lambda: m._compress_rows(m.k_compress, _dev(2, 2, 8, 64))) if dtype == BF16 else (lambda: m._compress(m.k_compress, _dev(2, 2, 3, 8, 64, dtype=F32)))
    with torch.no_grad():
        run()
        assert calls
        seen = []
        getattr(m.k_compress[0], hook)(lambda *args: seen.append(len(args)) or None)
        run()
    assert len(seen) == 1


def test_gate_logits_in_host_memory_are_refused(calls):
    branch = torch.zeros(1, 2, 3, 8).as_subclass(OnDevice)
    for logits in (torch.zeros(1, 3, 6, device="meta"), torch.zeros(1, 3, 6, dtype=BF16), torch.zeros(1, 3, 5)):
        with pytest.raises(RuntimeError):
            ops.gate_combine_f32(logits, branch, branch, branch)
    assert not calls


@pytest.mark.parametrize("rows, k, n, own", [
    (62, 512, 1536, True), (240, 512, 24, True), (256, 512, 256, True),       # the smallest layer's projections; few outputs
    (256, 512, 1536, False), (128, 512, 3072, False), (256, 256, 6144, False),    # more tiles than the chip takes at once
    (256, 256, 1024, True), (160, 256, 2048, False),
    (8, 512, 512, False), (31, 320, 300, False), (1, 512, 512, True), (32, 512, 512, True), (8, 256, 512, True),
    (257, 64, 64, False), (8, 520, 64, False), (8, 60, 64, False),
])
def test_fp32_projections_that_the_library_serves_better_stay_with_it(rows, k, n, own):
    assert ops.linear_f32_supported(_dev(rows, k, dtype=F32), _dev(n, k, dtype=F32)) is own
