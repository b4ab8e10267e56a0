"""What `SparseAttention._decode_whole` may hand to the kernels: caches and weights whose shapes agree.  The library call takes batch,
heads and lengths from one tensor of each pair, so everything else goes to the general path, which refuses it."""
import itertools

import pytest
import torch
from torch import nn

from native_sparse_attention_pytorch_amd import SparseAttention, ops
from native_sparse_attention_pytorch_amd.transformer import Transformer

BF16 = torch.bfloat16


def _layer_and_cache(b=4, n=40, hk=2, d=64):
    m = SparseAttention(dim=128, dim_head=d, heads=4, kv_heads=hk, causal=True, sliding_window_size=16, compress_block_size=16,
                        compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2).to(BF16)
    z = lambda rows, batch=b, heads=hk, width=d: torch.zeros(batch, heads, rows, width, dtype=BF16)
    return m, z, ((z(n), z(n)), ((z(n // 8), z(n // 8)), (z(8), z(8))))


@pytest.fixture
def reached(monkeypatch):
    calls = []

    def decode_step(*args, layer=None, **kwargs):
        calls.append(layer)
        return (torch.zeros_like(layer.x),)

    monkeypatch.setattr(ops, "decode_step", decode_step)
    return calls


class OnDevice(torch.Tensor):
    """A CPU tensor that says it lies on the GPU: with the library call replaced nothing reads its address."""
    is_cuda = True


def _run(m, cache, b=4):
    with torch.no_grad():
        return m._decode_whole(torch.zeros(b, 1, 128, dtype=BF16).as_subclass(OnDevice), cache)


def test_matching_shapes_take_the_call(reached):
    m, _, cache = _layer_and_cache()
    assert _run(m, cache) is not None and len(reached) == 1


@pytest.mark.parametrize("pair", [0, 1, 2])
@pytest.mark.parametrize("member", [0, 1])
@pytest.mark.parametrize("change", ["batch", "heads", "rows"])
def test_caches_that_disagree_do_not(reached, pair, member, change):
    m, z, ((k, v), ((ck, cv), (rk, rv))) = _layer_and_cache()
    pairs = [[k, v], [ck, cv], [rk, rv]]
    rows = pairs[pair][member].shape[2]
    pairs[pair][member] = dict(batch=z(rows, batch=2), heads=z(rows, heads=1), rows=z(rows - 1))[change]
    assert _run(m, (tuple(pairs[0]), (tuple(pairs[1]), tuple(pairs[2])))) is None and not reached


def test_all_caches_of_another_batch_do_not(reached):
    m, _, cache = _layer_and_cache(b=2)
    assert _run(m, cache) is None and not reached


@pytest.mark.parametrize("name, features", [("to_qkv", (128, 256)), ("to_qkv", (64, 512)), ("combine_heads", (256, 64)), ("combine_heads", (128, 128))])
def test_replaced_projections_of_another_size_do_not(reached, name, features):
    m, _, cache = _layer_and_cache()
    setattr(m, name, nn.Linear(*features, bias=False).to(BF16))
    assert _run(m, cache) is None and not reached


def test_host_tensors_never_reach_the_library(reached):
    """The library takes addresses: a layer, its caches or its frequencies in host memory are refused, whatever the grad mode."""
    m, _, cache = _layer_and_cache()
    with torch.no_grad():
        assert m._decode_whole(torch.zeros(4, 1, 128, dtype=BF16), cache) is None
        with pytest.raises(RuntimeError, match="GPU only"):
            m(torch.zeros(4, 1, 128, dtype=BF16), cache=cache)
    m.rotary_emb.freqs = nn.Parameter(m.rotary_emb.freqs.to("meta"), requires_grad=False)
    assert _run(m, cache) is None and not reached


@pytest.mark.parametrize("grad", [False, True])
def test_a_model_in_host_memory_is_refused(reached, grad):
    m = Transformer(num_tokens=16, dim=128, depth=2, heads=4, kv_heads=2, sparse_attn_kwargs=dict(
        sliding_window_size=16, compress_block_size=16, compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2)).to(BF16)
    _, _, cache = _layer_and_cache()
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="GPU only"):
        m(torch.zeros(4, 1, dtype=torch.long), cache=[cache, cache])
    assert not reached


def test_a_model_that_is_not_causal_is_refused(reached, monkeypatch):
    m = Transformer(num_tokens=16, dim=128, depth=1, heads=4, kv_heads=2, causal=False, sparse_attn_kwargs=dict(
        sliding_window_size=16, compress_block_size=16, compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2)).to(BF16)
    embedded = torch.zeros(4, 1, 128, dtype=BF16).as_subclass(OnDevice)
    monkeypatch.setattr(m.token_emb, "forward", lambda ids: embedded)
    _, _, cache = _layer_and_cache()
    with torch.no_grad(), pytest.raises(AssertionError, match="autoregressive"):
        m(torch.zeros(4, 1, dtype=torch.long), cache=[cache])
    assert not reached


@pytest.mark.parametrize("name, shape", [("to_strategy_combine.0.bias", (1,)), ("to_strategy_combine.0.bias", (6,)), ("combine_heads.bias", (1,)),
                                         ("norm.weight", (1,)), ("compress_mem_kv", (1, 2, 1, 64))])
def test_replaced_vectors_of_another_size_do_not(reached, name, shape):
    """The kernels read a whole vector from each; the layers broadcast or refuse the others."""
    m, _, cache = _layer_and_cache()
    owner, _, leaf = name.rpartition(".")
    setattr(m.get_submodule(owner), leaf, nn.Parameter(torch.zeros(shape, dtype=BF16)))
    assert _run(m, cache) is None and not reached


def _model_with_spied_layers(monkeypatch, depth=2):
    m = Transformer(num_tokens=16, dim=128, depth=depth, heads=4, kv_heads=2, sparse_attn_kwargs=dict(
        sliding_window_size=16, compress_block_size=16, compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2)).to(BF16)
    handed = []
    for i, (attn, _) in enumerate(m.layers):
        def forward(tokens, cache=None, return_cache=False, i=i):
            handed.append((i, cache))
            return torch.zeros_like(tokens), ("advanced", i)
        monkeypatch.setattr(attn, "forward", forward)
        monkeypatch.setattr(attn, "_decode_whole", lambda *a, **kw: None)
    return m, handed


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("kind", ["list", "tuple", "iterator", "endless", "longer"])
def test_layer_caches_from_any_iterable(monkeypatch, kind, grad):
    """One cache per layer, from whatever yields them; what is left over is not read."""
    m, handed = _model_with_spied_layers(monkeypatch)
    caches = {"list": ["a", "b"], "tuple": ("a", "b"), "iterator": iter("ab"), "endless": itertools.cycle("ab"), "longer": ["a", "b", "c"]}[kind]
    with torch.set_grad_enabled(grad):
        logits, new = m(torch.zeros(3, 5, dtype=torch.long), cache=caches, return_cache=True)
    assert handed == [(0, "a"), (1, "b")] and new == [("advanced", 0), ("advanced", 1)] and logits.shape == (3, 1, 16)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("caches", [[None, "b"], ["a"], []])
def test_a_layer_without_a_cache_starts_one(monkeypatch, caches, grad):
    m, handed = _model_with_spied_layers(monkeypatch)
    with torch.set_grad_enabled(grad):
        m(torch.zeros(3, 5, dtype=torch.long), cache=caches, return_cache=True)
    assert [c for _, c in handed] == (caches + [None, None])[:2]


def test_a_missing_cache_does_not_reach_the_layer_call():
    m, _, _ = _layer_and_cache()
    model = Transformer(num_tokens=16, dim=128, depth=1, heads=4, kv_heads=2).to(BF16)
    model.layers[0][0] = m
    with torch.no_grad(), pytest.raises(RuntimeError, match="GPU only"):      # the layer's own forward, which has no CPU path
        model(torch.zeros(4, 1, dtype=torch.long), cache=[None])


def test_layers_whose_forward_was_replaced_are_called(reached, monkeypatch):
    """A forward put on the instance (as offloading and tracing tools do) runs, for the layer itself and for the layers inside it."""
    m, _, cache = _layer_and_cache()
    seen = []
    for layer in (m.norm, m.to_qkv, m.to_strategy_combine[0], m.combine_heads):
        with monkeypatch.context() as patch:
            patch.setattr(layer, "forward", lambda x: seen.append(1) or x)
            assert _run(m, cache) is None and not reached
            if isinstance(layer, nn.Linear):
                SparseAttention._linear(layer, torch.zeros(1, 128, dtype=BF16))
    assert len(seen) == 3
    model = Transformer(num_tokens=16, dim=128, depth=1, heads=4, kv_heads=2).to(BF16)
    model.layers[0][0] = m
    monkeypatch.setattr(m, "forward", lambda tokens, cache=None, return_cache=False: (seen.append("attn") or torch.zeros_like(tokens), cache))
    monkeypatch.setattr(model.token_emb, "forward", lambda ids: torch.zeros(4, 1, 128, dtype=BF16).as_subclass(OnDevice))
    monkeypatch.setattr(model, "_decode_feed_forward", lambda ff, tokens: tokens)
    monkeypatch.setattr(model, "_decode_logits", lambda tokens: tokens)
    with torch.no_grad():
        model(torch.zeros(4, 1, dtype=torch.long), cache=[cache])
    assert seen[-1] == "attn" and not reached


def test_calls_that_are_not_plain_do_not(reached, monkeypatch):
    """Autocast, tracers and transforms around a step (ops.plain_call): the general path, from the layer and from the model."""
    m, _, cache = _layer_and_cache()
    model = Transformer(num_tokens=16, dim=128, depth=1, heads=4, kv_heads=2).to(BF16)
    model.layers[0][0] = m
    x = torch.zeros(4, 1, 128, dtype=BF16).as_subclass(OnDevice)
    monkeypatch.setattr(model.token_emb, "forward", lambda ids: x)

    class General(Exception):
        pass

    def split(self, t):
        raise General
    monkeypatch.setattr(SparseAttention, "_split_heads", split)
    for run in (lambda: m(x, cache=cache), lambda: model(torch.zeros(4, 1, dtype=torch.long), cache=[cache])):
        monkeypatch.setattr(ops, "plain_call", lambda: False)
        with torch.no_grad(), pytest.raises(General):
            run()
    assert not reached


def test_plain_calls():
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    assert ops.plain_call()
    seen = []
    look = lambda t: seen.append(ops.plain_call()) or t + 1
    one = torch.ones(2)
    torch.vmap(look)(one), torch.func.jvp(look, (one,), (one,)), make_fx(look)(one), make_fx(look, pre_dispatch=True)(one)
    torch.jit.trace(look, (one,), check_trace=False)
    with forward_ad.dual_level():
        look(one)
    assert seen and not any(seen) and ops.plain_call()
