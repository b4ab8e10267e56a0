"""A directly launched decode session takes what a replayed one takes, and is not disturbed by what happens around it."""
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu
DEV, BF16 = "cuda", torch.bfloat16


def _session(b=4, dim=128, heads=4, kv_heads=2):
    from native_sparse_attention_pytorch_amd import SparseAttention
    from native_sparse_attention_pytorch_amd.decode_session import DecodeSession
    torch.manual_seed(b)
    m = SparseAttention(dim=dim, dim_head=64, heads=heads, kv_heads=kv_heads, causal=True, sliding_window_size=16, compress_block_size=16,
                        compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2).to(DEV, BF16)
    with torch.no_grad():
        _, cache = m(torch.randn(b, 37, dim, device=DEV, dtype=BF16), return_cache=True)
        return m, cache, DecodeSession(m, cache, max_len=64)


def _off_boundary(t):
    flat = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
    return nn.Parameter(flat[1:].view(t.shape).copy_(t.detach()))


def _strided_bias(m):
    m.combine_heads.bias = nn.Parameter(torch.randn(256, device=DEV, dtype=BF16)[::2])


def _bias_of_one(m):
    m.combine_heads.bias = nn.Parameter(torch.randn(1, device=DEV, dtype=BF16))


def _weight_off_boundary(m):
    m.combine_heads.weight = _off_boundary(m.combine_heads.weight)


def _norm_off_boundary(m):
    m.norm.weight = _off_boundary(m.norm.weight)


@pytest.mark.parametrize("change", [_strided_bias, _bias_of_one, _weight_off_boundary, _norm_off_boundary])
def test_parameters_of_other_layouts(change):
    m, cache, session = _session()                        # (the parallel forward's norm kernel refuses a weight off a boundary)
    change(m)
    session = type(session)(m, cache, max_len=64)
    x = torch.randn(4, 1, 128, device=DEV, dtype=BF16)
    with torch.no_grad():
        want = m(x, cache=cache, return_cache=True)[0]
    got = session.step(x)
    torch.cuda.synchronize()
    # the same partial sums merged in another order, then one bf16 projection of 256 products: two roundings of its magnitude
    mag = want.float().abs().max().item()
    assert (got.float() - want.float()).abs().max().item() <= 2 ** -6 * mag


def test_tokens_are_taken_as_a_copy_into_the_buffer_takes_them():
    """`x` is broadcast to 'b 1 dim' and converted; what cannot be broadcast is refused."""
    m, cache, first = _session()
    one = torch.randn(128, device=DEV, dtype=BF16)
    want = first.step(one.expand(4, 1, 128).contiguous())
    for x in (one, one[None], one.view(1, 1, 128), one.expand(4, 1, 128), one.float().view(1, 1, 128), one.cpu()):
        assert torch.equal(type(first)(m, cache, max_len=64).step(x), want)
    for shape in ((4, 128), (1, 4, 128), (4, 2, 128), (512,)):
        with pytest.raises(RuntimeError):
            type(first)(m, cache, max_len=64).step(torch.zeros(shape, device=DEV, dtype=BF16))


def test_a_module_moved_afterwards_leaves_the_session_with_its_weights():
    """The session keeps the memory its steps read: moving the module's parameters away neither changes nor invalidates it."""
    m, cache, first = _session()
    x = torch.randn(4, 1, 128, device=DEV, dtype=BF16)
    want = first.step(x)
    second = type(first)(m, cache, max_len=64)
    m.norm.cpu(), m.combine_heads.cpu()
    assert torch.equal(second.step(x), want)
    third = type(first)(m.to(DEV), cache, max_len=64)
    with torch.no_grad():
        m.combine_heads.weight.mul_(2)                                 # values changed in place are followed, as by a replayed step
    torch.testing.assert_close(third.step(x), want * 2, rtol=0, atol=0)


def test_autocast_around_a_step_changes_nothing():
    """A direct step whose output projection is the library's: bf16, as a recorded step leaves it whatever the step is run under."""
    m, cache, _ = _session(dim=4096, heads=48, kv_heads=8)              # (35 MB of qkv and gate weights: launched directly)
    _bias_of_one(m)
    from native_sparse_attention_pytorch_amd.decode_session import DecodeSession
    sessions = [DecodeSession(m, cache, max_len=64) for _ in range(2)]
    assert sessions[0].direct and not sessions[0].own_out
    x = torch.randn(4, 1, 4096, device=DEV, dtype=BF16)
    with torch.autocast("cuda", dtype=torch.float16):
        got = sessions[0].step(x)
    assert got.dtype == BF16 and torch.equal(got, sessions[1].step(x))


def test_a_step_cannot_be_recorded():
    """The host's position would stand still while a replay moves the device's: refused, as replaying a graph inside a capture is."""
    m, cache, session = _session()
    x = torch.randn(4, 1, 128, device=DEV, dtype=BF16)
    kept, graph = torch.ones(4, device=DEV), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kept.add_(1)
        with pytest.raises(RuntimeError, match="recorded"):
            session.step(x)
    assert session.pos == 37
    assert torch.equal(session.step(x), type(session)(m, cache, max_len=64).step(x))


def test_a_direct_session_records_a_step_only_for_a_caller_that_replays_it():
    m, cache, session = _session()
    x = torch.randn(4, 1, 128, device=DEV, dtype=BF16)
    assert session.direct and session._graphs[0] is None and session._graphs[1] is not None
    session.x_buf.copy_(x)
    for replay in range(3):
        session.state[0] = 37
        session.graphs[0].replay()
        torch.cuda.synchronize()
        assert torch.equal(session.outs[0], type(session)(m, cache, max_len=64).step(x)) and int(session.state[0]) == 38
