"""Gradients taken inside an autocast region, where matrix products come out in the autocast type: what reaches a kernel by address
keeps the type the kernel reads."""
import pytest
import torch

from native_sparse_attention_pytorch_amd import _lib, ops


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("share", [True, False])
def test_importance_products_stay_fp32(dtype, share):
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g)
    q, ck, dp = r(2, 4, 24, 16).bfloat16(), r(2, 2, 9, 16).bfloat16(), r(2, 2 if share else 4, 24, 4)
    want = ops._importance_products_backward(q, ck, dp, 1, 4, 8, share, 0.25)
    with torch.autocast("cpu", dtype=dtype):
        got = ops._importance_products_backward(q, ck, dp, 1, 4, 8, share, 0.25)
    assert got[0].dtype == got[1].dtype == torch.float32
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and got[2] == want[2]


def test_a_summand_of_another_type_is_refused(monkeypatch):
    monkeypatch.setattr(_lib, "lib", lambda: pytest.fail("reached the library"))
    base = torch.zeros(1, 2, 8, 16, dtype=torch.bfloat16)
    for b, small in ((base, torch.zeros(1, 2, 8, 16, dtype=torch.bfloat16)), (base.half(), torch.zeros(1, 2, 8, 16)), (base, torch.zeros(1, 3, 8, 16)),
                     (base, torch.zeros(1, 2, 8, 8)), (base.transpose(1, 2), torch.zeros(1, 8, 2, 16))):
        with pytest.raises(RuntimeError):
            ops._add_repeated(b, small, torch.empty_like(base), 1, 0, 1, 1.0)


def test_scores_of_another_type_are_refused(monkeypatch):
    """The masked top-k and the gradient of its values read fp32 rows, as the top-k itself, which refuses others."""
    class OnDevice(torch.Tensor):
        is_cuda = True
    monkeypatch.setattr(_lib, "lib", lambda: pytest.fail("reached the library"))
    dev = lambda *s, dtype=torch.float32: torch.zeros(s, dtype=dtype).as_subclass(OnDevice)
    half, raw = dev(1, 2, 8, 4, dtype=torch.bfloat16), (0.25, 8, 2, 2)
    for call in (lambda: ops.importance_topk(half, 2, raw=raw), lambda: ops.importance_topk(torch.zeros(1, 2, 8, 4), 2, raw=raw),
                 lambda: ops.topk_bwd._init_fn(half, dev(1, 2, 8, 2, dtype=torch.int32), dev(1, 2, 8, 2)),
                 lambda: ops.topk_bwd._init_fn(dev(1, 2, 8, 4), dev(1, 2, 8, 2, dtype=torch.int64), dev(1, 2, 8, 2)),
                 lambda: ops.topk_bwd._init_fn(dev(1, 2, 8, 4), dev(1, 2, 8, 2, dtype=torch.int32), dev(1, 2, 8, 3)),
                 lambda: ops.topk_bwd._init_fn(dev(1, 2, 8, 4), dev(1, 2, 6, 2, dtype=torch.int32), dev(1, 2, 6, 2))):
        with pytest.raises(RuntimeError):
            call()


@pytest.mark.gpu
@pytest.mark.parametrize("share", [True, False])
def test_backward_inside_autocast_equals_backward_outside(share):
    """Differentiable top-k: the importance gradient joins the attention's.  The same module, the same forward outside autocast."""
    from native_sparse_attention_pytorch_amd import SparseAttention
    torch.manual_seed(0)
    with torch.device("cuda"):
        m = SparseAttention(dim=128, dim_head=64, heads=4, kv_heads=2, causal=True, sliding_window_size=16, compress_block_size=16, use_diff_topk=True,
                            compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2, query_heads_share_selected_kv=share).bfloat16()
        x, dy = torch.randn(2, 2, 200, 128, dtype=torch.bfloat16).unbind()
    grads = []
    for inside in (False, True):
        m.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_()
        y = m(xi)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=inside):
            y.backward(dy)
        grads.append([xi.grad] + [p.grad for p in m.parameters() if p.grad is not None])
    torch.cuda.synchronize()
    for a, b in zip(*grads):
        # (sums of other operators may be taken in bf16 there: within their rounding)
        assert (a.float() - b.float()).norm() <= 1e-2 * a.float().norm() + 1e-6
