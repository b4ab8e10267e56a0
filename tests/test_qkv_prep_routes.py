"""Which fp32 layers hand rotation and window split to the kernel: those whose frequencies and positions are the tensors
the kernel reads; the others keep the operators, which broadcast or refuse."""
import pytest
import torch
from torch import nn

from native_sparse_attention_pytorch_amd import SparseAttention, _lib, ops


class OnDevice(torch.Tensor):
    """A CPU tensor that says it lies on the GPU: with the library replaced nothing reads its address."""
    is_cuda = True


def _layer():
    return SparseAttention(dim=128, dim_head=64, heads=4, kv_heads=2, causal=True, sliding_window_size=16, compress_block_size=16,
                           compress_block_sliding_stride=8, selection_block_size=16, num_selected_blocks=2)


CHANGES = {
    "positions of one head": lambda m: setattr(m, "k_intrablock_positions", nn.Parameter(torch.zeros(1, 16, 64))),
    "positions of one row": lambda m: setattr(m, "v_intrablock_positions", nn.Parameter(torch.zeros(2, 1, 64))),
    "positions elsewhere": lambda m: setattr(m, "v_intrablock_positions", nn.Parameter(torch.zeros(2, 16, 64, device="meta"))),
    "frequencies elsewhere": lambda m: setattr(m.rotary_emb, "freqs", nn.Parameter(m.rotary_emb.freqs.to("meta"), requires_grad=False)),
    "fewer frequencies": lambda m: setattr(m.rotary_emb, "freqs", nn.Parameter(m.rotary_emb.freqs[:1].clone(), requires_grad=False)),
}


@pytest.mark.parametrize("change", CHANGES)
def test_tensors_the_kernel_cannot_read(monkeypatch, change):
    monkeypatch.setattr(_lib, "lib", lambda: pytest.fail("reached the library"))
    m = _layer()
    qkv = torch.zeros(2, 24, 512).as_subclass(OnDevice)
    assert m._prep_by_kernel(qkv, True) and m._prep_by_kernel(qkv, False)
    CHANGES[change](m)
    assert not m._prep_by_kernel(qkv, True) and not m._prep_by_kernel(qkv, False)
    with pytest.raises(RuntimeError):
        ops.qkv_prep_f32(qkv, m.rotary_emb.freqs, m.k_intrablock_positions, m.v_intrablock_positions, 4, 2, 64, 16, 8)
