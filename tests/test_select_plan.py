"""Work-unit tables of the block-selection backward as the workspace sizes show them (host arithmetic, no compute): at 128 features and blocks
of 33 .. 64 keys the walk with gate gradients is another kernel than the one without and has units of its own."""
import ctypes

import pytest


def sizes(b, hk, g, n, S, B, d):
    from native_sparse_attention_pytorch_amd import _lib
    dsc = _lib.SelectDesc()
    dsc.batch, dsc.kv_heads, dsc.group, dsc.seq, dsc.num_sel, dsc.block, dsc.dim_head, dsc.causal = b, hk, g, n, S, B, d, 1
    dsc.scale = d ** -0.5
    for name, h in (("q_stride", hk * g), ("k_stride", hk), ("v_stride", hk), ("o_stride", hk * g)):
        getattr(dsc, name)[:] = [h * n * d, n * d, d]
    sz = [ctypes.c_size_t() for _ in range(3)]
    assert _lib.lib().nsa_select_workspace_bytes(ctypes.byref(dsc), *[ctypes.byref(s) for s in sz]) == 0
    return [s.value for s in sz]


# batch, kv heads, group, tokens, slots; pairs in a unit of the walk with gate gradients
@pytest.mark.parametrize("b,hk,g,n,S,per", [
    (1, 2, 8, 300, 15, 64),
    (1, 8, 4, 400, 16, 64),           # 7 blocks: ten of 16 slots are dead
    (1, 2, 8, 2000, 15, 256),
    (1, 2, 8, 4096, 15, 256),         # (512 for the walk without: 256 units)
    (1, 8, 4, 1024, 16, 256),
    (1, 8, 4, 2048, 16, 256),
    (1, 8, 4, 4096, 16, 512),
    (1, 8, 4, 16384, 16, 1024),       # (2048)
    (1, 8, 4, 32768, 16, 2048),
])
def test_partials_of_both_walks_fit(b, hk, g, n, S, per):
    B, d = 64, 128
    up = lambda x: -(-x // 256) * 256
    rows = b * hk * g * n
    units = -(-n // B) + -(-n * (S + 1) // per)      # of a kv head: every block may end in a short one
    want = up(rows * 8) + up((rows * (S + 1) + g) * d * 2) + up(b * hk * units * 2 * 64 * d * 4) + up(4)
    assert sizes(b, hk, g, n, S, B, d)[2] == want
