"""How the backward of interval-masked attention cuts a key tile's queries into chunks, as its workspace size shows it (host arithmetic, no
compute): by the dK / dV walk that the call takes, which its strides and scale have a say in."""
import ctypes

import pytest


def chunks(mode, hk, g, n, ws, scale=128 ** -0.5, q_token=None, k_token=128):
    """Chunks of a tile of 64 keys."""
    from native_sparse_attention_pytorch_amd import _lib
    d = _lib.DenseDesc()
    mem = mode
    d.batch, d.kv_heads, d.group, d.seq, d.num_mem, d.dim_head, d.mode, d.causal = 1, hk, g, n, mem, 128, mode, 1
    d.num_keys, d.window, d.stride, d.sel_block, d.share, d.scale = (n, ws, 1, 1, 1, scale) if mode == 0 else (n // ws, 0, ws, 1, 1, scale)
    rows = d.num_keys + mem
    d.q_stride[:] = d.do_stride[:] = d.o_stride[:] = [hk * g * n * 128, n * 128, 128]
    if q_token:
        d.q_stride[:] = [n * q_token, 128, q_token]
    d.k_stride[:] = d.v_stride[:] = [hk * rows * k_token, rows * k_token, k_token]
    size = ctypes.c_size_t()
    assert _lib.lib().nsa_dense_workspace_bytes(ctypes.byref(d), ctypes.byref(size)) == 0
    up = lambda x: -(-x // 256) * 256
    part = size.value - up(hk * g * n * 8)
    tiles = -(-rows // 64)
    assert part % (hk * tiles * 2 * 64 * 128 * 4) == 0
    return part // (hk * tiles * 2 * 64 * 128 * 4)


@pytest.mark.parametrize("mode,hk,g,n,ws,keys,other", [
    (1, 8, 4, 32768, 16, 16, 32),       # chunks of 2048 queries; 1024 for the other walks
    (1, 8, 4, 8192, 16, 16, 32),        # 512; 256
    (0, 8, 4, 32768, 512, 1, 1),
    (0, 8, 4, 4096, 512, 1, 4),         # 512 work-groups; 2048
])
def test_chunks_are_those_of_the_walk(mode, hk, g, n, ws, keys, other):
    far = (1 << 30) // (n - 1) // 8 * 8 + 64      # a token stride at which the last row is 2 GB from the first
    assert chunks(mode, hk, g, n, ws) == keys
    assert chunks(mode, hk, g, n, ws, scale=-0.1) == other
    assert chunks(mode, hk, g, n, ws, q_token=far) == other
    assert chunks(mode, hk, g, n, ws, k_token=1 << 24) == other
