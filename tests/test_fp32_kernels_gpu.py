"""The fp32 forward kernels at the edges of their tiles, against float64: the kernel for many queries (32 rows x 32 keys) and the
kernel for one query per wave or per work-group (64 gathered keys), groups of every size, head dimensions that are no multiple of
a tile, key counts one off a tile, more slots than a wave has lanes, padding keys, decode offsets.

Bound: 1e-5 + 1e-5 |value|, the reference's own fp32 tolerance (tests/test_sparse_attn.py:86).  A logit is a sum of d <= 128
products, an output a weighted mean: their fp32 errors are below (d + 2) 2^-24 |q||k| / sqrt(d) ~ 1e-5 for unit normal inputs at
the very worst and ~1e-6 in practice."""
import math

import pytest
import torch

from oracle import nsa_oracle as O
from tests.util import assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("b,hq,hk,n,d,mode,causal,win,st,mem,qoff", [
    (1, 8, 1, 33, 64, 0, True, 31, 1, 0, 0),          # few queries: a work-group per query, window + 1 = half a tile
    (1, 5, 1, 1, 20, 0, True, 512, 1, 0, 700),        # a decode step: one query, 513 keys = 8 tiles + 1
    (2, 6, 2, 3, 128, 1, True, 0, 4, 64, 600),        # 64 memory slots: the first tile holds nothing else
    (2, 3, 3, 700, 64, 0, True, 63, 1, 0, 0),         # 4200 (query, kv head) pairs: the tile kernel, groups of 1
    (1, 20, 4, 1100, 100, 0, False, 40, 1, 0, 0),     # groups of 5: rows of a wave end inside a query
    (3, 16, 8, 181, 128, 1, True, 0, 16, 1, 0),       # 4344 pairs, strided prefixes that begin empty, d = 128
    (1, 8, 8, 513, 36, 1, False, 0, 5, 31, 0),        # 32-key tiles that end on a memory slot + 102 keys
])
def test_interval_masks(b, hq, hk, n, d, mode, causal, win, st, mem, qoff):
    from native_sparse_attention_pytorch_amd.ops import dense_attend_f32
    total = n + qoff
    keys = total if mode == 0 else total // st
    q, k, v = _rand((b, hq, n, d), n), _rand((b, hk, mem + keys, d), d), _rand((b, hk, mem + keys, d), 7)
    i, j = torch.arange(n)[:, None] + qoff, torch.arange(keys)[None, :]
    if mode == 0:
        see = (j <= i) & (i - j <= win) if causal else (i - j).abs() <= win
    else:
        see = torch.cat((torch.ones(n, mem, dtype=torch.bool), (j + 1) * st <= i if causal else torch.ones(n, keys, dtype=torch.bool)), dim=1)
    g = hq // hk
    kd, vd = k.double().repeat_interleave(g, 1), v.double().repeat_interleave(g, 1)
    sim = (q.double() @ kd.transpose(-1, -2) * d ** -0.5).masked_fill(~see, float("-inf"))
    got, lse = dense_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), mode, causal, win, st, mem, q_offset=qoff)
    torch.cuda.synchronize()
    assert_close(got, sim.softmax(-1) @ vd, 1e-5, 1e-5, "out")
    assert_close(lse, sim.logsumexp(-1), 1e-5, 1e-5, "lse")


@pytest.mark.parametrize("b,hq,hk,n,d,B,S,causal,qoff", [
    (1, 4, 1, 65, 64, 1, 3, True, 0),                 # blocks of one key
    (1, 7, 1, 64, 60, 5, 70, True, 0),                # more slots than lanes, blocks that straddle tiles, groups of 7
    (2, 2, 2, 1100, 128, 64, 2, True, 0),             # 4400 queries: a query per wave, groups of 1
    (1, 12, 4, 530, 64, 48, 4, False, 0),             # padding keys: the last block has 2 rows; groups of 3
    (1, 4, 2, 2, 128, 100, 3, True, 998),             # decode steps, blocks above a tile
    (1, 4, 2, 40, 64, 16, 0, True, 0),                # no slots: the own block only
])
def test_selection(b, hq, hk, n, d, B, S, causal, qoff):
    from native_sparse_attention_pytorch_amd.ops import native_sparse_attend_f32
    total = n + qoff
    q, k, v = _rand((b, hq, n, d), n), _rand((b, hk, total, d), d), _rand((b, hk, total, d), 7)
    g = torch.Generator().manual_seed(B)
    W = math.ceil(total / B)
    idx = torch.randint(0, W, (b, hk, n, S), generator=g)
    msk = torch.rand(b, hk, n, S, generator=g) > 0.3
    if S and not causal:
        msk[..., 0] = True                            # (a query with no live slot at all has its own test)
        idx[..., 0] = W - 1                           # the block that reaches past the end
    want, want_lse = O.select_attend(q.double(), k.double(), v.double(), idx, msk, B, causal=causal, return_lse=True, q_offset=qoff)
    got, lse = native_sparse_attend_f32(q.to(DEV), k.to(DEV), v.to(DEV), B, idx.to(DEV), msk.to(DEV), include_block_causal=causal, return_lse=True,
                                        q_offset=qoff)
    torch.cuda.synchronize()
    assert_close(got, want, 1e-5, 1e-5, "out")
    assert_close(lse, want_lse, 1e-5, 1e-5, "lse")
