"""The workloads whose time counts: what a user of this package has it do, through its public entry points, over the range
of sizes, types and options they are used with.

  layer    one `SparseAttention` layer: the parallel forward (prefill) or a training step (forward + backward)
  attend   the operator `native_sparse_attend`, forward + backward
  model    a training step of the small byte-level `Transformer`
  session  a layer decoding token by token from captured graphs over a long context (`DecodeSession`)
  chat     the `Transformer` decoding token by token through the caches its forward hands back

`listed()` are the workloads by name, `draw(rng)` gives others of the same ranges; `prepare` makes what a program holds
before the call, `run` is one pass, `work` the operations and bytes a pass cannot do without, `tolerance` how far another
correct implementation of the same precision may be off.
"""
import math

import torch

from native_sparse_attention_pytorch_amd import SparseAttention
from native_sparse_attention_pytorch_amd.decode_session import DecodeSession
from native_sparse_attention_pytorch_amd.ops import native_sparse_attend
from native_sparse_attention_pytorch_amd.transformer import Transformer

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}

# widths of the layers: input features, query heads, key / value heads, features per head
SMALL = dict(dim=512, heads=8, kv_heads=8, dim_head=64)           # heads not grouped (the module's default)
BYTES = dict(dim=512, heads=8, kv_heads=4, dim_head=64)           # the byte-level model
MEDIUM = dict(dim=1024, heads=16, kv_heads=4, dim_head=64)
LARGE = dict(dim=4096, heads=32, kv_heads=8, dim_head=128)        # a long-context model
# sparsity: sliding window, compression block and stride, selection block, selected blocks
README = dict(window=2, cbs=4, stride=2, block=4, sel=2)
FINE = dict(window=64, cbs=16, stride=8, block=16, sel=4)
COARSE = dict(window=512, cbs=32, stride=16, block=64, sel=16)

SESSION_STEPS = 16      # tokens of one pass of a session: one compression window is completed among them
SESSION_ROOM = 8192     # tokens that a session can decode beyond the context it starts with
CHAT_STEPS = 8


def layer(name, width, sparse, dtype, batch, seq, step, causal=True, diff_topk=False, share=True):
    return dict(name=name, kind="layer", dtype=dtype, batch=batch, seq=seq, step=step, causal=causal, diff_topk=diff_topk, share=share,
                **width, **sparse)


def listed():
    return [
        # the smallest call: the usage example of the package (fp32, not causal, 31 tokens); launches and latency are all of it
        layer("readme_forward", SMALL, README, "fp32", 2, 31, "forward", causal=False),
        # a layer left in the default type, evaluated on two prompts of an odd length that keep their caches
        layer("layer_prefill_fp32", MEDIUM, COARSE, "fp32", 2, 2053, "prefill"),
        # a layer of the byte-level model trained in the default type
        layer("layer_train_fp32", BYTES, FINE, "fp32", 8, 1024, "train"),
        # an ordinary training step of a medium layer in bf16
        layer("layer_train_4k", MEDIUM, COARSE, "bf16", 4, 4096, "train"),
        # long-context training: one sequence of 32k tokens through a large layer
        layer("layer_train_32k", LARGE, COARSE, "bf16", 1, 32768, "train"),
        # prefill of a long prompt of no round length, caches kept for the decoding that follows
        layer("layer_prefill_30k", LARGE, COARSE, "bf16", 1, 30011, "prefill"),
        # the selection operator alone, as a program with its own block selection calls it: an ordinary and a long sequence
        dict(name="attend_train_8k", kind="attend", dtype="bf16", batch=1, seq=8192, heads=16, kv_heads=4, dim_head=64, block=64, sel=15,
             gates=False),
        dict(name="attend_train_32k", kind="attend", dtype="bf16", batch=1, seq=32768, heads=32, kv_heads=8, dim_head=128, block=64, sel=15,
             gates=False),
        # training of the byte-level model with differentiable top-k: many small layers, bound by their number
        dict(name="model_train_1k", kind="model", batch=8, seq=1024, depth=6, diff_topk=True, **BYTES, **FINE),
        # serving: one user, and a full batch, decoding with 32k tokens of context
        dict(name="session_b1_32k", kind="session", batch=1, context=32768, **LARGE, **COARSE),
        dict(name="session_b32_32k", kind="session", batch=32, context=32768, **LARGE, **COARSE),
        # the model's cached decoding as its forward offers it, launch by launch, after a short prompt
        dict(name="chat_b8", kind="chat", batch=8, context=333, depth=6, **BYTES, **FINE),
    ]


def draw(rng):
    def spread(lo, hi):                      # whole numbers, even over their logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("layer", "layer", "layer", "attend", "attend", "model", "session", "chat"))
    if kind == "layer":
        dtype = rng.choice(("bf16", "bf16", "fp32"))
        width, sparse = rng.choice(((SMALL, README), (BYTES, FINE), (MEDIUM, COARSE), (MEDIUM, COARSE), (LARGE, COARSE)))
        step = rng.choice(("forward", "prefill", "train", "train"))
        most = 8192 if dtype == "fp32" else 32768
        tokens = spread(31, most if width is not LARGE else most // 2)
        batch = min(rng.choice((1, 1, 2, 3, 4, 8)), max(1, tokens // 31))
        causal = step == "prefill" or width is not SMALL or rng.random() < 0.5
        diff = step == "train" and rng.random() < 0.3
        share = width["heads"] == width["kv_heads"] or rng.random() < 0.85
        return {k: v for k, v in layer("", width, sparse, dtype, batch, max(31, tokens // batch), step, causal, diff, share).items() if k != "name"}
    if kind == "attend":
        heads, kv_heads, dim_head = rng.choice(((8, 8, 64), (8, 4, 64), (16, 4, 64), (32, 8, 128), (16, 2, 128)))
        return dict(kind="attend", dtype=rng.choice(("bf16", "bf16", "bf16", "fp32")), batch=rng.choice((1, 1, 2, 3)), seq=spread(200, 10000),
                    heads=heads, kv_heads=kv_heads, dim_head=dim_head, block=rng.choice((16, 32, 64, 64)), sel=rng.choice((4, 8, 15, 15, 16)),
                    gates=rng.random() < 0.25)
    if kind == "model":
        batch = rng.choice((1, 2, 4, 8))
        return dict(kind="model", batch=batch, seq=spread(64, 1024), depth=rng.choice((2, 4, 6)), diff_topk=rng.random() < 0.5, **BYTES, **FINE)
    if kind == "session":
        return dict(kind="session", batch=rng.choice((1, 2, 4, 8, 16, 32)), context=spread(1000, 32768),
                    **rng.choice(({**LARGE, **COARSE}, {**MEDIUM, **COARSE})))
    return dict(kind="chat", batch=rng.choice((1, 2, 4, 8)), context=spread(40, 1000), depth=rng.choice((2, 4, 6)), **BYTES, **FINE)


# ------------------------------------------------------------------------------------------------------------- prepare

def _sparse_kwargs(c):
    return dict(sliding_window_size=c["window"], compress_block_size=c["cbs"], compress_block_sliding_stride=c["stride"],
                selection_block_size=c["block"], num_selected_blocks=c["sel"])


def _trained(module, gen):
    """Parameters that start as zeros (gate weights, positions, memory slots) get values as training gives them."""
    with torch.no_grad():
        for p in module.parameters():
            if p.requires_grad and not p.any():
                p.copy_(torch.randn(p.shape, generator=gen, device=DEVICE) * 0.05)
    return module


def _layer(c, gen, seed, dtype):
    torch.manual_seed(seed)
    with torch.device(DEVICE):
        m = SparseAttention(dim=c["dim"], dim_head=c["dim_head"], heads=c["heads"], kv_heads=c["kv_heads"], causal=c.get("causal", True),
                            use_diff_topk=c.get("diff_topk", False), query_heads_share_selected_kv=c.get("share", True), **_sparse_kwargs(c))
    return _trained(m, gen).to(dtype)


def _model(c, gen, seed):
    torch.manual_seed(seed)
    with torch.device(DEVICE):
        m = Transformer(num_tokens=256, dim=c["dim"], depth=c["depth"], dim_head=c["dim_head"], heads=c["heads"], kv_heads=c["kv_heads"],
                        sparse_attn_kwargs=dict(use_diff_topk=c.get("diff_topk", False), **_sparse_kwargs(c)))
    return _trained(m, gen).bfloat16()


def _selection(c, gen):
    """Distinct blocks before the query's own block, evenly drawn; queries with too few of them have dead slots."""
    b, h, n, B, S = c["batch"], c["kv_heads"], c["seq"], c["block"], c["sel"]
    W = math.ceil(n / B)
    scores = torch.rand((b, h, n, W), generator=gen, device=DEVICE)
    own = (torch.arange(n, device=DEVICE) // B)[:, None]
    scores.masked_fill_(torch.arange(W, device=DEVICE)[None, :] >= own, -1.0)
    k = min(S, W)
    val, idx = scores.topk(k, dim=-1)
    live = val >= 0
    if k < S:
        idx, live = torch.nn.functional.pad(idx, (0, S - k)), torch.nn.functional.pad(live, (0, S - k))
    return idx.masked_fill(~live, 0).contiguous(), live.contiguous()


def prepare(case, seed):
    c = case
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    randn = lambda *shape: torch.randn(shape, generator=gen, device=DEVICE)
    ids = lambda *shape: torch.randint(0, 256, shape, generator=gen, device=DEVICE)
    if c["kind"] == "layer":
        dtype = DTYPES[c["dtype"]]
        m = _layer(c, gen, seed, dtype)
        x = randn(c["batch"], c["seq"], c["dim"]).to(dtype)
        s = dict(case=c, layer=m, x=x)
        if c["step"] == "train":
            x.requires_grad_()
            s["params"] = [p for p in m.parameters() if p.requires_grad]
            s["dout"] = randn(c["batch"], c["seq"], c["dim"]).to(dtype)
        return s
    if c["kind"] == "attend":
        dtype, d = DTYPES[c["dtype"]], c["dim_head"]
        make = lambda h: randn(c["batch"], h, c["seq"], d).mul_(d ** -0.5).to(dtype)
        q, dout = make(c["heads"]), make(c["heads"])
        k, v = make(c["kv_heads"]), make(c["kv_heads"])
        idx, live = _selection(c, gen)
        gates = torch.ones(idx.shape, device=DEVICE, requires_grad=True) if c["gates"] else None
        return dict(case=c, q=q.requires_grad_(), k=k.requires_grad_(), v=v.requires_grad_(), dout=dout, idx=idx, live=live, gates=gates)
    if c["kind"] == "model":
        m = _model(c, gen, seed)
        return dict(case=c, model=m, params=[p for p in m.parameters() if p.requires_grad], ids=ids(c["batch"], c["seq"] + 1))
    if c["kind"] == "session":
        m = _layer(c, gen, seed, torch.bfloat16)
        b, hk, d, t = c["batch"], c["kv_heads"], c["dim_head"], c["context"]
        rows = lambda n: torch.randn((b, hk, n, d), generator=gen, device=DEVICE, dtype=torch.bfloat16)
        windows = t // c["stride"]
        open_rows = t - windows * c["stride"] + c["cbs"] - c["stride"]      # rows of the compression window that is not complete
        cache = ((rows(t), rows(t)), ((rows(windows), rows(windows)), (rows(open_rows), rows(open_rows))))
        return dict(case=c, layer=m, cache=cache, session=DecodeSession(m, cache, max_len=t + SESSION_ROOM),
                    x=randn(SESSION_STEPS, b, 1, c["dim"]).bfloat16())
    m = _model(c, gen, seed)
    with torch.no_grad():
        _, cache = m(ids(c["batch"], c["context"]), return_cache=True)
    return dict(case=c, model=m, cache=cache, ids=ids(c["batch"], CHAT_STEPS))


# ----------------------------------------------------------------------------------------------------------------- run

def _flat(params):
    """All parameter gradients as one vector, as a data-parallel reducer or a flat optimizer takes them."""
    return torch.cat([p.grad.reshape(-1) for p in params if p.grad is not None])


def run(state):
    s = state
    c = s["case"]
    if c["kind"] == "layer":
        if c["step"] == "train":
            s["layer"].zero_grad(set_to_none=True)
            s["x"].grad = None
            out = s["layer"](s["x"])
            out.backward(s["dout"])
            return out.detach(), s["x"].grad, _flat(s["params"])
        with torch.no_grad():
            return s["layer"](s["x"], return_cache=c["step"] == "prefill")
    if c["kind"] == "attend":
        leaves = [t for t in (s["q"], s["k"], s["v"], s["gates"]) if t is not None]
        for t in leaves:
            t.grad = None
        out = native_sparse_attend(s["q"], s["k"], s["v"], c["block"], s["idx"], s["live"], sel_scale=s["gates"])
        out.backward(s["dout"])
        return [out.detach()] + [t.grad for t in leaves]
    if c["kind"] == "model":
        s["model"].zero_grad(set_to_none=True)
        loss = s["model"](s["ids"], return_loss=True)
        loss.backward()
        return loss.detach(), _flat(s["params"])
    if c["kind"] == "session":
        if s["session"].pos + SESSION_STEPS > s["session"].max_len:      # the conversation is full: the next one begins
            s["session"] = DecodeSession(s["layer"], s["cache"], max_len=c["context"] + SESSION_ROOM)
        return torch.cat([s["session"].step(x) for x in s["x"]], dim=1)
    with torch.no_grad():
        cache, logits = s["cache"], []
        for i in range(CHAT_STEPS):
            out, cache = s["model"](s["ids"][:, i:i + 1], cache=cache, return_cache=True)
            logits.append(out)
        return torch.cat(logits, dim=1), cache


# ---------------------------------------------------------------------------------------------------------------- work

def _pairs(c, n):
    """Attended (query, key) pairs of one head over a sequence of n tokens: compressed, selected, sliding."""
    windows, W, B = n // c["stride"], math.ceil(n / c["block"]), c["block"]
    if c.get("causal", True):
        compressed = n + c["stride"] * windows * (windows - 1) // 2 + (n - windows * c["stride"]) * windows      # + a memory slot
        per_block = [min(B, n - w * B) * (min(w, c["sel"]) * B) for w in range(W)]
        selected = sum(per_block) + sum(s * (s + 1) // 2 for s in (min(B, n - w * B) for w in range(W)))
        band = min(c["window"] + 1, n)
        sliding = band * (band + 1) // 2 + (n - band) * band
    else:
        compressed = n * (windows + 1)
        selected = n * min(n, c["sel"] * B)
        sliding = n * min(n, 2 * c["window"] + 1)
    return compressed, selected, sliding


def _layer_work(c, tokens, seqs, train):
    """(flops, parameters) of a layer over `seqs` sequences of `tokens` tokens."""
    n, d, h, hk, dim = tokens, c["dim_head"], c["heads"], c["kv_heads"], c["dim"]
    wide = c["cbs"] * d
    project = dim * (h + 2 * hk) * d + h * d * dim + dim * 3 * h
    compress = 2 * (wide * wide + wide * d)
    gemm = 2 * seqs * (n * project + hk * (n // c["stride"]) * compress)
    attend = 4 * d * seqs * h * sum(_pairs(c, n))
    return (3 * gemm + 3.5 * attend) if train else gemm + attend, project + compress


def work(case):
    c = case
    if c["kind"] == "layer":
        size, train = (4 if c["dtype"] == "fp32" else 2), c["step"] == "train"
        flops, params = _layer_work(c, c["seq"], c["batch"], train)
        rows = c["batch"] * c["seq"] * c["dim"] * size
        kept = c["batch"] * c["kv_heads"] * c["dim_head"] * 2 * (c["seq"] + c["seq"] // c["stride"]) * size if c["step"] == "prefill" else 0
        return dict(flops=flops, bytes=(2 if train else 1) * (2 * rows + params * size) + kept)
    if c["kind"] == "attend":
        b, n, h, hk, d = c["batch"], c["seq"], c["heads"], c["kv_heads"], c["dim_head"]
        W = math.ceil(n / c["block"])
        sizes = [min(c["block"], n - w * c["block"]) for w in range(W)]
        pairs = b * h * sum(s * min(w, c["sel"]) * c["block"] + s * (s + 1) // 2 for w, s in enumerate(sizes))
        size = 4 if c["dtype"] == "fp32" else 2
        slots = b * hk * n * c["sel"]
        return dict(flops=14 * d * pairs, bytes=size * b * n * d * (4 * h + 4 * hk) + slots * (9 + (8 if c["gates"] else 0)))
    if c["kind"] == "model":
        flops, params = _layer_work(c, c["seq"], c["batch"], True)
        ff = 8 * c["dim"] ** 2
        tokens = c["batch"] * c["seq"]
        return dict(flops=c["depth"] * (flops + 6 * tokens * ff) + 6 * tokens * 256 * c["dim"],
                    bytes=2 * 2 * (c["depth"] * (params + ff) + 2 * 256 * c["dim"]) + tokens * 8)
    b, d, h, hk, t = c["batch"], c["dim_head"], c["heads"], c["kv_heads"], c["context"]
    project = c["dim"] * (h + 2 * hk) * d + h * d * c["dim"] + c["dim"] * 3 * h
    keys = t // c["stride"] + min(t, (c["sel"] + 1) * c["block"]) + min(t, c["window"] + 1)
    attend_bytes, attend_flops = b * hk * keys * d * 2 * 2, 4 * b * h * keys * d
    if c["kind"] == "session":
        wide = c["cbs"] * d
        compress = 2 * (wide * wide + wide * d)                                # once in `stride` tokens
        runs = SESSION_STEPS // c["stride"]
        return dict(flops=SESSION_STEPS * (2 * b * project + attend_flops) + runs * 2 * b * hk * compress,
                    bytes=SESSION_STEPS * (2 * project + attend_bytes) + runs * 2 * compress)
    per_token = c["depth"] * (project + 8 * c["dim"] ** 2) + 256 * c["dim"]
    return dict(flops=CHAT_STEPS * (2 * b * per_token + c["depth"] * attend_flops), bytes=CHAT_STEPS * (2 * per_token + c["depth"] * attend_bytes))


# ----------------------------------------------------------------------------------------------------------- tolerance

def tolerance(case):
    c = case
    if c.get("dtype") == "fp32" and c.get("step") in ("forward", "prefill"):
        # the attention in fp32 against float64: 3.4e-7 (the largest element 3.8e-6); a layer puts its projections around that
        return {"rel": 1e-5, "max": 1e-3}
    if c["kind"] == "attend":
        # bf16 operands and results against float64: 2.4e-3 to 2.7e-3, the largest element 0.08
        return {"rel": 1e-2, "max": 0.3}
    # bf16 layers against themselves through other kernels (projections, norm, windows and selection one by one instead of
    # fused): 1.1e-3 to 4.4e-3, the largest element 0.2 - where two blocks score alike another one may be selected
    return {"rel": 1.5e-2, "max": 0.8}
