#!/usr/bin/env python3
"""Headline benchmark: block-selection attention forward+backward at sequence 32k in bf16
(batch 1, 32 query heads, 8 kv heads, dim_head 128,
selection_block_size 64, 16 blocks per query = 15 selected + the query's own block).

One "step" = inverse-index build + forward + backward through the C ABI of libnsa_hip.so with
all inputs resident in HBM.  Prints ONE JSON line (see the keys below).  `value` is the
algorithmic TFLOP/s of the whole step: 14*d*P FLOP, P = attended (query, key) pairs summed over
query heads, causal-discounted own block.  Kernel durations come from HIP events recorded on the
launch stream between the kernels (nsa_select_*_timed).
"""
from __future__ import annotations

import argparse
import ctypes as C
import json
import math
import os
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

MFMA_PEAK_TFLOPS = 2500.0      # MI355X dense bf16

CFG = dict(batch=1, seq=32768, heads=32, kv_heads=8, dim_head=128, block=64, num_sel=15)

# Bytes per launch on this workload between L2 and the memory side (HBM and the 256 MB cache in front of it: rows which that serves are in
# them) come from the tracked rocprofv3 summary (FETCH_SIZE / WRITE_SIZE per dispatch, scaled by streaming kernels of known size; the file
# states the commands), not from literals kept here
TRAFFIC_SUMMARY = os.path.join(ROOT, "profiles", "select_fwd_bwd_seq32k_hbm_traffic.txt")
TRAFFIC_KERNELS = {"sel_fwd_rows_kernel": "fwd_block_walk", "sel_fwd_combine_kernel": "fwd_merge", "sel_bwd_dq_combine_kernel": "bwd_dq_merge",
                   "sel_bwd_block_kernel": "bwd_dkv_walk", "sel_bwd_dkv_reduce_kernel": "bwd_dkv_reduce", "sel_delta_kernel": "bwd_delta"}


def measured_traffic_bytes():
    """{bench kernel name: bytes per launch behind L2} from the summary's table (columns: kernel, raw counters, fetch_GB, write_GB,
    total_GB); empty when the file is missing."""
    out = {}
    try:
        for line in open(TRAFFIC_SUMMARY):
            f = line.split()
            if len(f) == 6 and f[0] in TRAFFIC_KERNELS:
                out[TRAFFIC_KERNELS[f[0]]] = float(f[5]) * 1e9
    except OSError:
        pass
    return out


def selection(b, h, n, B, S, seed, device):
    """15 distinct causal blocks per query, uniform over the blocks before the query's own
    block (random-score top-k), fixed seed; dead slots for early queries."""
    g = torch.Generator(device=device).manual_seed(seed)
    W = math.ceil(n / B)
    scores = torch.rand(b, h, n, W, generator=g, device=device)
    blk = (torch.arange(n, device=device) // B)[None, None, :, None]
    scores = scores.masked_fill(torch.arange(W, device=device)[None, None, None, :] >= blk, -1.0)
    vals, idx = scores.topk(min(S, W), dim=-1)
    mask = vals >= 0
    return idx.masked_fill(~mask, 0).contiguous(), mask.contiguous()


def exchange_bytes(cfg):
    """Bytes per step that must cross HBM in a block-major walk: per live (query, kv head, slot) pair one G*d bf16 partial written and read
    again in each direction - what is written between is far larger than any cache - and every tensor once.  (The three gathered rows a
    pair, Q in the forward, Q and dO in the backward, come from a set that the memory-side cache holds.)"""
    b, n, hq, hk, d, B, S = cfg["batch"], cfg["seq"], cfg["heads"], cfg["kv_heads"], cfg["dim_head"], cfg["block"], cfg["num_sel"]
    W = math.ceil(n / B)
    pairs = b * hk * sum(B * (min(w, S) + 1) for w in range(W))
    row = (hq // hk) * d * 2
    once = (4 * b * hq * n * d + 6 * b * hk * n * d) * 2            # q, out, dO, dq; k, v, dk, dv (k, v read twice)
    return pairs * row * 4 + once


def attended_pairs(b, hq, n, B, s_total):
    W = math.ceil(n / B)
    return b * hq * sum(B * (min(w, s_total - 1) * B + (B + 1) / 2) for w in range(W))


class HipEvents:
    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so")
        self.hip.hipEventCreate.argtypes = [C.POINTER(C.c_void_p)]
        self.hip.hipEventElapsedTime.argtypes = [C.POINTER(C.c_float), C.c_void_p, C.c_void_p]
        self.hip.hipEventRecord.argtypes = [C.c_void_p, C.c_void_p]

    def make(self, n):
        arr = (C.c_void_p * n)()
        for i in range(n):
            e = C.c_void_p()
            assert self.hip.hipEventCreate(C.byref(e)) == 0
            arr[i] = e
        return arr

    def record(self, ev, stream):
        assert self.hip.hipEventRecord(ev, stream) == 0

    def ms(self, a, b):
        out = C.c_float()
        rc = self.hip.hipEventElapsedTime(C.byref(out), a, b)
        assert rc == 0, rc
        return out.value


def cpu_baseline(cfg, q, k, v, do, idx, msk, nq=8192, dtype=torch.float32):
    """The CPU oracle (restatement of the reference's pure-torch path, in `dtype`) on a bounded sample:
    the last `nq` queries of the same workload against the full-length K/V, forward+backward."""
    from oracle import nsa_oracle as O
    n = cfg["seq"]
    sl = slice(n - nq, n)
    qc = q[:, :, sl].to(dtype).cpu().requires_grad_()
    kc, vc = k.to(dtype).cpu().requires_grad_(), v.to(dtype).cpu().requires_grad_()
    doc = do[:, :, sl].to(dtype).cpu()
    ic, mc = idx[:, :, sl].cpu(), msk[:, :, sl].cpu()
    t0 = time.perf_counter()
    out = O.select_attend(qc, kc, vc, ic, mc, cfg["block"], causal=True, q_offset=n - nq, chunk=128)
    (out * doc).sum().backward()
    dt = time.perf_counter() - t0
    return dict(value=nq * cfg["batch"] / dt, unit="tokens/s", cores=torch.get_num_threads(), kind="port",
                sample=f"last {nq} of {n} queries (each attends 16 blocks), full-length K/V, {str(dtype).split('.')[-1]} fwd+bwd, {dt:.1f} s; "
                       f"host has {os.cpu_count()} logical CPUs"), out.detach()


class _Skip(Exception):
    """Raised inside an optional leg that --headline-only turns off."""


def graphed_train_leg():
    """BASELINE configs[4] training step with forward + backward replayed from one HIP graph (training.GraphedStep) on a bf16
    model, Adam on fp32 master weights outside the graph.  Runs in a process of its own (see main): prints one JSON object."""
    import torch
    from native_sparse_attention_pytorch_amd.transformer import Transformer
    from native_sparse_attention_pytorch_amd.training import Fp32Masters, GraphedStep
    dev = "cuda"
    torch.manual_seed(0)
    model = Transformer(num_tokens=256, dim=512, depth=6, dim_head=64, heads=8, kv_heads=4,
                        sparse_attn_kwargs=dict(sliding_window_size=64, compress_block_size=16, compress_block_sliding_stride=8,
                                                selection_block_size=16, num_selected_blocks=4)).to(dev)
    ids = torch.randint(0, 256, (8, 1025), device=dev)
    mw = Fp32Masters(model)
    opt = torch.optim.Adam(mw.masters, lr=1e-4, fused=True)       # (one kernel per parameter list instead of one per operation)
    gstep = GraphedStep(model, ids)

    def step():
        loss = gstep(ids)
        mw.step(opt)
        return loss
    for _ in range(3):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(10):
        last = step()
    torch.cuda.synchronize()
    tt = (time.perf_counter() - t0) / 10
    print(json.dumps(dict(ms_per_step=round(tt * 1e3, 3), tokens_per_s=round(8 * 1024 / tt, 1), loss_after=round(last.item(), 4))), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--headline-only", action="store_true", help="only the headline workload (for profiler runs): no compressed-branch, module or decode legs")
    ap.add_argument("--skip", default="", help="comma-separated legs to leave out: select_config2, rowtraffic, compressed, module, decode, train, generate")
    ap.add_argument("--child-leg", default="", help=argparse.SUPPRESS)
    args = ap.parse_args()
    if args.child_leg == "graphtrain":
        graphed_train_leg()
        return
    skip = set(filter(None, args.skip.split(","))) | ({"select_config2", "rowtraffic", "compressed", "module", "decode", "train", "generate"} if args.headline_only else set())

    def leg(name):
        """Announce a leg on stderr (a long profiler run must not look hung) or skip it."""
        if name in skip:
            raise _Skip()
        print(f"bench.py: {name} leg", file=sys.stderr, flush=True)

    if args.gpus != 1:
        print("bench.py: this build runs on ONE GPU only (no sharding, no collectives); use --gpus 1", file=sys.stderr)
        sys.exit(2)
    # The graph-replayed training step runs first, in a child process started before this process touches the GPU: a
    # recording that goes wrong ends its process, and that must not take the headline with it.  Not under a profiler
    # (its preloaded library has the GPU initialised already, and a process in that state must not start another program).
    graphed_train = None
    profiled = any(k.startswith(("ROCPROF", "ROCP_")) for k in os.environ) or "rocprof" in os.environ.get("LD_PRELOAD", "")
    if "train" not in skip and not profiled:
        print("bench.py: graph-replayed train leg (child process)", file=sys.stderr, flush=True)
        try:
            import subprocess
            cp = subprocess.run([sys.executable, os.path.abspath(__file__), "--child-leg", "graphtrain"], capture_output=True, text=True, timeout=600)
            lines = [ln for ln in cp.stdout.strip().splitlines() if ln.startswith("{")]
            graphed_train = json.loads(lines[-1]) if cp.returncode == 0 and lines else dict(error=f"child exited with {cp.returncode}")
        except Exception as ex:
            graphed_train = dict(error=repr(ex))
    if not torch.cuda.is_available():
        print("bench.py needs an MI355X (no CPU fallback for the product path)", file=sys.stderr)
        sys.exit(2)

    from native_sparse_attention_pytorch_amd import _lib, ops
    L = _lib.lib()
    dev = "cuda"
    stream = torch.cuda.current_stream().cuda_stream
    hev = HipEvents()
    P = lambda t: t.data_ptr()

    def run_select(cfg, steps, warmup, seed=0):
        """`steps` timed steps (index build + forward + backward of block-selection attention through the C ABI) on the workload
        `cfg`; returns (ms per step, per-step event arrays, tensors)."""
        b, n, hq, hk, d, B, S = cfg["batch"], cfg["seq"], cfg["heads"], cfg["kv_heads"], cfg["dim_head"], cfg["block"], cfg["num_sel"]
        g = torch.Generator(device=dev).manual_seed(seed)
        mk = lambda h: (torch.randn(b, h, n, d, generator=g, device=dev) * d ** -0.5).to(torch.bfloat16)
        q, k, v, do = mk(hq), mk(hk), mk(hk), mk(hq)
        idx, msk = selection(b, hk, n, B, S, seed, dev)
        fm = msk.view(torch.uint8)
        out = torch.empty_like(q)
        lse = torch.empty(b, hq, n, dtype=torch.float32, device=dev)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        dsc = ops._select_desc(q, k, v, out, S, B, True, d ** -0.5, True)
        ib, fb, wb = ops._ws_sizes(dsc)
        iws = torch.empty(ib, dtype=torch.uint8, device=dev)
        # forward and backward workspaces are never live together: share one allocation
        ws = torch.empty(max(fb, wb), dtype=torch.uint8, device=dev)

        def step(ev):
            if ev is not None:
                hev.record(ev[0], stream)
            _lib.check(L.nsa_select_build_index(C.byref(dsc), P(idx), P(fm), P(iws), ib, stream), "build_index")
            fe = C.cast(C.byref(ev, 1 * C.sizeof(C.c_void_p)), C.c_void_p) if ev is not None else None
            be = C.cast(C.byref(ev, 4 * C.sizeof(C.c_void_p)), C.c_void_p) if ev is not None else None
            _lib.check(L.nsa_select_fwd_timed(C.byref(dsc), P(q), P(k), P(v), P(idx), P(fm), P(iws), P(ws), fb, P(out), P(lse), stream,
                                              fe, 3 if ev is not None else 0), "fwd")
            _lib.check(L.nsa_select_bwd_timed(C.byref(dsc), P(q), P(k), P(v), P(out), P(do), None, P(lse), P(idx), P(fm), P(iws), P(ws), wb,
                                              P(dq), P(dk), P(dv), None, stream, be, 6 if ev is not None else 0), "bwd")

        for _ in range(warmup):
            step(None)
        torch.cuda.synchronize()
        evs = [hev.make(10) for _ in range(steps)]
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for e in evs:
            step(e)
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / steps * 1e3, evs, (q, k, v, do, idx, msk, out)

    cfg = CFG
    b, n, hq, hk, d, B, S = cfg["batch"], cfg["seq"], cfg["heads"], cfg["kv_heads"], cfg["dim_head"], cfg["block"], cfg["num_sel"]
    ms_step, evs, (q, k, v, do, idx, msk, out) = run_select(cfg, args.steps, args.warmup)

    names = ["index_build", "fwd_block_walk", "fwd_merge", None, "bwd_delta", "bwd_dq_walk", "bwd_dkv_walk", "bwd_dq_merge", "bwd_dkv_reduce"]
    kern = {}
    for i, nm in enumerate(names):
        if nm is not None:
            kern[nm] = sum(hev.ms(e[i], e[i + 1]) for e in evs) / len(evs)

    pairs = attended_pairs(b, hq, n, B, S + 1)
    flop_unit = 2.0 * d * pairs                        # one d-deep contraction over all attended pairs
    total_flop = 7 * flop_unit                         # fwd 4dP + bwd 10dP
    value = total_flop / (ms_step * 1e-3) / 1e12
    # algorithmic work of each MFMA kernel: forward 4dP; the backward walk does all of 10dP (the separate dQ walk only
    # runs when gate gradients are requested, which this benchmark does not)
    kflop = {"fwd_block_walk": 2 * flop_unit, "bwd_dkv_walk": 5 * flop_unit}
    dom = max(kflop, key=lambda nm: kern[nm])
    achieved = kflop[dom] / (kern[dom] * 1e-3) / 1e12
    traffic_all = measured_traffic_bytes()
    traffic = traffic_all.get(dom)
    roofline = dict(bound="mfma", kernel=dom, achieved=round(achieved, 2), peak=MFMA_PEAK_TFLOPS, unit="TFLOP/s",
                    frac=round(achieved / MFMA_PEAK_TFLOPS, 4), traffic=traffic,
                    step_frac=round(value / MFMA_PEAK_TFLOPS, 4),
                    # what this selection law allows at any kernel quality: a pair's partial results cross HBM (4 KB, written and
                    # read, forward and backward together) at the 6 TB/s that plain streams reach
                    ceiling_exchange_only_frac=round(total_flop / (exchange_bytes(cfg) / 6.0e12) / 1e12 / MFMA_PEAK_TFLOPS, 4),
                    # measured bytes behind L2 over measured time, to read beside the rowtraffic leg's rates
                    behind_l2_GBs={nm: round(traffic_all[nm] / (kern[nm] * 1e-3) / 1e9, 1) for nm in traffic_all},
                    behind_l2_GBs_step=round(sum(traffic_all.values()) / (ms_step * 1e-3) / 1e9, 1) if traffic_all else None,
                    traffic_source=os.path.relpath(TRAFFIC_SUMMARY, ROOT))

    res = dict(metric="NSA selection-attention fwd+bwd TFLOP/s at seq 32k (bf16)", value=round(value, 2), unit="TFLOP/s",
               n_gpus=1, steps=args.steps, warmup=args.warmup, ms_per_step=round(ms_step, 4), higher_is_better=True,
               scaling="weak", vs_baseline=None, dtype="bf16", data="synthetic",
               config=dict(workload="BASELINE configs[3]: selection attention fwd+bwd, b1 n32768 Hq32 Hkv8 d128 B64, 15 selected + own block",
                           tokens_per_s=round(b * n / (ms_step * 1e-3), 1), attended_pairs=int(pairs), flop_per_step=total_flop),
               kernels_ms={k_: round(v_, 4) for k_, v_ in kern.items()},
               roofline=roofline)

    # the isolated selection kernels at b1 n8192 Hq16 Hkv4 d64 B64, 15 selected + own block (the d = 64
    # family of the same kernels), timed the same way with its own roofline block
    try:
        leg("select_config2")
        cfg2 = dict(batch=1, seq=8192, heads=16, kv_heads=4, dim_head=64, block=64, num_sel=15)
        ms2, evs2, _t2 = run_select(cfg2, max(args.steps, 20), max(args.warmup, 3), seed=2)
        kern2 = {nm: sum(hev.ms(e[i], e[i + 1]) for e in evs2) / len(evs2) for i, nm in enumerate(names) if nm is not None}
        pairs2 = attended_pairs(1, 16, 8192, 64, 16)
        unit2 = 2.0 * 64 * pairs2
        dom2 = max(("fwd_block_walk", "bwd_dkv_walk"), key=lambda nm: kern2[nm])
        ach2 = (2 if dom2 == "fwd_block_walk" else 5) * unit2 / (kern2[dom2] * 1e-3) / 1e12
        res["select_config2"] = dict(workload="BASELINE configs[1]: selection attention fwd+bwd, b1 n8192 Hq16 Hkv4 d64 B64, 15 selected + own block",
                                     ms_per_step=round(ms2, 4), tflops=round(7 * unit2 / (ms2 * 1e-3) / 1e12, 2),
                                     tokens_per_s=round(8192 / (ms2 * 1e-3), 1), attended_pairs=int(pairs2), flop_per_step=7 * unit2,
                                     kernels_ms={k_: round(v_, 4) for k_, v_ in kern2.items()},
                                     roofline=dict(bound="mfma", kernel=dom2, achieved=round(ach2, 2), peak=MFMA_PEAK_TFLOPS, unit="TFLOP/s",
                                                   frac=round(ach2 / MFMA_PEAK_TFLOPS, 4),
                                                   step_frac=round(7 * unit2 / (ms2 * 1e-3) / 1e12 / MFMA_PEAK_TFLOPS, 4)))
        del _t2
    except _Skip:
        pass
    except Exception as ex:
        res["select_config2"] = dict(error=repr(ex))

    # the other half of BASELINE configs[3]: compressed attention with fused importance logits +
    # top-k over 2048 compressed keys (+1 memory slot), forward and backward, reported beside the headline
    try:
        leg("compressed")
        g2 = torch.Generator(device=dev).manual_seed(1)
        nc = n // 16
        ck = (torch.randn(b, hk, nc + 1, d, generator=g2, device=dev) * d ** -0.5).to(torch.bfloat16).requires_grad_()
        cv = (torch.randn(b, hk, nc + 1, d, generator=g2, device=dev) * d ** -0.5).to(torch.bfloat16).requires_grad_()
        qc = q.clone().requires_grad_()
        # six rounds queued without a host synchronisation in between (HIP events bracket each call; with a
        # synchronisation per round the first call of a round also times the host's allocations), the first two discarded
        evs_c = []
        for it in range(6):
            qc.grad = ck.grad = cv.grad = None      # a step's gradients start from None (no accumulation pass in the timing)
            e0, e1, e2, e3, e4 = (torch.cuda.Event(enable_timing=True) for _ in range(5))
            e0.record()
            # as the module calls it without differentiable top-k: the forward kernel makes the selection, no logits in memory
            c_out, idx_, fm_ = ops.compress_attend_topk(qc, ck, cv, 1, 16, True, B, S + 1)
            e1.record()
            c_out.backward(do)
            e2.record()
            # for comparison, the two-kernel path (logits below each row's causal limit written out, then the top-k kernel)
            with torch.no_grad():
                _, imp, prefix = ops.compress_attend(qc, ck, cv, 1, 16, True, sel_block=B, share=True, prefix_only=True)
                e3.record()
                ops.importance_topk(imp, S + 1, prefix=prefix)
                e4.record()
            evs_c.append((e0, e1, e2, e3, e4))
        torch.cuda.synchronize()
        tms = [tuple(e[i].elapsed_time(e[i + 1]) for i in range(4)) for e in evs_c]
        p_cmp = b * hq * sum(i // 16 + 1 for i in range(n))
        best = min(tms[2:], key=lambda t: t[0] + t[1])
        cf, cb = 4 * d * p_cmp / (best[0] * 1e-3) / 1e12, 10 * d * p_cmp / (best[1] * 1e-3) / 1e12
        res["compressed_branch"] = dict(fwd_with_selection_ms=round(best[0], 4), bwd_ms=round(best[1], 4),
                                        attended_pairs=p_cmp, fwd_bwd_tflops=round(14 * d * p_cmp / ((best[0] + best[1]) * 1e-3) / 1e12, 2),
                                        two_kernel_path=dict(fwd_with_logits_ms=round(best[2], 4), topk_ms=round(best[3], 4)),
                                        # its own roofline: algorithmic 4dP forward (attention + block selection in one kernel) / 10dP
                                        # backward (delta + dQ + dK/dV + reduce kernels together) over the HIP-event time of each call
                                        roofline=dict(bound="mfma", peak=MFMA_PEAK_TFLOPS, unit="TFLOP/s",
                                                      fwd=dict(kernel="dense_fwd_kernel<128,4,true>", achieved=round(cf, 2), frac=round(cf / MFMA_PEAK_TFLOPS, 4)),
                                                      bwd=dict(kernel="dense_bwd_dq_kernel<128> + dense_bwd_dkv_keys_kernel", achieved=round(cb, 2),
                                                               frac=round(cb / MFMA_PEAK_TFLOPS, 4))))
    except _Skip:
        pass
    except Exception as ex:  # the headline must still be printed
        res["compressed_branch"] = dict(error=repr(ex))

    # the callers either side of the path, reported beside the headline: the whole SparseAttention
    # module (b4 n4096 dim1024, forward + backward) and one decode step of a
    # configs[3]-sized layer over a 32k-token cache
    try:
        leg("module")
        from native_sparse_attention_pytorch_amd import SparseAttention
        torch.manual_seed(0)
        mod = SparseAttention(dim=1024, dim_head=64, heads=16, kv_heads=4, sliding_window_size=512, compress_block_size=32,
                              compress_block_sliding_stride=16, selection_block_size=64, num_selected_blocks=16, causal=True).to(dev).bfloat16()
        xm = torch.randn(4, 4096, 1024, device=dev, dtype=torch.bfloat16, requires_grad=True)
        dom = torch.randn_like(xm)
        def mod_step():
            # a training step's forward + backward: gradients start from None, as after optimizer.zero_grad()
            mod.zero_grad(set_to_none=True)
            xm.grad = None
            mod(xm).backward(dom)
        for _ in range(2):
            mod_step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(5):
            mod_step()
        torch.cuda.synchronize()
        tm = (time.perf_counter() - t0) / 5
        res["module_config3"] = dict(ms_per_step=round(tm * 1e3, 3), tokens_per_s=round(4 * 4096 / tm, 1))
        del mod, xm, dom
    except _Skip:
        pass
    except Exception as ex:
        res["module_config3"] = dict(error=repr(ex))
    try:
        leg("decode")
        from native_sparse_attention_pytorch_amd import SparseAttention
        torch.manual_seed(0)
        ctx = 32768
        mod = SparseAttention(dim=hq * d, dim_head=d, heads=hq, kv_heads=hk, sliding_window_size=512, compress_block_size=32,
                              compress_block_sliding_stride=16, selection_block_size=B, num_selected_blocks=S + 1, causal=True).to(dev).bfloat16()
        from native_sparse_attention_pytorch_amd.decode_session import DecodeSession
        dec = {}
        for bd in (1, 32):
            def filled(rows, cap):          # a cache tensor as the module hands it back: prefix of a buffer with spare rows
                buf = torch.randn(bd, hk, cap, d, device=dev, dtype=torch.bfloat16)
                buf._nsa_filled = rows
                return buf[:, :, :rows]
            cache = ((filled(ctx, ctx + 256), filled(ctx, ctx + 256)),
                     ((filled(ctx // 16, ctx // 16 + 64), filled(ctx // 16, ctx // 16 + 64)),
                      (torch.zeros(bd, hk, 16, d, device=dev, dtype=torch.bfloat16), torch.zeros(bd, hk, 16, d, device=dev, dtype=torch.bfloat16))))
            xt = torch.randn(bd, 1, hq * d, device=dev, dtype=torch.bfloat16)
            # the same steps replayed from a captured HIP graph (fixed-capacity caches, lengths read on the device)
            sess = DecodeSession(mod, cache, max_len=ctx + 256)
            for _ in range(40):             # includes the first compression step (one-time library initialisation)
                _, cache = mod(xt, cache=cache, return_cache=True)
                sess.step(xt)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(100):
                _, cache = mod(xt, cache=cache, return_cache=True)
            torch.cuda.synchronize()
            td = (time.perf_counter() - t0) / 100
            t0 = time.perf_counter()
            for _ in range(100):
                sess.step(xt)
            torch.cuda.synchronize()
            tg = (time.perf_counter() - t0) / 100
            dec[f"batch{bd}"] = dict(us_per_step=round(td * 1e6, 1), tokens_per_s=round(bd / td, 1),
                                     graph_us_per_step=round(tg * 1e6, 1), graph_tokens_per_s=round(bd / tg, 1))
            del sess, cache
        res["decode_layer_32k"] = dec
        del mod
    except _Skip:
        pass
    except Exception as ex:
        res["decode_layer_32k"] = dict(error=repr(ex))

    # end-to-end training step of the small NSA transformer on byte tokens
    # (depth 6, dim 512, 8/4 heads, batch 8 x 1024 tokens; fp32 master weights, bf16 autocast, Adam)
    try:
        leg("train")
        from native_sparse_attention_pytorch_amd.transformer import Transformer
        torch.manual_seed(0)
        model = Transformer(num_tokens=256, dim=512, depth=6, dim_head=64, heads=8, kv_heads=4,
                            sparse_attn_kwargs=dict(sliding_window_size=64, compress_block_size=16, compress_block_sliding_stride=8,
                                                    selection_block_size=16, num_selected_blocks=4)).to(dev)
        opt = torch.optim.Adam(model.parameters(), lr=1e-4)
        ids = torch.randint(0, 256, (8, 1025), device=dev)

        def train_step():
            with torch.autocast("cuda", dtype=torch.bfloat16):
                loss = model(ids, return_loss=True)
            loss.backward()
            opt.step()
            opt.zero_grad()
            return loss
        for _ in range(3):
            train_step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(10):
            last = train_step()
        torch.cuda.synchronize()
        tt = (time.perf_counter() - t0) / 10
        res["train_config5"] = dict(ms_per_step=round(tt * 1e3, 3), tokens_per_s=round(8 * 1024 / tt, 1), loss_after=round(last.item(), 4))
        del model, opt
        # the same step with the model in bf16 and the optimizer on fp32 master weights (no per-layer casts: the step is bound by
        # its kernel launches)
        from native_sparse_attention_pytorch_amd.training import Fp32Masters
        torch.manual_seed(0)
        model = Transformer(num_tokens=256, dim=512, depth=6, dim_head=64, heads=8, kv_heads=4,
                            sparse_attn_kwargs=dict(sliding_window_size=64, compress_block_size=16, compress_block_sliding_stride=8,
                                                    selection_block_size=16, num_selected_blocks=4)).to(dev)
        mw = Fp32Masters(model)
        opt = torch.optim.Adam(mw.masters, lr=1e-4, fused=True)       # (one kernel per parameter list instead of one per operation)

        def master_step():
            loss = model(ids, return_loss=True)
            loss.backward()
            mw.step(opt)
            return loss
        for _ in range(3):
            master_step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(10):
            last = master_step()
        torch.cuda.synchronize()
        tt = (time.perf_counter() - t0) / 10
        res["train_config5"]["fp32_masters"] = dict(ms_per_step=round(tt * 1e3, 3), tokens_per_s=round(8 * 1024 / tt, 1), loss_after=round(last.item(), 4))
        if graphed_train is not None:
            res["train_config5"]["graphed_fp32_masters"] = graphed_train
        del model, opt, mw
    except _Skip:
        pass
    except Exception as ex:
        res["train_config5"] = dict(error=repr(ex))

    # generation with the same model in bf16: greedy sampling from a 128-token prompt to 384 tokens, batch 8, through the
    # per-layer caches - launched step by step, and replayed from a captured whole-model HIP graph
    try:
        leg("generate")
        from native_sparse_attention_pytorch_amd.transformer import Transformer
        torch.manual_seed(0)
        model = Transformer(num_tokens=256, dim=512, depth=6, dim_head=64, heads=8, kv_heads=4,
                            sparse_attn_kwargs=dict(sliding_window_size=64, compress_block_size=16, compress_block_sliding_stride=8,
                                                    selection_block_size=16, num_selected_blocks=4)).to(dev).bfloat16()
        prompt = torch.randint(0, 256, (8, 128), device=dev)
        gen = {}
        for name, kw in (("cached", dict(use_cache_kv=True)), ("graph", dict(use_cache_kv=True, use_graph=True))):
            model.sample(prompt, 160, temperature=0., **kw)          # warm-up (and one-time library initialisation)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            new = model.sample(prompt, 384, temperature=0., **kw)
            torch.cuda.synchronize()
            tg = time.perf_counter() - t0
            gen[name] = dict(ms_per_token=round(tg / new.shape[1] * 1e3, 3), tokens_per_s=round(new.numel() / tg, 1))
        res["generate_config5_bf16"] = gen
        del model
    except _Skip:
        pass
    except Exception as ex:
        res["generate_config5_bf16"] = dict(error=repr(ex))

    # what the memory system gives the walks' access pattern (random 1 KB rows, loads of a round in flight together): the
    # rates to read the behind_l2_GBs figures against.  2 GB buffers = HBM; a 2 MB source = rows that stay in L2.
    try:
        leg("rowtraffic")
        big = 2 << 30
        src = torch.zeros(big // 4, dtype=torch.float32, device=dev)
        dst = torch.zeros(big // 4, dtype=torch.float32, device=dev)
        rows_big, waves, iters = big // 1024, 8192, 64
        probe = {}
        for name, sr, rd, wr in (("gather_hbm", rows_big, 2, 0), ("scatter_hbm", rows_big, 0, 2), ("gather1_scatter1_hbm", rows_big, 1, 1),
                                 ("gather2_scatter1_hbm", rows_big, 2, 1), ("gather1_scatter2_hbm", rows_big, 1, 2),
                                 ("gather_l2_scatter_hbm", 2048, 1, 1),
                                 # gather sets that fit the 256 MB memory-side cache: the Q rows of one kv head at 32k (forward walk), its Q and
                                 # dO rows (backward walk), twice that
                                 ("gather_32MB_scatter_hbm", (32 << 20) // 1024, 1, 1), ("gather2_64MB_scatter1_hbm", (64 << 20) // 1024, 2, 1),
                                 ("gather2_128MB_scatter1_hbm", (128 << 20) // 1024, 2, 1), ("gather_128MB", (128 << 20) // 1024, 2, 0)):
            best = None
            for rep in range(4):
                e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                e0.record()
                _lib.check(L.nsa_probe_row_traffic(P(src), sr, P(dst), rows_big, rd, wr, iters, waves, 1, 1000 * rep, stream), "probe")
                e1.record()
                torch.cuda.synchronize()
                t = e0.elapsed_time(e1)
                best = t if rep > 0 and (best is None or t < best) else best
            probe[name] = round(waves * iters * 4 * (rd + wr) * 1024 / (best * 1e-3) / 1e9, 1)
        res["row_traffic_GBs"] = probe
        del src, dst
    except _Skip:
        pass
    except Exception as ex:
        res["row_traffic_GBs"] = dict(error=repr(ex))

    if not args.no_cpu:
        torch.set_num_threads(min(16, os.cpu_count() or 1))
        base, ref = cpu_baseline(cfg, q, k, v, do, idx, msk)
        res["cpu_baseline"] = base
        # the same path with the module cast to bf16, as the reference's torch path runs then (smaller sample: bf16 CPU GEMMs are slow)
        base16, _ = cpu_baseline(cfg, q, k, v, do, idx, msk, nq=1024, dtype=torch.bfloat16)
        res["cpu_baseline_bf16"] = base16
        err = (out[:, :, n - ref.shape[2]:].float().cpu() - ref).abs().max().item()
        res["config"]["max_abs_err_vs_oracle_sample"] = round(err, 5)
        res["config"]["gpu_over_cpu"] = round(res["config"]["tokens_per_s"] / base["value"], 1)
    print(json.dumps(res))


if __name__ == "__main__":
    main()
