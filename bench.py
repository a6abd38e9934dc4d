#!/usr/bin/env python3
"""Benchmark of the paged-KV decode step at Qwen3-ASR decoder shapes.

A step is one decode step of the hot path over one batch: for each of the 28
decoder layers, reshape_and_cache of the batch's new K/V rows followed by
paged_attention over the paged cache (the per-layer calls of
vasr-models/src/model/thinker_text.rs:1101-1139); the decode work list is
built once per step (paged_attention_plan) and shared by the 28 calls. Default workload: c3 —
bf16, batch 256, 16 q heads / 8 kv heads / head_dim 128, block 16, context
lengths clip(Geom(mean 800), 16, 4096), every layer with its own pool and
random block allocation. Inputs are synthetic (seeded) and resident in HBM
before the timed region starts.

The timed step is a HIP graph of the 28 layers replayed K times (vASR
replays its decode step from a CUDA graph, vasr-paged-attn/src/cuda_graph.rs:
204-225); `--eager` times eager launches instead. HIP events sit only at the
two ends of each timed region.

Prints one JSON line. `value` is the whole-step HBM throughput: algorithmic
bytes of all appends and decodes of a step divided by the step time. Each op
is also timed on its own from a graph of the step's layers: the `roofline`
object covers the dominant op (paged_attention: plan, rows and merge
launches), with the rate of the same reads with no compute
(`vpa_paged_cache_read`) as `measured_peak`; `decode_in_step_*` is the
decode as the step runs it, right after its layer's append (step minus the
appends alone); `append_*` is reshape_and_cache; `decode_seeds` repeats the
decode over c3 seeds 1-5; `cpu_baseline` times the oracle's restatement of
the reference CPU path on a bounded sample; `prefill_c4` reports the
chunked-prefill row (append + MFMA prefill) on c4;
`decode_append_fused_small_batches` times the step at batches 1, 8 and 32
with each layer's append and decode behind
vpa_reshape_and_cache_paged_attention (one launch at those sizes) against
the two calls. `--fused-append` runs the timed step through that entry point.
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for _p in (ROOT, os.path.join(ROOT, "qwen3asr.rs_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

HBM_PEAK_GBPS = 8000.0  # MI355X HBM3E, 8 TB/s
MFMA_BF16_PEAK_TFLOPS = 2500.0  # MI355X dense bf16 MFMA
METRIC = "paged-attn decode HBM GB/s (% of peak) + KV-append GB/s at Qwen3-ASR shapes"


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", default="c3", choices=["c2", "c3", "c5"])
    ap.add_argument("--layers", type=int, default=None, help="override the layer count")
    ap.add_argument("--cpu-seconds", type=float, default=12.0,
                    help="CPU baseline budget (0 disables it)")
    ap.add_argument("--seed", type=int, default=None)
    ap.add_argument("--eager", action="store_true",
                    help="time the step as eager launches instead of a HIP graph replay")
    ap.add_argument("--no-prefill", dest="prefill", action="store_false",
                    help="skip the c4 chunked-prefill measurement")
    ap.add_argument("--no-fp8", dest="fp8", action="store_false",
                    help="skip the fp8-cache decode measurement")
    ap.add_argument("--no-device-step", dest="device_step", action="store_false",
                    help="skip the device-resident whole-step measurement")
    ap.add_argument("--seeds", default="1,2,3,4,5",
                    help="c3 seeds of the decode sweep (empty: skip it)")
    ap.add_argument("--fused-append", action="store_true",
                    help="run each layer's append + decode through "
                         "vpa_reshape_and_cache_paged_attention instead of the two calls")
    ap.add_argument("--no-small-batches", dest="small_batches", action="store_false",
                    help="skip the small-batch comparison of the fused append + decode")
    return ap.parse_args()


def build_workload(args):
    from vpa import workloads

    kw = {}
    if args.seed is not None:
        kw["seed"] = args.seed
    if args.layers is not None and args.workload in ("c3", "c5"):
        kw["num_layers"] = args.layers
    return workloads.CONFIGS[args.workload](**kw)


def device_tensors(w, dev):
    import numpy as np
    import torch

    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[w.dtype]
    g = torch.Generator(device=dev)
    g.manual_seed(w.seed)
    x = 16 // w.elem_bytes
    B, H, KVH, D, BS = w.num_seqs, w.num_heads, w.num_kv_heads, w.head_dim, w.block_size
    layers = []
    pool = None
    for i, layer in enumerate(w.layers):
        if pool is None or not w.shared_pool:
            kc = torch.randn((layer.num_blocks, KVH, D // x, BS, x), generator=g, device=dev,
                             dtype=dt)
            vc = torch.randn((layer.num_blocks, KVH, D, BS), generator=g, device=dev, dtype=dt)
            pool = (kc, vc)
        kc, vc = pool
        layers.append(dict(
            kc=kc, vc=vc,
            q=torch.randn((B, H, D), generator=g, device=dev, dtype=dt),
            k=torch.randn((B, KVH, D), generator=g, device=dev, dtype=dt),
            v=torch.randn((B, KVH, D), generator=g, device=dev, dtype=dt),
            out=torch.empty((B, H, D), device=dev, dtype=dt),
            bt=torch.from_numpy(layer.block_tables).to(dev),
            slots=torch.from_numpy(layer.slot_mapping.astype(np.int64)).to(dev),
        ))
    ctx = torch.from_numpy(w.context_lens).to(dev)
    return layers, ctx


def plan_step(layers, ctx, w, ws):
    """The step's decode work list, built once for all layers (the layers
    share the step's context lengths and block-table width)."""
    import torch

    import vpa

    L = layers[0]
    vpa.paged_attention_plan(ctx, w.max_context_len, L["bt"].shape[1], w.num_heads, L["kc"],
                             L["vc"], L["q"].dtype, ws)


def decode_ops(layers, ctx, w, ws):
    """Per layer: paged_attention over the layer's cache (thinker_text.rs:1126-1139)."""
    import vpa

    scale = w.head_dim ** -0.5
    plan_step(layers, ctx, w, ws)
    for L in layers:
        vpa.paged_attention(L["q"], None, None, L["kc"], L["vc"], L["bt"], ctx, None,
                            w.max_context_len, scale, 1.0, None, out=L["out"], workspace=ws,
                            planned=True)


def append_ops(layers):
    """Per layer: reshape_and_cache of the batch's new K/V (thinker_text.rs:1101-1109)."""
    import vpa

    for L in layers:
        vpa.reshape_and_cache(L["k"], L["v"], None, None, L["kc"], L["vc"], L["slots"])


def run_step(layers, ctx, w, ws):
    """One decode step of the hot path: the step's work list, then for each
    layer append and attend."""
    import vpa

    scale = w.head_dim ** -0.5
    plan_step(layers, ctx, w, ws)
    for L in layers:
        vpa.reshape_and_cache(L["k"], L["v"], None, None, L["kc"], L["vc"], L["slots"])
        vpa.paged_attention(L["q"], None, None, L["kc"], L["vc"], L["bt"], ctx, None,
                            w.max_context_len, scale, 1.0, None, out=L["out"], workspace=ws,
                            planned=True)


def run_step_fused(layers, ctx, w, ws):
    """The same step with each layer's append and attention behind one call
    (vpa_reshape_and_cache_paged_attention: one launch for small batches)."""
    import vpa

    scale = w.head_dim ** -0.5
    plan_step(layers, ctx, w, ws)
    for L in layers:
        vpa.reshape_and_cache_paged_attention(L["q"], L["k"], L["v"], None, None, L["kc"],
                                              L["vc"], L["bt"], ctx, w.max_context_len, scale,
                                              out=L["out"], workspace=ws, planned=True)


def small_batches(dev, reps, warmup, batches=(1, 8, 32)):
    """c3's length rule at small batches (28 layers, graphs of the step): the
    two calls per layer against vpa_reshape_and_cache_paged_attention, which
    appends inside the decode launch at these sizes."""
    import torch

    import vpa
    from vpa import workloads

    rows = []
    for b in batches:
        w = workloads.c3(batch=b)
        layers, ctx = device_tensors(w, dev)
        ws = vpa.paged_attention_workspace(w.num_seqs, w.num_heads, w.head_dim,
                                           w.max_context_len, dev)
        two = graph_of(lambda: run_step(layers, ctx, w, ws))
        one = graph_of(lambda: run_step_fused(layers, ctx, w, ws))
        for _ in range(warmup):
            two.replay()
            one.replay()
        t_two = timed_ms(two.replay, reps)
        t_one = timed_ms(one.replay, reps)
        rows.append({"batch": b, "mean_context": round(float(w.context_lens.mean()), 1),
                     "two_calls_us_per_step": round(t_two * 1e3, 2),
                     "fused_us_per_step": round(t_one * 1e3, 2),
                     "speedup": round(t_two / t_one, 3)})
        del layers, ws, two, one
        torch.cuda.empty_cache()
    return {"workload": "c3 length rule, 28 layers", "rows": rows,
            "what": "us per decode step (graph replay): reshape_and_cache + paged_attention "
                    "per layer, against vpa_reshape_and_cache_paged_attention per layer"}


def timed_ms(fn, reps):
    """Milliseconds per call of fn over `reps` back-to-back calls: HIP events
    on the current stream at the two ends of the region only, with a device
    synchronisation on both sides."""
    import torch

    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    torch.cuda.synchronize()
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps


def cpu_baseline(w, layers, budget_s):
    """Time the oracle's restatement of the reference CPU decode path on a
    bounded sample of the same workload: groups of up to 256 sequences of a
    layer (c3: whole layers), in order, until the time budget is spent. Each
    group's blocks are copied to host memory with its tables renumbered over
    them (the c5 pool does not fit host memory)."""
    import numpy as np
    import torch

    from oracle import oracle as orc
    from vpa import workloads

    code = {"bf16": orc.BF16, "f16": orc.F16, "f32": orc.F32}[w.dtype]

    def host(t):
        t = t.detach().cpu().contiguous()
        if t.dtype == torch.float32:
            return t.numpy()
        return t.view(torch.int16).numpy().view(np.uint16)

    scale = w.head_dim ** -0.5
    kvb = w.kv_bytes_per_token()
    group = min(w.num_seqs, 256)
    done_bytes = 0
    elapsed = 0.0
    seq_layers = 0
    groups = 0
    threads = 1
    for i, L in enumerate(layers):
        meta = w.layers[i]
        for s0 in range(0, w.num_seqs, group):
            sl = slice(s0, s0 + group)
            lens = w.context_lens[sl]
            blocks, bt, slots = workloads.compact_tables(meta.block_tables[sl], lens,
                                                         w.block_size, meta.slot_mapping[sl])
            idx = torch.from_numpy(blocks).to(L["kc"].device)
            kc, vc = host(L["kc"].index_select(0, idx)), host(L["vc"].index_select(0, idx))
            q, k, v = host(L["q"][sl]), host(L["k"][sl]), host(L["v"][sl])
            t0 = time.perf_counter()
            _, threads = orc.cpu_baseline_decode_step(q, k, v, slots, kc, vc, bt, lens, scale,
                                                      dtype=code)
            elapsed += time.perf_counter() - t0
            n = lens.astype(np.int64)
            done_bytes += int((n * kvb + 2 * w.num_heads * w.head_dim * w.elem_bytes
                               + 4 * ((n + w.block_size - 1) // w.block_size) + 4
                               + 2 * kvb + 8).sum())
            seq_layers += len(n)
            groups += 1
            if elapsed >= budget_s:
                break
        if elapsed >= budget_s:
            break
    gbps = done_bytes / elapsed / 1e9
    return {
        "value": round(gbps, 3),
        "unit": "GB/s",
        "cores": int(threads),
        "cpu_model": cpu_model(),
        "kind": "port",
        "sample": (f"{groups} group(s) of up to {group} sequences of one layer of {w.name} "
                   f"({seq_layers} sequence-layers of {w.num_seqs} x {len(layers)}, append + "
                   f"decode), {elapsed:.1f} s on {os.cpu_count()} visible host CPUs"),
    }


def decode_fp8(w, dev, reps, warm_s=0.25):
    """The decode-only region of the step over fp8 (E4M3FN) caches: the same
    block tables, lengths and bf16 queries, K/V bytes halved; plan once, then
    the planned call per layer. Returns GB/s of the fp8 op's algorithmic
    bytes and its fraction of the HBM peak."""
    import numpy as np
    import torch

    import vpa

    B, H, KVH, D, BS = w.num_seqs, w.num_heads, w.num_kv_heads, w.head_dim, w.block_size
    g = torch.Generator(device=dev)
    g.manual_seed(w.seed + 1)
    one = torch.ones(1, dtype=torch.float32, device=dev)

    def fp8_cache(shape):
        b = torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
        b[(b & 0x7F) == 0x7F] = 0x38  # no NaN codes
        return b.view(torch.float8_e4m3fn)

    layers = []
    pool = None
    for layer in w.layers:
        if pool is None or not w.shared_pool:
            pool = (fp8_cache((layer.num_blocks, KVH, D // 16, BS, 16)),
                    fp8_cache((layer.num_blocks, KVH, D, BS)))
        layers.append(dict(kc=pool[0], vc=pool[1],
                           q=torch.randn((B, H, D), generator=g, device=dev, dtype=torch.bfloat16),
                           out=torch.empty((B, H, D), device=dev, dtype=torch.bfloat16),
                           bt=torch.from_numpy(layer.block_tables).to(dev)))
    ctx = torch.from_numpy(w.context_lens).to(dev)
    ws = vpa.paged_attention_workspace(B, H, D, w.max_context_len, dev)
    scale = D ** -0.5

    def run():
        L0 = layers[0]
        vpa.paged_attention_plan(ctx, w.max_context_len, L0["bt"].shape[1], H, L0["kc"],
                                 L0["vc"], torch.bfloat16, ws)
        for L in layers:
            vpa.paged_attention(L["q"], one, one, L["kc"], L["vc"], L["bt"], ctx, None,
                                w.max_context_len, scale, 1.0, None, out=L["out"],
                                workspace=ws, planned=True)

    # the same tiles read with no compute (vpa_paged_cache_read over the same
    # work list): the gather rate the fp8 pattern can reach
    sink = torch.zeros(1, dtype=torch.uint32, device=dev)

    def read():
        L0 = layers[0]
        vpa.paged_attention_plan(ctx, w.max_context_len, L0["bt"].shape[1], H, L0["kc"],
                                 L0["vc"], torch.bfloat16, ws)
        for L in layers:
            vpa.paged_cache_read(L["kc"], L["vc"], L["bt"], w.max_context_len, H, ws, sink)

    # (after the CPU baseline the GPU has idled: run for warm_s first)
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < warm_s:
        timed_ms(run, 2)
    ms = timed_ms(run, reps) / len(layers)
    read_ms = timed_ms(read, reps) / len(layers)
    lens = w.context_lens.astype(np.int64)
    per = (lens * 2 * KVH * D + 2 * H * D * 2 + 4 * ((lens + BS - 1) // BS) + 4)
    nbytes = int(per.sum())
    gbps = nbytes / (ms * 1e-3) / 1e9
    read_gbps = nbytes / (read_ms * 1e-3) / 1e9
    del layers, ws
    torch.cuda.empty_cache()
    return {"workload": w.name, "cache": "fp8_e4m3 (k_scale = v_scale = 1)", "query": "bf16",
            "us_per_launch": round(ms * 1e3, 2), "algorithmic_bytes_per_launch": nbytes,
            "gbps": round(gbps, 2), "frac_of_peak": round(gbps / HBM_PEAK_GBPS, 4),
            "read_us_per_launch": round(read_ms * 1e3, 2), "measured_peak": round(read_gbps, 2),
            "measured_peak_what": "vpa_paged_cache_read over the fp8 caches (same work list, "
                                  "no compute)",
            "frac_of_measured": round(gbps / read_gbps, 4)}


def device_step(w, dev, reps, warmup):
    """The whole decode step kept on the device (vpa.DeviceDecodeStep) on c3's
    batch and lengths: token bookkeeping, block growth and step metadata,
    the work list, 28 x (append + attention) and the argmax over a
    [256, 151936] logits buffer, captured as one HIP graph and replayed back
    to back. Beside it the same step driven from the host the way the
    reference's loop runs it (paged_batch_engine.rs:629-722): read the ids
    back, EOS bookkeeping on the host, grow blocks with the host block
    manager, upload slot_mapping / context_lens / block tables, then replay
    a graph of the device work (work list, layers, argmax). The layers
    share one block table (one block manager per model), each with its own
    cache pool. Host work here is this package's host mirror (numpy and
    the C++ block manager through ctypes), slower than the reference's Rust
    loop; the device step's figure does not depend on it."""
    import numpy as np
    import torch

    import vpa
    from vpa import host

    B, H, KVH, D, BS = w.num_seqs, w.num_heads, w.num_kv_heads, w.head_dim, w.block_size
    vocab, eos = 151936, [151643, 151645]  # Qwen3 vocabulary, <|endoftext|> / <|im_end|>
    n_steps = 3 * (reps + warmup) + 4
    prompts = (w.context_lens.astype(np.int64) - 1)
    max_ctx = int(prompts.max()) + n_steps + 1
    need = int(((prompts + n_steps + BS) // BS).sum())
    nb = need + 1 + need // 8
    bf = torch.bfloat16
    g = torch.Generator(device=dev)
    g.manual_seed(w.seed + 2)
    layers = [dict(kc=torch.randn((nb, KVH, D // 8, BS, 8), generator=g, device=dev, dtype=bf),
                   vc=torch.randn((nb, KVH, D, BS), generator=g, device=dev, dtype=bf),
                   q=torch.randn((B, H, D), generator=g, device=dev, dtype=bf),
                   k=torch.randn((B, KVH, D), generator=g, device=dev, dtype=bf),
                   v=torch.randn((B, KVH, D), generator=g, device=dev, dtype=bf),
                   out=torch.empty((B, H, D), device=dev, dtype=bf)) for _ in range(len(w.layers))]
    logits = torch.randn((B, vocab), generator=g, device=dev, dtype=bf)
    st = vpa.DeviceDecodeStep(B, nb, BS, max_ctx, H, D, eos, n_steps + 1, dev)
    st.admit(torch.from_numpy(prompts.astype(np.uint32)).to(dev))
    L0 = layers[0]

    def work():  # the device work of a step after its metadata
        vpa.paged_attention_plan(st.allocator.context_lens, max_ctx, st.cols, H, L0["kc"],
                                 L0["vc"], bf, st.workspace)
        for L in layers:
            st.layer(L["q"], L["k"], L["v"], L["kc"], L["vc"], L["out"])
        st.end(logits)

    def book():  # the step's bookkeeping and metadata launches
        st.tokens.consume(st.allocator.slot_mapping)
        st.allocator.step(st.tokens.finished)

    def full():
        book()
        work()

    torch.cuda.synchronize()
    g_full, g_work, g_book = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g_full):
        full()
    with torch.cuda.graph(g_work):
        work()
    with torch.cuda.graph(g_book):
        book()
    torch.cuda.synchronize()
    for _ in range(warmup):
        g_full.replay()
    dev_ms = timed_ms(g_full.replay, reps)

    # host-driven: the host block manager follows the device allocator's state
    mgr = host.BlockManager(nb, BS)
    pos = (st.allocator.positions.cpu().numpy().astype(np.int64))
    tables = st.allocator.block_tables.cpu().numpy()
    nblk = st.allocator.row_blocks.cpu().numpy().astype(np.int64)
    fin = st.tokens.finished.cpu().numpy().astype(bool)
    for r in range(B):
        assert mgr.try_allocate_slots(r, int(nblk[r]) * BS)
        tables[r, :nblk[r]] = mgr.block_ids(r)  # same FIFO order as the ring: ids differ
    st.allocator.block_tables.copy_(torch.from_numpy(tables))
    pin = dict(slots=torch.empty(B, dtype=torch.int64).pin_memory(),
               ctx=torch.empty(B, dtype=torch.uint32).pin_memory(),
               tables=torch.empty(tables.shape, dtype=torch.uint32).pin_memory(),
               ids=torch.empty(B, dtype=torch.uint32).pin_memory())
    eos_arr = np.array(eos, dtype=np.uint32)
    generated = [[] for _ in range(B)]

    def host_step():
        ids = pin["ids"]
        ids.copy_(st.tokens.next_ids)  # read-back: waits for the previous step
        idv = ids.numpy()
        hit = np.isin(idv, eos_arr) & ~fin
        fin[hit] = True
        for r in np.flatnonzero(~fin):
            generated[r].append(int(idv[r]))
        slots = np.full(B, -1, dtype=np.int64)
        ctx = np.ones(B, dtype=np.uint32)
        for r in np.flatnonzero(~fin):
            p = int(pos[r])
            if p // BS >= nblk[r]:
                if not mgr.try_allocate_slots(r, p + 1):
                    continue
                tables[r, nblk[r]] = mgr.block_ids(r)[-1]
                nblk[r] += 1
            slots[r] = int(tables[r, p // BS]) * BS + p % BS
            ctx[r] = p + 1
            pos[r] = p + 1
        pin["slots"].numpy()[:] = slots
        pin["ctx"].numpy()[:] = ctx
        pin["tables"].numpy()[:] = tables
        st.allocator.slot_mapping.copy_(pin["slots"], non_blocking=True)
        st.allocator.context_lens.copy_(pin["ctx"], non_blocking=True)
        st.allocator.block_tables.copy_(pin["tables"], non_blocking=True)
        g_work.replay()

    for _ in range(warmup):
        host_step()
    host_ms = timed_ms(host_step, reps)
    # the bookkeeping and metadata launches alone (each replay is one more
    # step of the allocator; the pool is sized for these steps too)
    torch.cuda.synchronize()
    for _ in range(warmup):
        g_book.replay()
    book_ms = timed_ms(g_book.replay, reps)
    del layers, logits, st, g_full, g_work, g_book
    torch.cuda.empty_cache()
    return {"workload": w.name, "layers": len(w.layers), "vocab": vocab,
            "device_resident_ms_per_step": round(dev_ms, 4),
            "device_bookkeeping_ms_per_step": round(book_ms, 4),
            "host_driven_ms_per_step": round(host_ms, 4),
            "what": "one decode step: bookkeeping + block growth + metadata + work list + "
                    "28 x (append + attention) + argmax; device-resident = one graph replay "
                    "per step, no host read; device bookkeeping = a graph of the step's "
                    "bookkeeping and metadata launches alone; host-driven = ids read back, host "
                    "bookkeeping and block manager, metadata upload, then a graph of the device "
                    "work"}


def prefill_c4(dev, reps=20, warm_s=0.25):
    """Row a3 measured alongside the headline: c4 (64 sequences x 512 new
    tokens over 0..1024 prior tokens, bf16) append with reshape_and_cache,
    then causal chunked-prefill attention over the paged cache, the same
    prefill over fp8 caches, and gather_kv_cache of every sequence's whole
    context to packed rows (the reference's step before its flash prefill);
    HIP events around each op on the current stream."""
    import numpy as np
    import torch

    import vpa
    from vpa import workloads

    w = workloads.c4()
    h, kvh, d, bs = w.num_heads, w.num_kv_heads, w.head_dim, w.block_size
    g = torch.Generator(device=dev)
    g.manual_seed(w.seed)
    bf = torch.bfloat16
    kc = torch.randn((w.num_blocks, kvh, d // 8, bs, 8), generator=g, device=dev, dtype=bf)
    vc = torch.randn((w.num_blocks, kvh, d, bs), generator=g, device=dev, dtype=bf)
    tq = int(w.query_lens.sum())
    q = torch.randn((tq, h, d), generator=g, device=dev, dtype=bf)
    kn = torch.randn((tq, kvh, d), generator=g, device=dev, dtype=bf)
    vn = torch.randn((tq, kvh, d), generator=g, device=dev, dtype=bf)
    slots = torch.from_numpy(w.slot_mapping()).to(dev)
    bt = torch.from_numpy(w.block_tables.astype(np.uint32)).to(dev)
    cl = torch.from_numpy(w.context_lens).to(dev)
    cu = torch.from_numpy(w.cu_seqlens_q).to(dev)
    out = torch.empty_like(q)
    mq, mk = int(w.query_lens.max()), int(w.context_lens.max())

    def append():
        vpa.reshape_and_cache(kn, vn, None, None, kc, vc, slots)

    def prefill():
        vpa.paged_attention_varlen_prefill(q, kc, vc, bt, cl, cu, None, None, d ** -0.5, 1.0,
                                           causal=True, max_query_len=mq, max_context_len=mk,
                                           out=out)

    # the same prefill over fp8 (E4M3FN) caches, scales 1
    one = torch.ones(1, dtype=torch.float32, device=dev)

    def fp8_cache(shape):
        b = torch.randint(0, 256, shape, generator=g, device=dev, dtype=torch.uint8)
        b[(b & 0x7F) == 0x7F] = 0x38  # no NaN codes
        return b.view(torch.float8_e4m3fn)

    kc8 = fp8_cache((w.num_blocks, kvh, d // 16, bs, 16))
    vc8 = fp8_cache((w.num_blocks, kvh, d, bs))
    out8 = torch.empty_like(q)

    def prefill_fp8():
        vpa.paged_attention_varlen_prefill(q, kc8, vc8, bt, cl, cu, one, one, d ** -0.5, 1.0,
                                           causal=True, max_query_len=mq, max_context_len=mk,
                                           out=out8)

    cu_kv = torch.from_numpy(np.concatenate([[0], np.cumsum(w.context_lens)]).astype(np.uint32)
                             ).to(dev)
    kv_tokens = int(w.context_lens.sum())

    def gather():
        vpa.gather_kv_cache(kc, vc, None, None, bt, cu_kv, bf, total_tokens=kv_tokens)

    # Each op is timed twice: over its first calls (after 2 untimed ones),
    # and again once it has run back to back for warm_s seconds. The GPU's
    # clock climbs under a sustained MFMA load: the c4 prefill measured
    # 390-400 us over its first calls and 305-320 us from ~40 ms on
    # (s_memtime against s_memrealtime inside the kernel: 1.99 GHz cold,
    # 2.26 GHz warm). The warm figure is the op's throughput in a stream of
    # prefills; both are reported.
    def timed(fn, n):
        e0 = torch.cuda.Event(enable_timing=True)
        e1 = torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        e0.record()
        for _ in range(n):
            fn()
        e1.record()
        torch.cuda.synchronize()
        return e0.elapsed_time(e1) * 1e3 / n  # us per call

    res, first = {}, {}
    for name, fn in (("append", append), ("prefill", prefill), ("prefill_fp8", prefill_fp8),
                     ("gather", gather)):
        for _ in range(2):
            fn()
        t0 = time.perf_counter()
        first[name] = timed(fn, reps)
        while time.perf_counter() - t0 < warm_s:
            timed(fn, 10)
        res[name] = timed(fn, reps)
    app_bytes = 2 * tq * 2 * kvh * d * 2 + 8 * tq
    gather_bytes = 2 * 2 * kv_tokens * kvh * d * 2  # read the K/V tiles, write the rows
    flops = w.flops()
    tflops = flops / (res["prefill"] * 1e-6) / 1e12
    return {
        "workload": "c4",
        "append_us": round(res["append"], 2),
        "append_first_calls_us": round(first["append"], 2),
        "append_gbps": round(app_bytes / (res["append"] * 1e-6) / 1e9, 2),
        "append_frac_of_peak": round(app_bytes / (res["append"] * 1e-6) / 1e9 / HBM_PEAK_GBPS, 4),
        "prefill_us": round(res["prefill"], 2),
        "prefill_first_calls_us": round(first["prefill"], 2),
        "prefill_tflops": round(tflops, 2),
        "prefill_fp8_cache_us": round(res["prefill_fp8"], 2),
        "prefill_fp8_cache_first_calls_us": round(first["prefill_fp8"], 2),
        "prefill_fp8_cache_tflops": round(flops / (res["prefill_fp8"] * 1e-6) / 1e12, 2),
        "gather_tokens": kv_tokens,
        "gather_us": round(res["gather"], 2),
        "gather_first_calls_us": round(first["gather"], 2),
        "gather_gbps": round(gather_bytes / (res["gather"] * 1e-6) / 1e9, 2),
        "roofline": {"kernel": "chunked_prefill_paged_attention", "bound": "mfma",
                     "achieved": round(tflops, 2), "peak": MFMA_BF16_PEAK_TFLOPS,
                     "unit": "TFLOP/s", "frac": round(tflops / MFMA_BF16_PEAK_TFLOPS, 4),
                     "algorithmic_flops_per_launch": flops},
    }


def graph_of(fn):
    """fn's launches captured once as a HIP graph (after a device sync)."""
    import torch

    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    torch.cuda.synchronize()
    return g


def read_ops(layers, ctx, w, ws, sink):
    """Per layer: the decode's reads with no compute (vpa_paged_cache_read),
    over the step's work list: the achievable gather rate of the pattern."""
    import vpa

    plan_step(layers, ctx, w, ws)
    for L in layers:
        vpa.paged_cache_read(L["kc"], L["vc"], L["bt"], w.max_context_len, w.num_heads, ws, sink)


def op_timings(layers, ctx, w, ws, reps, warmup, sink=None):
    """us per layer of the step's ops, each from a graph of all the step's
    layers replayed back to back (launch gaps of the eager path do not enter):
    decode alone (plan + 28 planned calls), append alone, the whole step, the
    decode inside the step (step minus the appends alone: the decode that
    follows its layer's append, thinker_text.rs:1101-1139, with whatever the
    append leaves behind charged to it) and, with `sink`, the read ceiling."""
    nl = len(layers)
    graphs = {
        "decode": graph_of(lambda: decode_ops(layers, ctx, w, ws)),
        "append": graph_of(lambda: append_ops(layers)),
        "step": graph_of(lambda: run_step(layers, ctx, w, ws)),
    }
    if sink is not None:
        graphs["read"] = graph_of(lambda: read_ops(layers, ctx, w, ws, sink))
    res = {}
    for name, g in graphs.items():
        for _ in range(warmup):
            g.replay()
        res[name] = timed_ms(g.replay, reps) * 1e3 / nl  # us per layer
    res["decode_in_step"] = res["step"] - res["append"]
    return res


def cpu_model() -> str:
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    import platform

    return platform.processor() or "unknown"


def traffic_from_profile(w):
    """HBM bytes per decode launch from the committed rocprofv3 --pmc summary
    of this workload, with the hash of the decode kernels' source it was
    measured on: null when that source has changed since (stale)."""
    import hashlib

    path = os.path.join("profiles", f"paged_decode_{w.name}_traffic.json")
    full = os.path.join(ROOT, path)
    srcs = [os.path.join(ROOT, "qwen3asr.rs_amd", "csrc", f)
            for f in ("decode_rows.h", "decode_kernels.hip")]
    if not os.path.exists(full):
        return None, {"source": path, "status": "absent"}
    with open(full) as f:
        j = json.load(f)
    digest = hashlib.sha256()
    for src in srcs:
        with open(src, "rb") as f:
            digest.update(f.read())
    sha = digest.hexdigest()[:16]
    measured = j.get("decode_kernels_sha256_16")
    stale = measured != sha
    info = {"source": path, "measured_on_decode_kernels_sha256_16": measured,
            "current_decode_kernels_sha256_16": sha, "status": "stale" if stale else "current",
            "how": "rocprofv3 --pmc FETCH_SIZE and --pmc WRITE_SIZE runs of bench.py, per-dispatch "
                   "KiB scaled by a plain-copy calibration (commands in the file)"}
    return (None if stale else j.get("bytes_per_launch")), info


def c3_expected_mean_context():
    """E[clip(Geom(p = 1/800), 16, 4096)], c3's context-length rule (about
    795.4 tokens; a 256-sequence draw scatters around it)."""
    import numpy as np

    p = 1.0 / 800.0
    k = np.arange(1, 200_000, dtype=np.float64)
    pmf = (1.0 - p) ** (k - 1) * p
    return float((np.clip(k, 16, 4096) * pmf).sum())


def decode_seeds(dev, seeds, reps, warmup):
    """The c3 decode over several seeds of its generation rule (each seed
    draws its own lengths and tables): decode alone and inside the step, us
    per layer and fraction of the HBM peak, with each seed's mean context,
    and the read-only pass over the seed's tiles with the decode's fraction
    of it."""
    import numpy as np
    import torch

    import vpa
    from vpa import workloads

    rows = []
    for sd in seeds:
        w = workloads.c3(seed=sd)
        layers, ctx = device_tensors(w, dev)
        ws = vpa.paged_attention_workspace(w.num_seqs, w.num_heads, w.head_dim,
                                           w.max_context_len, dev)
        run_step(layers, ctx, w, ws)
        sink = torch.zeros(1, dtype=torch.uint32, device=dev)
        t = op_timings(layers, ctx, w, ws, reps, warmup, sink=sink)
        b = w.decode_bytes_per_layer()
        rows.append({
            "seed": sd,
            "mean_context": round(float(np.mean(w.context_lens)), 1),
            "decode_us": round(t["decode"], 2),
            "decode_frac_of_peak": round(b / (t["decode"] * 1e-6) / 1e9 / HBM_PEAK_GBPS, 4),
            "decode_in_step_us": round(t["decode_in_step"], 2),
            "decode_in_step_frac_of_peak": round(
                b / (t["decode_in_step"] * 1e-6) / 1e9 / HBM_PEAK_GBPS, 4),
            "read_us": round(t["read"], 2),
            "read_frac_of_peak": round(b / (t["read"] * 1e-6) / 1e9 / HBM_PEAK_GBPS, 4),
            "decode_frac_of_measured": round(t["read"] / t["decode"], 4),
        })
        del layers, ws, ctx
        torch.cuda.empty_cache()
    # the seed whose mean context is nearest the generation rule's expected
    # mean, and the median over the seeds: the representative figures
    expected = c3_expected_mean_context()
    rep = min(rows, key=lambda r: abs(r["mean_context"] - expected))
    return {
        "workload": "c3",
        "seeds": rows,
        "expected_mean_context": round(expected, 1),
        "representative_seed": rep["seed"],
        "representative_decode_frac_of_peak": rep["decode_frac_of_peak"],
        "representative_decode_in_step_frac_of_peak": rep["decode_in_step_frac_of_peak"],
        "median_decode_frac_of_peak": float(np.median([r["decode_frac_of_peak"] for r in rows])),
        "median_decode_in_step_frac_of_peak": float(
            np.median([r["decode_in_step_frac_of_peak"] for r in rows])),
        "min_decode_frac_of_peak": min(r["decode_frac_of_peak"] for r in rows),
        "min_decode_in_step_frac_of_peak": min(r["decode_in_step_frac_of_peak"] for r in rows),
        "min_decode_frac_of_measured": min(r["decode_frac_of_measured"] for r in rows),
    }


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {args.gpus}); the "
              "paged-KV path is measured on one GPU's share: decode and prefill shard by "
              "sequence or by kv head with no exchange inside attention",
              file=sys.stderr)
        sys.exit(2)

    import torch

    import vpa

    dev = torch.device("cuda:0")
    w = build_workload(args)
    layers, ctx = device_tensors(w, dev)
    ws = vpa.paged_attention_workspace(w.num_seqs, w.num_heads, w.head_dim, w.max_context_len,
                                       dev)
    sink = torch.zeros(1, dtype=torch.uint32, device=dev)
    nl = len(layers)

    for _ in range(args.warmup):
        run_step(layers, ctx, w, ws)
    torch.cuda.synchronize()

    # the step as vASR runs decode on the GPU: one HIP graph of the 28 layers
    # (vasr-paged-attn/src/cuda_graph.rs:204-225), replayed; eager launches
    # with --eager
    step_fn = run_step_fused if args.fused_append else run_step
    step = lambda: step_fn(layers, ctx, w, ws)  # noqa: E731
    execution = "eager launches"
    if not args.eager:
        graph = graph_of(step)
        step = graph.replay
        execution = "hip graph replay of the whole step"
        for _ in range(args.warmup):
            step()
    wall0 = time.perf_counter()
    ms_per_step = timed_ms(step, args.steps)
    wall = time.perf_counter() - wall0

    # the eager step for comparison, then each op on its own (graphs of the
    # step's layers): decode, append, decode inside the step, read ceiling
    eager_ms = timed_ms(lambda: step_fn(layers, ctx, w, ws), args.steps)
    ops = op_timings(layers, ctx, w, ws, args.steps, args.warmup, sink=sink)

    dec_bytes = w.decode_bytes_per_layer()
    app_bytes = w.append_bytes_per_layer()
    step_bytes = nl * (dec_bytes + app_bytes)
    value = step_bytes / (ms_per_step * 1e-3) / 1e9

    def gbps(nbytes, us):
        return nbytes / (us * 1e-6) / 1e9

    dec_gbps = gbps(dec_bytes, ops["decode"])
    in_step_gbps = gbps(dec_bytes, ops["decode_in_step"])
    app_gbps = gbps(app_bytes, ops["append"])
    read_gbps = gbps(dec_bytes, ops["read"])
    traffic, traffic_info = traffic_from_profile(w)

    cpu = None
    if args.cpu_seconds > 0:
        cpu = cpu_baseline(w, layers, args.cpu_seconds)
    del layers, ws
    torch.cuda.empty_cache()
    seeds = None
    if args.seeds and w.name == "c3":
        seeds = decode_seeds(dev, [int(x) for x in args.seeds.split(",")], args.steps,
                             args.warmup)
    f8 = None
    if args.fp8 and w.dtype == "bf16":
        f8 = decode_fp8(w, dev, args.steps)
    dstep = None
    if args.device_step and w.name == "c3":
        dstep = device_step(w, dev, args.steps, args.warmup)
    pf = None
    if args.prefill:
        pf = prefill_c4(dev)
    small = None
    if args.small_batches and w.name == "c3":
        small = small_batches(dev, args.steps, args.warmup)

    line = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": w.dtype,
        "data": "synthetic (seeded)",
        "config": {
            "workload": w.name,
            "execution": execution + (" (append + decode per layer behind "
                                      "vpa_reshape_and_cache_paged_attention)"
                                      if args.fused_append else ""),
            "num_seqs": w.num_seqs,
            "layers": nl,
            "q_heads": w.num_heads,
            "kv_heads": w.num_kv_heads,
            "head_dim": w.head_dim,
            "block_size": w.block_size,
            "context_tokens": int(w.context_lens.sum()),
            "mean_context": round(float(w.context_lens.mean()), 1),
            "max_context_len": w.max_context_len,
            "seed": w.seed,
        },
        "eager_ms_per_step": round(eager_ms, 4),
        "eager_value": round(step_bytes / (eager_ms * 1e-3) / 1e9, 2),
        "decode_gbps": round(dec_gbps, 2),
        "decode_frac_of_peak": round(dec_gbps / HBM_PEAK_GBPS, 4),
        "decode_in_step_us": round(ops["decode_in_step"], 2),
        "decode_in_step_gbps": round(in_step_gbps, 2),
        "decode_in_step_frac_of_peak": round(in_step_gbps / HBM_PEAK_GBPS, 4),
        "append_gbps": round(app_gbps, 2),
        "append_us_per_launch": round(ops["append"], 2),
        "wall_s_timed_region": round(wall, 4),
        "roofline": {
            "kernel": "paged_attention (rows + merge launches per layer, plus one plan "
                      "launch per step), a graph of the step's decodes replayed back to back",
            "bound": "hbm",
            "achieved": round(dec_gbps, 2),
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": round(dec_gbps / HBM_PEAK_GBPS, 4),
            "traffic": traffic,
            "traffic_source": traffic_info,
            "algorithmic_bytes_per_launch": dec_bytes,
            "us_per_launch": round(ops["decode"], 2),
            "measured_peak": round(read_gbps, 2),
            "measured_peak_what": "vpa_paged_cache_read: the decode's tile reads (same work "
                                  "list, waves and 16-byte loads) with no compute, same layers",
            "frac_of_measured": round(dec_gbps / read_gbps, 4),
            "read_us_per_launch": round(ops["read"], 2),
        },
        "cpu_baseline": cpu,
        "decode_seeds": seeds,
        "decode_frac_of_peak_representative": (
            None if seeds is None else {
                "seed": seeds["representative_seed"],
                "decode_frac_of_peak": seeds["representative_decode_frac_of_peak"],
                "median_over_seeds": seeds["median_decode_frac_of_peak"],
                "what": "c3 decode at the swept seed whose mean context is nearest the "
                        "rule's expected mean, and the median over the swept seeds; the "
                        "headline config above is seed %d" % w.seed}),
        "decode_fp8": f8,
        "device_step": dstep,
        "prefill_c4": pf,
        "decode_append_fused_small_batches": small,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
