"""The paged-KV work a Qwen3-ASR server has this package do, as measurable cases.

Four kinds of pass, all through the package's public calls:

* ``step``    one decode step of a batch: the step's work list, then every layer's
              append + attention, then the next ids from the step's logits. Captured
              once as a HIP graph and replayed, as decode loops run it; the graph's
              ``max_context_len`` is frozen at its table width (a power of two of
              columns), as the package's graph cache freezes it.
* ``decode``  one layer's ``paged_attention``, called eagerly.
* ``prefill`` one layer of a chunked prefill, called eagerly: the new tokens'
              ``reshape_and_cache``, then ``paged_attention_varlen_prefill``.
* ``gather``  ``gather_kv_cache`` of every sequence's whole context.

A case's context lengths come from its own fields (``rule``, ``lo``, ``hi``, ``lens_seed``);
the seed given to ``prepare`` makes everything else: rows, cache contents, block tables.
"""

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("qwen3asr.rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}
# fp8 scales of a cache whose values reach about 4.5 standard deviations
_K_SCALE, _V_SCALE = 4.5 / 448.0, 4.0 / 448.0


def _case(name, kind, **over):
    c = {"name": name, "kind": kind, "dtype": "bf16", "fp8": False, "heads": 16, "kv_heads": 8,
         "head_dim": 128, "block_size": 16, "batch": 1, "rule": "uniform", "lo": 512, "hi": 512,
         "lens_seed": 1}
    if kind == "step":
        c.update(layers=28, vocab=151936, fused=True)
    if kind == "prefill":
        c.update(new_lo=512, new_hi=512, causal=True)
    c.update(over)
    return c


def listed():
    return [
        # the smallest call: one f32 sequence of 512 tokens, one layer, eager
        _case("decode_f32_one", "decode", dtype="f32"),
        # single-stream transcription: one request's whole decode step (30 s of audio
        # plus the text so far)
        _case("step_one_stream", "step", lo=450, hi=450),
        # a lightly loaded server: 32 requests of mixed length, one step
        _case("step_batch32", "step", batch=32, lo=100, hi=1500, layers=8, lens_seed=2),
        # a loaded server: 256 requests with a geometric length mix
        _case("step_batch256", "step", batch=256, rule="geom", lo=800, hi=4096, layers=4,
              fused=False, lens_seed=5),
        # a few long recordings decoding at once
        _case("decode_long_few", "decode", batch=4, lo=6000, hi=8192, dtype="f16", lens_seed=3),
        # the quantised cache at the loaded server's batch
        _case("decode_fp8", "decode", batch=256, rule="geom", lo=800, hi=4096, fp8=True,
              lens_seed=3),
        # the largest: 1024 sequences of up to 8192 tokens
        _case("decode_batch1024", "decode", batch=1024, lo=256, hi=8192, lens_seed=5),
        # admission of a batch: 64 requests of 512 new tokens over mixed prior contexts
        _case("prefill_batch64", "prefill", batch=64, lo=0, hi=1024, lens_seed=4),
        # one chunk of one long recording
        _case("prefill_one_long", "prefill", batch=1, lo=6000, hi=6000, lens_seed=6),
        # full-precision prefill of a few ragged requests
        _case("prefill_f32", "prefill", dtype="f32", batch=8, lo=0, hi=1024, new_lo=64,
              new_hi=512, lens_seed=7),
        # eight query heads per kv head, f16, ragged
        _case("prefill_group8", "prefill", dtype="f16", heads=32, kv_heads=4, batch=12, lo=0,
              hi=700, new_lo=33, new_hi=450, lens_seed=8),
        # whole contexts copied out of the cache as packed rows
        _case("gather_batch64", "gather", batch=64, lo=512, hi=1536, lens_seed=4),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step"] * 4 + ["decode"] * 3 + ["prefill"] * 4 + ["gather"])
    c = _case("", kind, lens_seed=rng.randrange(1, 1 << 20))
    del c["name"]
    c["block_size"] = rng.choice([16, 16, 16, 32])
    c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if kind in ("step", "decode"):
        # tokens a layer reads, at most the largest listed case's for one layer and
        # a step's over its layers
        c["batch"] = _log_int(rng, 1, 256 if kind == "step" else 1024)
        top = (262144 if kind == "step" else 2097152) // c["batch"]
        mean = _log_int(rng, 64, max(64, min(4096 if kind == "step" else 8192, top)))
        if c["batch"] >= 16 and rng.random() < 0.5:
            c.update(rule="geom", lo=min(mean, 1024), hi=4096)
        else:
            c.update(lo=rng.randrange(mean // 4, mean + 1), hi=mean)
        if kind == "step":
            c["layers"] = 28 if c["batch"] * mean < 20000 else 8 if c["batch"] * mean < 100000 else 4
            c["fused"] = rng.random() < 0.7
            c["fp8"] = rng.random() < 0.15
        else:
            c["heads"], c["kv_heads"] = rng.choice([(16, 8), (16, 8), (32, 8), (24, 8), (16, 16)])
            c["head_dim"] = rng.choice([128, 128, 64])
            c["fp8"] = rng.random() < 0.25
            if not c["fp8"] and c["batch"] * mean < 200000 and rng.random() < 0.25:
                c["dtype"] = "f32"
    elif kind == "prefill":
        c["heads"], c["kv_heads"] = rng.choice([(16, 8), (16, 8), (16, 8), (32, 4), (24, 8)])
        c["causal"] = rng.random() < 0.8
        c["batch"] = _log_int(rng, 1, 64)
        new = _log_int(rng, 16, max(16, min(1024, 32768 // c["batch"])))
        c.update(new_lo=rng.randrange(max(1, new // 3), new + 1), new_hi=new)
        prior = rng.choice([0, 0, _log_int(rng, 16, 1024), _log_int(rng, 16, 6000)])
        if c["batch"] * new * (new + prior) > 32768 * 1100:
            prior = min(prior, 512)
        c.update(lo=rng.randrange(0, prior + 1), hi=prior)
        group = c["heads"] // c["kv_heads"]
        small = c["batch"] * new * (new + prior) * c["heads"] < 16 * 4000000
        if small and rng.random() < 0.25:
            c["dtype"] = "f32"
        elif not small and group not in (1, 2, 4):
            c["heads"], c["kv_heads"] = 16, 8
        if c["dtype"] != "f32":
            c["fp8"] = rng.random() < 0.2
    else:
        c["batch"] = _log_int(rng, 1, 128)
        mean = _log_int(rng, 64, max(64, min(8192, 131072 // c["batch"])))
        c.update(lo=rng.randrange(mean // 4, mean + 1), hi=mean)
        c["fp8"] = rng.random() < 0.25
    return c


# ---- sizes, from the case alone ------------------------------------------------------


def _lens(case):
    """(tokens each sequence's cache holds, new tokens of them) as int64 arrays."""
    rng = np.random.default_rng(case["lens_seed"])
    b = case["batch"]
    if case["rule"] == "geom":
        ctx = np.clip(rng.geometric(1.0 / case["lo"], size=b), 16, case["hi"])
    else:
        ctx = rng.integers(case["lo"], case["hi"], size=b, endpoint=True)
    ctx = ctx.astype(np.int64)
    if case["kind"] == "prefill":
        new = rng.integers(case["new_lo"], case["new_hi"], size=b, endpoint=True).astype(np.int64)
        return ctx + new, new
    return np.maximum(ctx, 1), np.ones(b, np.int64)


def _blocks(case, lens):
    return (lens + case["block_size"] - 1) // case["block_size"]


def _kv_bytes(case):
    """K and V bytes of one cached token of one layer."""
    return 2 * case["kv_heads"] * case["head_dim"] * (1 if case["fp8"] else _BYTES[case["dtype"]])


def work(case):
    lens, new = _lens(case)
    e, kvb = _BYTES[case["dtype"]], _kv_bytes(case)
    rows = 2 * case["kv_heads"] * case["head_dim"] * e  # new K and V of one token
    q_row = case["heads"] * case["head_dim"]
    meta = 4 * int(_blocks(case, lens).sum()) + 4 * len(lens)
    total = int(lens.sum())
    if case["kind"] == "gather":
        return {"bytes": total * (kvb + rows) + meta, "flops": 0}
    if case["kind"] == "prefill":
        keys = new * (lens - new) + new * (new + 1) // 2 if case["causal"] else new * lens
        n = int(new.sum())
        return {"bytes": total * kvb + n * (rows + kvb) + 2 * n * q_row * e + 8 * n + meta,
                "flops": 4 * q_row * int(keys.sum())}
    b = len(lens)
    one = total * kvb + 2 * b * q_row * e + meta
    if case["kind"] == "decode":
        return {"bytes": one, "flops": 4 * q_row * total}
    return {"bytes": case["layers"] * (one + b * (rows + kvb)) + b * case["vocab"] * 2,
            "flops": case["layers"] * 4 * q_row * total}


def tolerance(case):
    # 32-bit sums in another order; one 16-bit rounding of probabilities and outputs
    if case["kind"] == "gather":
        return "exact" if not case["fp8"] else {"rel": 1e-6}
    if case["dtype"] == "f32":
        return {"rel": 2e-6, "max": 1e-4}
    if case["dtype"] == "f16" and not case["fp8"]:
        return {"rel": 2e-3, "max": 3e-2}
    return {"rel": 1.2e-2, "max": 1.5e-1}


# ---- inputs ---------------------------------------------------------------------------


def _inputs(case, seed):
    """Plain tensors of one pass; no call of the package."""
    dev = torch.device("cuda")
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    lens, new = _lens(case)
    need = _blocks(case, lens)
    b, bs, d, kvh = len(lens), case["block_size"], case["head_dim"], case["kv_heads"]
    dt = _TORCH[case["dtype"]]
    total = int(need.sum())
    nb = total + 1 + total // 8  # block 0 is the null block; some slack
    cols = int(need.max())
    if case["kind"] == "step":  # the width a captured graph is keyed by
        cols = max(1 << (cols - 1).bit_length(), 256 // bs)
    ids = rng.permutation(np.arange(1, nb, dtype=np.int64))[:total]
    tables = np.zeros((b, cols), np.uint32)
    at = np.concatenate([[0], np.cumsum(need)])
    for s in range(b):
        tables[s, :need[s]] = ids[at[s]:at[s + 1]]
    cu_q = np.concatenate([[0], np.cumsum(new)])
    pos = [np.arange(n - k, n) for n, k in zip(lens, new)]
    slots = np.concatenate([tables[s, p // bs].astype(np.int64) * bs + p % bs
                            for s, p in enumerate(pos)])
    t = {"tables": torch.from_numpy(tables).to(dev),
         "lens": torch.from_numpy(lens.astype(np.uint32)).to(dev),
         "cu_q": torch.from_numpy(cu_q.astype(np.uint32)).to(dev),
         "cu_kv": torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)).to(dev),
         "slots": torch.from_numpy(slots).to(dev),
         "np_tables": tables, "np_lens": lens, "np_new": new}

    def rand(*shape):
        return torch.empty(shape, dtype=dt, device=dev).normal_(generator=gen)

    layers = case.get("layers", 1)
    x = 16 if case["fp8"] else 16 // _BYTES[case["dtype"]]

    def cache(shape, scale):
        if not case["fp8"]:
            return rand(layers, *shape)
        c = torch.empty((layers,) + shape, dtype=torch.uint8, device=dev)
        for lay in range(layers):
            c[lay] = (rand(*shape) / scale).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        return c

    t["kc"] = cache((nb, kvh, d // x, bs, x), _K_SCALE)
    t["vc"] = cache((nb, kvh, d, bs), _V_SCALE)
    t["ks"] = t["vs"] = None
    if case["fp8"]:
        t["ks"] = torch.tensor([_K_SCALE], dtype=torch.float32, device=dev)
        t["vs"] = torch.tensor([_V_SCALE], dtype=torch.float32, device=dev)
    if case["kind"] != "gather":
        n = int(new.sum())
        t["q"] = rand(layers, n, case["heads"], d)
        t["k"] = rand(layers, n, kvh, d)
        t["v"] = rand(layers, n, kvh, d)
    if case["kind"] == "step":
        t["logits"] = torch.empty((b, case["vocab"]), dtype=torch.bfloat16,
                                  device=dev).normal_(generator=gen)
    return t


def _step_pass(vpa, case, t, max_ctx, ws):
    outs, ids = t["out"], t["ids"]
    vpa.paged_attention_plan(t["lens"], max_ctx, t["tables"].shape[1], case["heads"], t["kc"][0],
                             t["vc"][0], t["q"].dtype, ws)
    scale = case["head_dim"] ** -0.5
    for i in range(case["layers"]):
        q, k, v, kc, vc = t["q"][i], t["k"][i], t["v"][i], t["kc"][i], t["vc"][i]
        if case["fused"]:
            vpa.reshape_and_cache_paged_attention(q, k, v, t["ks"], t["vs"], kc, vc, t["tables"],
                                                  t["lens"], max_ctx, scale, out=outs[i],
                                                  workspace=ws, planned=True)
        else:
            vpa.reshape_and_cache(k, v, t["ks"], t["vs"], kc, vc, t["slots"])
            vpa.paged_attention(q, t["ks"], t["vs"], kc, vc, t["tables"], t["lens"], None, max_ctx,
                                scale, 1.0, None, out=outs[i], workspace=ws, planned=True)
    vpa.argmax_token_ids_from_logits(t["logits"], out=ids)


def prepare(case, seed):
    import vpa

    t = _inputs(case, seed)
    state = {"case": case, "t": t, "max_ctx": int(t["np_lens"].max()),
             "max_new": int(t["np_new"].max()), "total": int(t["np_lens"].sum())}
    if case["kind"] == "step":
        max_ctx = t["tables"].shape[1] * case["block_size"]
        t["out"] = torch.empty_like(t["q"])
        t["ids"] = torch.empty(case["batch"], dtype=torch.uint32, device="cuda")
        ws = vpa.paged_attention_workspace(case["batch"], case["heads"], case["head_dim"], max_ctx,
                                           "cuda")
        _step_pass(vpa, case, t, max_ctx, ws)  # warm-up before the capture
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            _step_pass(vpa, case, t, max_ctx, ws)
        state.update(graph=graph, workspace=ws)
    return state


def run(state):
    import vpa

    case, t = state["case"], state["t"]
    if case["kind"] == "step":
        state["graph"].replay()
        return {"out": t["out"], "ids": t["ids"].view(torch.int32), "key_cache": t["kc"],
                "value_cache": t["vc"]}
    kc, vc = t["kc"][0], t["vc"][0]
    scale = case["head_dim"] ** -0.5
    if case["kind"] == "decode":
        return vpa.paged_attention(t["q"][0], t["ks"], t["vs"], kc, vc, t["tables"], t["lens"],
                                   None, state["max_ctx"], scale, 1.0, None)
    if case["kind"] == "gather":
        return vpa.gather_kv_cache(kc, vc, t["ks"], t["vs"], t["tables"], t["cu_kv"],
                                   _TORCH[case["dtype"]], total_tokens=state["total"])
    vpa.reshape_and_cache(t["k"][0], t["v"][0], t["ks"], t["vs"], kc, vc, t["slots"])
    out = vpa.paged_attention_varlen_prefill(
        t["q"][0], kc, vc, t["tables"], t["lens"], t["cu_q"], t["ks"], t["vs"], scale, 1.0,
        causal=case["causal"], max_query_len=state["max_new"], max_context_len=state["max_ctx"])
    return {"out": out, "key_cache": kc, "value_cache": vc}


# ---- the same in 64 bits with plain torch ------------------------------------------------


def _fp8_bytes(x, scale):
    return (x.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)


def exact(case, seed):
    t = _inputs(case, seed)
    bs, d, h, kvh = case["block_size"], case["head_dim"], case["heads"], case["kv_heads"]
    lens, new = t["np_lens"], t["np_new"]
    starts = np.concatenate([[0], np.cumsum(new)])
    tables = t["tables"].view(torch.int32).long()

    def rows(layer, s):
        """K and V of sequence s, [kv_heads, tokens, head_dim] in 64 bits."""
        ids = tables[s, :int(_blocks(case, lens[s]))]
        k, v = t["kc"][layer][ids], t["vc"][layer][ids]
        if case["fp8"]:
            k, v = k.view(torch.float8_e4m3fn), v.view(torch.float8_e4m3fn)
        k = k.double().permute(1, 0, 3, 2, 4).reshape(kvh, -1, d)[:, :lens[s]]
        v = v.double().permute(1, 0, 3, 2).reshape(kvh, -1, d)[:, :lens[s]]
        return (k * t["ks"].double(), v * t["vs"].double()) if case["fp8"] else (k, v)

    if case["kind"] == "gather":
        both = [rows(0, s) for s in range(len(lens))]
        return tuple(torch.cat([p[i].transpose(0, 1) for p in both]) for i in (0, 1))
    scale, group = d ** -0.5, h // kvh
    causal = case["kind"] != "prefill" or case["causal"]
    eps = 0.0 if case["kind"] == "prefill" and case["causal"] else 1e-6
    outs = []
    for layer in range(case.get("layers", 1)):
        out = torch.empty(t["q"][layer].shape, dtype=torch.float64, device="cuda")
        for s in range(len(lens)):
            k, v = rows(layer, s)
            a, b, n = int(starts[s]), int(starts[s + 1]), int(lens[s])
            if case["kind"] != "decode":  # the new rows, as the cache then holds them
                nk, nv = t["k"][layer][a:b], t["v"][layer][a:b]
                if case["fp8"]:
                    nk = _fp8_bytes(nk, t["ks"]).view(torch.float8_e4m3fn).double() * t["ks"].double()
                    nv = _fp8_bytes(nv, t["vs"]).view(torch.float8_e4m3fn).double() * t["vs"].double()
                k, v = k.clone(), v.clone()
                k[:, n - (b - a):] = nk.double().transpose(0, 1)
                v[:, n - (b - a):] = nv.double().transpose(0, 1)
            q = t["q"][layer][a:b].double().reshape(b - a, kvh, group, d).permute(1, 2, 0, 3)
            score = torch.matmul(q.reshape(kvh, group * (b - a), d), k.transpose(1, 2).contiguous())
            score = score.reshape(kvh, group, b - a, n) * scale
            if causal and b - a > 1:
                at = torch.arange(n, device="cuda")
                last = torch.arange(n - (b - a), n, device="cuda")
                score.masked_fill_(at[None, :] > last[:, None], -math.inf)
            p = torch.exp(score - score.max(dim=-1, keepdim=True).values)
            p = p / (p.sum(dim=-1, keepdim=True) + eps)
            o = torch.matmul(p.reshape(kvh, group * (b - a), n), v)
            out[a:b] = o.reshape(kvh, group, b - a, d).permute(2, 0, 1, 3).reshape(b - a, h, d)
        outs.append(out)
    if case["kind"] == "decode":
        return outs[0]
    if case["kind"] == "prefill":
        return {"out": outs[0], "key_cache": None, "value_cache": None}
    return {"out": torch.stack(outs), "ids": None, "key_cache": None, "value_cache": None}
