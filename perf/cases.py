"""The calls a serving engine makes into this framework, as timed cases.

Every case is one pass through the package's public entry points: the KV
write of a layer, the FP8 attention reader behind the FA3 entry (decode,
speculative decode, prefill, chunked prefill), a captured decode step, the
MLA latent cache, the gather of long contexts and copy_blocks.  Model shapes:
Llama-3-8B (32 query heads over 8 kv heads of 128), Qwen3 (32 over 4), their
tensor-parallel shards, and DeepSeek-V3's latent (512 + 64).

``listed()`` are the cases themselves, ``draw(rng)`` another of the same
ranges, ``prepare`` what an engine holds before the call, ``run`` the call,
``work`` what it cannot do without, ``exact`` its result in 64 bits.
"""

from __future__ import annotations

import math
import random

import torch

from pipeswift_amd import attention, cache_ops, cudagraph, fp8_kv, impl_utils, mla_fp8
from pipeswift_amd.metadata import KVCacheInfo

D = 128  # head dim of the GQA models
NOPE, ROPE, Q_LORA = 512, 64, 1536  # DeepSeek-V3's latent row and the projection it is a column slice of
DEV = "cuda"


# --------------------------------------------------------------------------- #
# the cases
# --------------------------------------------------------------------------- #


def _attention(kind, seqs, new, ctx_lo, ctx_hi, hq, hkv, page=16, q="fp8", mix=1):
    """new: query tokens of every sequence (decode), or of the whole step, split unevenly (prefill)."""
    return {"kind": kind, "seqs": seqs, "new": new, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "hq": hq, "hkv": hkv,
            "page": page, "q": q, "mix": mix}


def listed():
    return [
        # One layer's KV write of a decode step: 128 sequences, bf16 K and V
        # quantized into the FP8 cache.  The smallest call there is.
        {"name": "append_decode_fp8", "kind": "append", "tokens": 128, "heads": 8, "page": 16, "cache": "fp8",
         "run": 1, "pages": 8192},
        # One layer's KV write of a large prefill batch.
        {"name": "append_prefill_fp8", "kind": "append", "tokens": 16384, "heads": 8, "page": 16, "cache": "fp8",
         "run": 512, "pages": 8192},
        # A layer of a chunked MLA prefill over the tile-scaled FP8 latent
        # cache: the chunk's rows are written, then the whole context is read
        # back as bf16 rows for the prefill attention.
        {"name": "mla_chunk_fp8", "kind": "mla", "tokens": 4096, "seqs": 6, "ctx_lo": 5000, "ctx_hi": 40000, "mix": 4},
        # Long contexts of an FP8 cache read back as contiguous bf16 K and V.
        {"name": "gather_fp8", "kind": "gather", "seqs": 6, "ctx_lo": 7500, "ctx_hi": 60000, "heads": 4, "page": 16,
         "cache": "fp8", "mix": 3},
        # Prefix-cache copy-on-write over a 61-layer stack.
        {"name": "copy_blocks", "kind": "copy", "pairs": 256, "layers": 61, "pages": 1024},
        # A decode step as an engine runs it: captured once, its metadata
        # refreshed and the graph replayed; 8 layers of KV write and attention.
        {"name": "decode_step_graph", "kind": "step", "layers": 8, "seqs": 32, "ctx_lo": 128, "ctx_hi": 8192,
         "hq": 32, "hkv": 8, "page": 16, "mix": 7},
        # One layer's decode attention at a large batch of mixed contexts.
        {"name": "decode_batch128"} | _attention("decode", 128, 1, 128, 32768, 32, 8, mix=2),
        # One long-context request alone on the GPU.
        {"name": "decode_one_131072"} | _attention("decode", 1, 1, 131072, 131072, 32, 8),
        # Speculative decode: 4 causal draft tokens per sequence.
        {"name": "decode_spec4"} | _attention("decode", 32, 4, 512, 16384, 32, 8, mix=5),
        # A chunked-prefill step: 4096 tokens over 6 sequences with long prefixes.
        {"name": "prefill_chunked"} | _attention("prefill", 6, 4096, 14000, 45000, 32, 4, mix=3),
        # A fresh prompt of ordinary length, nothing cached before it.
        {"name": "prefill_prompt"} | _attention("prefill", 1, 2000, 0, 0, 32, 8),
        # The last chunk of a long prompt: few new tokens over a long prefix.
        {"name": "prefill_tail"} | _attention("prefill", 1, 512, 32768, 32768, 32, 8, q="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["append", "decode", "decode", "decode", "prefill", "prefill", "prefill", "step", "gather", "mla",
                       "copy"])
    hq, hkv = rng.choice([(32, 8), (32, 8), (32, 4), (32, 4), (16, 4), (8, 2), (8, 1), (16, 2)])
    page = rng.choice([16, 16, 16, 32, 64, 24])
    mix = rng.randrange(1, 1 << 20)
    if kind == "append":
        return {"kind": kind, "tokens": _log_int(rng, 1, 32768), "heads": rng.choice([1, 2, 4, 8]), "page": page,
                "cache": rng.choice(["fp8", "fp8", "bf16"]), "run": rng.choice([1, 37, 512]), "pages": 8192}
    if kind == "mla":
        hi = _log_int(rng, 2000, 60000)
        return {"kind": kind, "tokens": _log_int(rng, 64, 8192), "seqs": rng.randint(1, 8), "ctx_lo": hi // 8,
                "ctx_hi": hi, "mix": mix}
    if kind == "gather":
        hi = _log_int(rng, 2000, 60000)
        return {"kind": kind, "seqs": rng.randint(1, 8), "ctx_lo": hi // 8, "ctx_hi": hi,
                "heads": rng.choice([1, 2, 4, 8]), "page": page, "cache": rng.choice(["fp8", "bf16"]), "mix": mix}
    if kind == "copy":
        return {"kind": kind, "pairs": _log_int(rng, 4, 400), "layers": rng.randint(8, 61), "pages": 1024}
    if kind == "step":
        return {"kind": kind, "layers": rng.randint(2, 8), "seqs": _log_int(rng, 1, 128), "ctx_lo": 64,
                "ctx_hi": _log_int(rng, 512, 8192), "hq": hq, "hkv": hkv, "page": page, "mix": mix}
    if kind == "decode":
        seqs = _log_int(rng, 1, 256)
        # at most 700k cached tokens in all
        hi = min(_log_int(rng, 256, 131072), max(256, 2 * 700000 // seqs), 131072)
        new = rng.choice([n for n in (1, 1, 1, 2, 3, 4) if n * (hq // hkv) <= 16])
        return _attention("decode", seqs, new, max(16, hi // rng.choice([1, 4, 64])), hi, hq, hkv, page,
                          rng.choice(["fp8", "bf16"]), mix)
    new = _log_int(rng, 48, 8192)
    seqs = rng.randint(1, min(8, new // 24))
    hi = rng.choice([0, _log_int(rng, 256, 45000)])
    case = _attention("prefill", seqs, new, hi // 4, hi, hq, hkv, page, rng.choice(["fp8", "bf16"]), mix)
    while work(case)["flops"] > 1.9e12:
        case["ctx_lo"], case["ctx_hi"], case["new"] = case["ctx_lo"] // 2, case["ctx_hi"] // 2, case["new"] * 3 // 4
    return case


# --------------------------------------------------------------------------- #
# shapes that follow from a case alone
# --------------------------------------------------------------------------- #


def _contexts(case):
    """Cached tokens of each sequence before its new ones, log-uniform in [ctx_lo, ctx_hi]."""
    r = random.Random(case["mix"])
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    if hi <= lo:
        return [hi] * case["seqs"]
    a = math.log(max(lo, 1))
    return [int(math.exp(r.uniform(a, math.log(hi)))) for _ in range(case["seqs"])]


def _lengths(case):
    """(query tokens, all tokens) of each sequence of an attention case."""
    ctx = _contexts(case)
    if case["kind"] != "prefill":
        n = [case.get("new", 1)] * case["seqs"]
        return n, [max(c, n[0]) for c in ctx]  # the new tokens are the context's last
    r = random.Random(case["mix"] + 1)
    cuts = sorted(r.sample(range(1, case["new"]), case["seqs"] - 1)) if case["seqs"] > 1 else []
    n = [b - a for a, b in zip([0] + cuts, cuts + [case["new"]])]
    return n, [c + k for c, k in zip(ctx, n)]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, shape, scale=1.0, outliers=False):
    x = torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * scale
    if outliers:  # 1 % of the activations 20 times as large
        x = torch.where(torch.rand(shape, generator=g, device=DEV) < 0.01, x * 20.0, x)
    return x


def _fp8_cache(g, layers, pages, page, heads, dtype=torch.float8_e4m3fn):
    """[layers, pages, 2, page, heads, D] of values ~N(0, 1)."""
    cache = torch.empty(layers, pages, 2, page, heads, D, dtype=dtype, device=DEV)
    flat = cache.view(-1)
    step = 1 << 26
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=g, device=DEV).to(dtype)
    return cache


def _tables(g, lens, page, spare=1):
    """A random page table over the lengths (page 0 is never handed out), and the pages of the cache."""
    need = [-(-n // page) for n in lens]
    pages = sum(need) + spare
    perm = (torch.randperm(pages - 1, generator=g, device=DEV) + 1).to(torch.int32)
    table = torch.zeros(len(lens), max(need + [1]), dtype=torch.int32, device=DEV)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    return table, pages


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _cumulative(values):
    out = [0]
    for v in values:
        out.append(out[-1] + v)
    return out


def _slots_of_tail(table, lens, new, page):
    """The slot of each sequence's last ``new[b]`` tokens, sequence by sequence."""
    got = []
    for b, (n, k) in enumerate(zip(lens, new)):
        pos = torch.arange(n - k, n, device=DEV)
        got.append(table[b, pos // page].to(torch.int64) * page + pos % page)
    return torch.cat(got)


# --------------------------------------------------------------------------- #
# prepare
# --------------------------------------------------------------------------- #


def _prepare_append(case, seed):
    g = _gen(seed)
    n, h, page = case["tokens"], case["heads"], case["page"]
    fp8 = case["cache"] == "fp8"
    # every run of tokens sits in whole pages drawn at random, a decode token at a random place of one
    run = case["run"]
    need, runs = -(-run // page), -(-n // run)
    pages = max(case["pages"] * 16 // page, runs * need + 1)
    kv = h * D
    # K and V are column slices of the qkv projection (4 query heads per kv head)
    qkv = torch.empty(n, 6 * kv, dtype=torch.bfloat16, device=DEV)
    qkv[:, :4 * kv] = 0
    qkv[:, 4 * kv:] = _randn(g, (n, 2 * kv), 2.0, outliers=True).to(torch.bfloat16)
    perm = (torch.randperm(pages - 1, generator=g, device=DEV) + 1)[:runs * need].view(runs, need)
    i = torch.arange(n, device=DEV)
    start = torch.randint(0, page, (runs,), generator=g, device=DEV) if run == 1 else torch.zeros(
        runs, dtype=torch.int64, device=DEV)
    pos = i % run + start[i // run]
    slots = perm[i // run, pos // page] * page + pos % page
    cache = _fp8_cache(g, 1, pages, page, h, torch.float8_e4m3fn if fp8 else torch.bfloat16)
    k = qkv[:, 4 * kv:5 * kv].view(n, h, D)
    v = qkv[:, 5 * kv:].view(n, h, D)
    scale = torch.tensor([0.2], dtype=torch.float32, device=DEV) if fp8 else None
    info = KVCacheInfo(kv_cache=(cache[:, :, 0], cache[:, :, 1]), slot_mapping=slots, k_scale=scale, v_scale=scale)
    return {"kind": "append", "k": k, "v": v, "info": info, "cache": cache}


def _prepare_attention(case, seed):
    g = _gen(seed)
    new, lens = _lengths(case)
    hq, hkv, page = case["hq"], case["hkv"], case["page"]
    table, pages = _tables(g, lens, page)
    cache = _fp8_cache(g, 1, pages, page, hkv)[0]
    # logits of standard deviation 2
    q = _randn(g, (sum(new), hq, D), 2.0).to(torch.bfloat16)
    if case["q"] == "fp8":
        q = fp8_kv.quantize(q)
    one = fp8_kv.unit_descale(len(lens), hkv, torch.device(DEV, torch.cuda.current_device()))
    return {"kind": "attention", "q": q, "cache": cache, "max_q": max(new), "cu": _i32(_cumulative(new)),
            "lens": _i32(lens), "table": table, "descale": one}


def _prepare_step(case, seed):
    g = _gen(seed)
    _, lens = _lengths(case)
    b, layers, hq, hkv, page = case["seqs"], case["layers"], case["hq"], case["hkv"], case["page"]
    table, pages = _tables(g, lens, page)
    cache = _fp8_cache(g, layers, pages, page, hkv)
    qkv = _randn(g, (layers, b, (hq + 2 * hkv) * D)).to(torch.bfloat16)
    qkv[:, :, :hq * D] *= 2
    live = KVCacheInfo(page_table=table, slot_mapping=_slots_of_tail(table, lens, [1] * b, page),
                       actual_lens_q=_i32([1] * b), actual_lens_kv=_i32(lens),
                       cu_seqlens_q=_i32(list(range(b + 1))))
    static = cudagraph.initialize_graph_kvcacheinfo(b, table.shape[1], device=DEV)
    static.kv_cache = (cache[:, :, 0], cache[:, :, 1])
    info = cudagraph.slice_kvcache_info(static, b)
    one = fp8_kv.unit_descale(b, hkv, torch.device(DEV, torch.cuda.current_device()))

    def step():
        outs = []
        for layer in range(layers):
            row = qkv[layer]
            q = row[:, :hq * D].view(b, hq, D)
            k = row[:, hq * D:(hq + hkv) * D].view(b, hkv, D)
            v = row[:, (hq + hkv) * D:].view(b, hkv, D)
            impl_utils.append_kv_cache(k, v, info, layer)
            outs.append(attention.flash_attn_varlen_func(
                q, info.kv_cache[0][layer], info.kv_cache[1][layer], 1, info.cu_seqlens_q, None, info.actual_lens_kv,
                info.page_table, softmax_scale=D ** -0.5, causal=True, q_descale=one, k_descale=one, v_descale=one))
        return outs

    cudagraph.set_graph_kvcacheinfo(static, live, b)
    step()  # once outside the capture, as torch asks
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    return {"kind": "step", "graph": graph, "static": static, "live": live, "b": b, "outs": outs, "cache": cache,
            "qkv": qkv}


def _prepare_gather(case, seed):
    g = _gen(seed)
    lens = _contexts(case)
    h, page = case["heads"], case["page"]
    fp8 = case["cache"] == "fp8"
    table, pages = _tables(g, lens, page)
    cache = _fp8_cache(g, 1, pages, page, h, torch.float8_e4m3fn if fp8 else torch.bfloat16)[0]
    out = torch.empty(2, sum(lens), h, D, dtype=torch.bfloat16, device=DEV)
    return {"kind": "gather", "cache": cache, "out": out, "table": table, "cu": _i32(_cumulative(lens)),
            "scale": torch.tensor([0.03125 * 1.3], dtype=torch.float32, device=DEV) if fp8 else None}


def _mla_lengths(case):
    """(new tokens, all tokens) of each sequence: the chunk is split evenly."""
    ctx, n = _contexts(case), case["tokens"]
    new = [n // case["seqs"] + (1 if b < n % case["seqs"] else 0) for b in range(case["seqs"])]
    return new, [c + k for c, k in zip(ctx, new)]


def _prepare_mla(case, seed):
    g = _gen(seed)
    new, lens = _mla_lengths(case)
    page, n = 64, case["tokens"]
    table, pages = _tables(g, lens, page)
    cache = torch.empty(1, pages, page, mla_fp8.entry_bytes(), dtype=torch.uint8, device=DEV)
    e = cache.view(pages * page, -1)
    e[:, :NOPE] = (torch.randn(e.shape[0], NOPE, generator=g, device=DEV) * 120).clamp(-448, 448).to(
        torch.float8_e4m3fn).view(torch.uint8)
    s = torch.exp2(torch.rand(e.shape[0], 4, generator=g, device=DEV) * 4 - 10)
    e[:, NOPE:NOPE + 16] = s.view(torch.uint8)
    e[:, NOPE + 16:] = torch.randn(e.shape[0], ROPE, generator=g, device=DEV).to(torch.bfloat16).view(torch.uint8)
    latent = _randn(g, (n, Q_LORA + NOPE + ROPE)).to(torch.bfloat16)
    kv_c = _randn(g, (n, NOPE), 1.0, outliers=True).to(torch.bfloat16)
    info = KVCacheInfo(mla_cache_tensor=cache, slot_mapping=_slots_of_tail(table, lens, new, page))
    out = torch.empty(sum(lens), NOPE + ROPE, dtype=torch.bfloat16, device=DEV)
    return {"kind": "mla", "kv_c": kv_c, "k_pe": latent[:, Q_LORA + NOPE:], "info": info, "cache": cache, "out": out,
            "table": table, "cu": _i32(_cumulative(lens))}


def _prepare_copy(case, seed):
    g = _gen(seed)
    layers, pages, n = case["layers"], case["pages"], case["pairs"]
    cache = torch.empty(layers, pages, 2, 16, 8, D, dtype=torch.bfloat16, device=DEV)
    flat = cache.view(torch.int32).view(-1)
    flat.random_(generator=g)
    perm = torch.randperm(pages, generator=torch.Generator().manual_seed(seed))
    pairs = torch.stack([perm[:n], perm[n:2 * n]], 1).contiguous()
    return {"kind": "copy", "cache": cache, "pairs": pairs}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _prepare_attention(case, seed)
    return {"append": _prepare_append, "step": _prepare_step, "gather": _prepare_gather, "mla": _prepare_mla,
            "copy": _prepare_copy}[kind](case, seed)


# --------------------------------------------------------------------------- #
# run
# --------------------------------------------------------------------------- #


def run(s):
    kind = s["kind"]
    if kind == "append":
        impl_utils.append_kv_cache(s["k"], s["v"], s["info"], 0)
        return _bytes(s["cache"])
    if kind == "attention":
        one = s["descale"]
        return attention.flash_attn_varlen_func(
            s["q"], s["cache"][:, 0], s["cache"][:, 1], s["max_q"], s["cu"], None, s["lens"], s["table"],
            softmax_scale=D ** -0.5, causal=True, q_descale=one, k_descale=one, v_descale=one)
    if kind == "step":
        cudagraph.set_graph_kvcacheinfo(s["static"], s["live"], s["b"])
        s["graph"].replay()
        return {"out": s["outs"], "cache": _bytes(s["cache"])}
    if kind == "gather":
        cache_ops.gather_cache(s["cache"][:, 0], s["out"][0], s["table"], s["cu"], scale=s["scale"],
                               src_cache_v=s["cache"][:, 1], dst_v=s["out"][1])
        return s["out"]
    if kind == "mla":
        impl_utils.append_mla_kv_cache(s["kv_c"], s["k_pe"], s["info"], 0)
        mla_fp8.gather_mla_fp8_tiles(s["cache"][0], s["out"], s["table"], s["cu"])
        return {"rows": s["out"], "cache": s["cache"]}
    cache_ops.copy_blocks(s["cache"], s["pairs"])
    return _bytes(s["cache"])


def _bytes(cache):
    """The cache's own memory as whole numbers: its values are bit copies or FP8 codes."""
    return cache.view(torch.uint8 if cache.dtype == torch.float8_e4m3fn else torch.int16)


# --------------------------------------------------------------------------- #
# work, tolerance
# --------------------------------------------------------------------------- #


def _visible(new, lens):
    """(query token, key) pairs under the causal mask."""
    return sum(n * (L - n) + n * (n + 1) // 2 for n, L in zip(new, lens))


def _attention_work(case, new, lens):
    hq, hkv = case["hq"], case["hkv"]
    rows = sum(new) * hq * D
    q_bytes = 1 if case.get("q") == "fp8" else 2
    pages = sum(-(-n // case["page"]) for n in lens)
    return {"bytes": sum(lens) * hkv * D * 2 + rows * (q_bytes + 2) + 4 * pages,
            "flops": 4 * D * hq * _visible(new, lens)}


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _attention_work(case, *_lengths(case))
    if kind == "step":
        new, lens = _lengths(case)
        w = _attention_work(case, new, lens)
        append = case["seqs"] * (case["hkv"] * D * 2 * 3 + 8)
        return {k: case["layers"] * (v + (append if k == "bytes" else 0)) for k, v in w.items()}
    if kind == "append":
        row = 2 * case["heads"] * D
        return {"bytes": case["tokens"] * (row * (3 if case["cache"] == "fp8" else 4) + 8), "flops": 0}
    if kind == "gather":
        lens = _contexts(case)
        row = 2 * case["heads"] * D * (3 if case["cache"] == "fp8" else 4)
        return {"bytes": sum(lens) * row + 4 * sum(-(-n // case["page"]) for n in lens), "flops": 0}
    if kind == "mla":
        _, lens = _mla_lengths(case)
        row = 2 * (NOPE + ROPE)
        entry = NOPE + 16 + 2 * ROPE
        return {"bytes": case["tokens"] * (row + entry + 8) + sum(lens) * (entry + row), "flops": 0}
    return {"bytes": case["pairs"] * (case["layers"] * 2 * 65536 + 16), "flops": 0}


def tolerance(case):
    # Attention writes bf16 (2^-9 relative per element); another order of its
    # fp32 sums, or another grid of its probabilities (11 bits or more), moves
    # single elements by one bf16 step (2^-8).  Measured against exact():
    # 1.7e-3; everything else is a bit copy or a defined rounding.
    if case["kind"] in ("decode", "prefill", "step"):
        return {"rel": 4e-3, "max": 0.03}
    return "exact"


# --------------------------------------------------------------------------- #
# exact
# --------------------------------------------------------------------------- #


def _exact_attention(q, kc, vc, table, lens, new):
    """q [T, Hq, D] (FP8, or bf16 rounded to it as the cache's reader takes its
    query), kc and vc [pages, page, Hkv, D]; float64 [T, Hq, D], causal, each
    sequence's query tokens its last positions."""
    if q.dtype != torch.float8_e4m3fn:
        q = q.float().clamp(-448, 448).to(torch.float8_e4m3fn)
    hq, hkv = q.shape[1], kc.shape[2]
    group = hq // hkv
    out = torch.empty(q.shape[0], hq, D, dtype=torch.float64, device=q.device)
    at = 0
    for b, (n, length) in enumerate(zip(new, lens)):
        ids = table[b, :-(-length // kc.shape[1])].long()
        k = kc[ids].flatten(0, 1)[:length]
        v = vc[ids].flatten(0, 1)[:length]
        key = torch.arange(length, device=q.device)
        for h in range(hkv):
            kh, vh = k[:, h].double(), v[:, h].double()
            step = max(1, (1 << 27) // (length * group))
            for i in range(0, n, step):
                m = min(step, n - i)
                x = q[at + i:at + i + m, h * group:(h + 1) * group].double().reshape(m * group, D)
                y = torch.mm(x, kh.t()) * D ** -0.5
                seen = length - n + 1 + i + torch.arange(m, device=q.device)
                y.view(m, group, length).masked_fill_((key[None, :] >= seen[:, None])[:, None, :], -math.inf)
                out[at + i:at + i + m, h * group:(h + 1) * group] = torch.mm(torch.softmax(y, 1), vh).view(m, group, D)
        at += n
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("append", "copy"):
        return None  # bytes: the append's codes and the copies are compared as whole numbers
    s = prepare(case, seed)
    if kind in ("decode", "prefill"):
        new, lens = _lengths(case)
        return _exact_attention(s["q"], s["cache"][:, 0], s["cache"][:, 1], s["table"], lens, new)
    if kind == "step":
        new, lens = _lengths(case)
        hq, hkv, page, b = case["hq"], case["hkv"], case["page"], case["seqs"]
        slots = s["live"].slot_mapping
        outs = []
        for layer in range(case["layers"]):
            row = s["qkv"][layer]
            kv = [s["cache"][layer, :, i].clone() for i in range(2)]
            for i in range(2):
                x = row[:, (hq + i * hkv) * D:(hq + (i + 1) * hkv) * D].view(b, hkv, D)
                x = x.float().clamp(-448, 448).to(torch.float8_e4m3fn)
                kv[i].view(torch.uint8)[slots // page, slots % page] = x.view(torch.uint8)
            outs.append(_exact_attention(row[:, :hq * D].view(b, hq, D), kv[0], kv[1], s["live"].page_table, lens, new))
        return {"out": outs, "cache": None}
    if kind == "gather":
        lens = _contexts(case)
        rows = _rows(s["table"], lens, case["page"])
        scale = 1.0 if s["scale"] is None else s["scale"].double()
        return torch.stack([s["cache"][:, i].reshape(-1, case["heads"], D)[rows].double() * scale for i in range(2)])
    # MLA: quantize the chunk (one float32 scale per 128 elements), then read every entry
    e = s["cache"][0].view(-1, s["cache"].shape[-1]).clone()
    x = s["kv_c"].float().view(-1, 4, 128)
    sc = (x.abs().amax(2) / 448.0).clamp_min(2.0 ** -126)
    codes = (x / sc[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn).view(-1, NOPE).view(torch.uint8)
    slots = s["info"].slot_mapping
    e[slots] = torch.cat([codes, sc.view(torch.uint8), s["k_pe"].contiguous().view(torch.uint8)], 1)
    _, lens = _mla_lengths(case)
    e = e[_rows(s["table"], lens, 64)]
    val = e[:, :NOPE].contiguous().view(torch.float8_e4m3fn).double().view(-1, 4, 128)
    val = (val * e[:, NOPE:NOPE + 16].contiguous().view(torch.float32).double()[:, :, None]).view(-1, NOPE)
    rope = e[:, NOPE + 16:].contiguous().view(torch.bfloat16).double()
    return {"rows": torch.cat([val, rope], 1), "cache": None}


def _rows(table, lens, page):
    """The cache row of every token, sequence by sequence."""
    got = []
    for b, n in enumerate(lens):
        pos = torch.arange(n, device=table.device)
        got.append(table[b, pos // page].long() * page + pos % page)
    return torch.cat(got)
