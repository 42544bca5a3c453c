"""Performance cases of the attention path: what a serving program has this library do, one attention layer a pass.

Five kinds of pass, through the public Python entry points (zllm_amd.ops), with the cache planes, block tables, rotary
tables, weights and the split workspace that a serving loop keeps prepared beforehand:

  gqa_decode   one new token per sequence over a paged cache (Q8g64 or f16 rows), batches of equal or ragged lengths
  gqa_prefill  a chunk of a prompt: its K/V rows are written into the pages, then it attends to them and to its prefix
  block        packed independent segments (encoders, re-rankers): every row attends to its own segment, nothing cached
  mla_decode   absorbed multi-latent attention of one new token per sequence
  mla_prefill  the same for a chunk of a prompt

K, V and latents are ~N(0, 1) (1 % of the GQA channels eight times larger), quantized by the library's own appends;
pages lie in a random order over a pool a quarter larger than the call needs.
"""
from __future__ import annotations

import math

import torch

from zllm_amd import capi, ops

_DEV = "cuda"
_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_LATENT, _ROPE = 512, 64
_GOLDEN = 0.6180339887498949


def listed():
    return [
        # one chat, a short context, a small model: what a token costs when nothing is large (norm + RoPE + append + attention)
        _gqa_decode(name="gqa_step_4k", batch=1, context=4096, heads=16, kv_heads=4, dim=128, query="f32", append=True),
        # long-context serving batch, the headline workload of bench.py
        _gqa_decode(name="gqa_decode_32k", batch=8, context=32768, heads=64, kv_heads=8, dim=128),
        # the same model serving sequences of unequal lengths
        _gqa_decode(name="gqa_decode_ragged", batch=8, context=32768, heads=64, kv_heads=8, dim=128, ragged=True),
        # many short conversations of a small-head model at once
        _gqa_decode(name="gqa_decode_many", batch=61, context=2048, heads=32, kv_heads=8, dim=64, ragged=True),
        # alternating full and sliding-window layers over f16 rows with a soft cap, one layer of each
        _gqa_decode(name="gqa_decode_f16_window", batch=4, context=8192, heads=16, kv_heads=8, dim=256, cache="f16", window=1024, softcap=50.0),
        # an ordinary prompt, prefilled in one piece
        _gqa_prefill(name="gqa_prefill_prompt", rows=1000, prefix=0, heads=32, kv_heads=8, dim=128),
        # a chunk far into a long document
        _gqa_prefill(name="gqa_prefill_50k", rows=2048, prefix=50000, heads=64, kv_heads=8, dim=128),
        # a chunk of the alternating-layer f16 model, one layer of each
        _gqa_prefill(name="gqa_prefill_f16_window", rows=2048, prefix=6144, heads=16, kv_heads=8, dim=256, cache="f16", window=1024, softcap=50.0),
        # packed segments of unequal lengths
        _case("block", name="block_segments", rows=4100, segments=9, heads=16, kv_heads=16, dim=128),
        # one long chat on one GPU's share of the heads, 8-bit weights, append included
        _mla_decode(name="mla_step_32k", batch=1, context=32768, heads=32, weights=8, append=True),
        # long-context serving batch
        _mla_decode(name="mla_decode_64k", batch=4, context=65536, heads=128),
        # a chunk of a long prompt
        _mla_prefill(name="mla_prefill_16k", rows=512, prefix=16384, heads=128),
    ]


def draw(rng):
    """Another case of the same ranges: sizes over their logarithm, and the options that occur with them."""
    kind = rng.choice(["gqa_decode", "gqa_decode", "gqa_prefill", "gqa_prefill", "block", "mla_decode", "mla_prefill"])
    if kind == "gqa_decode":
        heads, kv_heads, dim, cache = _draw_heads(rng)
        batch = _log_int(rng, 1, 64)
        context = _log_int(rng, 512, 65536)
        most = 550e6 / _row_bytes(cache, kv_heads, dim)
        context = max(256, min(context, int(most / batch)))
        window = 1024 if cache == "f16" and dim == 256 else 0
        return _gqa_decode(batch=batch, context=context, heads=heads, kv_heads=kv_heads, dim=dim, cache=cache, ragged=batch > 1 and rng.random() < 0.6,
                           window=window, softcap=50.0 if window else 0.0, page=rng.choice([16, 16, 32, 64]),
                           query=rng.choice(["bf16", "bf16", "f32"]), append=batch == 1)
    if kind == "gqa_prefill":
        heads, kv_heads, dim, cache = _draw_heads(rng)
        rows = _log_int(rng, 8, 4096)
        prefix = rng.choice([0, _log_int(rng, 200, 50000)])
        most = 1.0e12 / (4.0 * dim * heads)  # (row, key) pairs
        rows = max(8, min(rows, int(most / (prefix + 1)) if prefix else int(math.sqrt(2 * most))))
        window = 1024 if cache == "f16" and dim == 256 else 0
        return _gqa_prefill(rows=rows, prefix=prefix, heads=heads, kv_heads=kv_heads, dim=dim, cache=cache, window=window,
                            softcap=50.0 if window else 0.0, page=rng.choice([16, 16, 32, 64]))
    if kind == "block":
        heads, kv_heads = rng.choice([(16, 16), (16, 4), (32, 8), (16, 8)])
        rows = _log_int(rng, 100, 8000)
        return _case("block", rows=rows, segments=min(max(1, rows // 64), _log_int(rng, 1, 24)), heads=heads, kv_heads=kv_heads, dim=rng.choice([128, 128, 256]))
    heads = rng.choice([16, 32, 64, 128])
    nope, value = rng.choice([(128, 128), (128, 128), (192, 256)])
    weights = rng.choice([16, 16, 8, 4])
    if kind == "mla_decode":
        batch = _log_int(rng, 1, 32)
        context = min(_log_int(rng, 512, 131072), int(2.5e7 / (batch * heads)))
        return _mla_decode(batch=batch, context=context, heads=heads, nope=nope, value=value, weights=weights, ragged=batch > 1 and rng.random() < 0.6,
                           page=rng.choice([16, 64, 64]), append=batch == 1)
    rows = _log_int(rng, 16, 1024)
    prefix = rng.choice([0, _log_int(rng, 200, 32768)])
    rows = max(16, min(rows, int(4e8 / (heads * (prefix + rows)))))
    return _mla_prefill(rows=rows, prefix=prefix, heads=heads, nope=nope, value=value, weights=weights, page=rng.choice([16, 64, 64]))


def prepare(case, seed):
    gen = torch.Generator(device=_DEV)
    gen.manual_seed(seed)
    return {"gqa_decode": _prepare_gqa_decode, "gqa_prefill": _prepare_gqa_prefill, "block": _prepare_block, "mla_decode": _prepare_mla,
            "mla_prefill": _prepare_mla}[case["kind"]](case, gen)


def run(state):
    return state["run"](state)


def work(case):
    """Every input read once and every output written once; multiply-adds of the (row, key) pairs that are visible."""
    kind = case["kind"]
    if kind == "mla_decode" or kind == "mla_prefill":
        heads, latent, rope = case["heads"], _LATENT, _ROPE
        if kind == "mla_decode":
            rows, keys = case["batch"], sum(_lengths(case))
            pairs, out_bytes = keys, 4
        else:
            rows, keys = case["rows"], case["prefix"] + case["rows"]
            pairs, out_bytes = rows * case["prefix"] + rows * (rows + 1) // 2, 2
        weight = heads * (case["nope"] + case["value"]) * latent
        size = keys * (latent + latent // 64 * 2 + rope * 2) + weight * case["weights"] // 8
        size += rows * heads * ((case["nope"] + rope) * 2 + case["value"] * out_bytes)
        return {"bytes": size, "flops": heads * pairs * 2 * (2 * latent + rope) + 2 * rows * weight}
    heads, dim, kv_heads = case["heads"], case["dim"], case["kv_heads"]
    if kind == "block":
        lens, rows = _segment_lengths(case), case["rows"]
        return {"bytes": rows * (2 * heads + 2 * 2 * kv_heads) * dim, "flops": 4 * dim * heads * sum(n * n for n in lens)}
    row_bytes = _row_bytes(case["cache"], kv_heads, dim)
    windows = [0, case["window"]] if case["window"] else [0]
    q_size = 4 if case.get("query") == "f32" else 2
    size = flops = 0
    for window in windows:
        if kind == "gqa_decode":
            keys = pairs = sum(min(n, window) if window else n for n in _lengths(case))
            rows = case["batch"]
        else:
            rows, prefix = case["rows"], case["prefix"]
            keys = min(prefix + rows, window + rows) if window else prefix + rows
            pairs = sum(min(prefix + r + 1, window) for r in range(rows)) if window else rows * prefix + rows * (rows + 1) // 2
        size += keys * row_bytes + rows * heads * dim * (q_size + 4)
        flops += 4 * dim * heads * pairs
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times the distance from the same attention in 64 bits, the largest over the listed and 40 drawn cases:
    decode (probabilities in two terms, 32-bit sums) 2.5e-6 / 3.3e-5; chunks and segments (f16 probabilities) 1.6e-4 /
    5.2e-3; MLA decode (f16 probabilities, bf16 absorbed query) 2.2e-4 / 1.2e-3; MLA chunks, stored as bf16, 1.7e-3 /
    4.4e-3.  Appended codes and scales are whole numbers and stay the same."""
    return {"gqa_decode": {"rel": 1e-5, "max": 1.5e-4}, "gqa_prefill": {"rel": 6e-4, "max": 2e-2}, "block": {"rel": 6e-4, "max": 2e-2},
            "mla_decode": {"rel": 9e-4, "max": 5e-3}, "mla_prefill": {"rel": 6e-3, "max": 2e-2}}[case["kind"]]


# ---- case builders ------------------------------------------------------------------------------------------------------


def _case(kind, **fields):
    return {"kind": kind, **fields}


def _gqa_decode(batch, context, heads, kv_heads, dim, cache="q8", ragged=False, window=0, softcap=0.0, page=16, query="bf16", append=False, **name):
    return _case("gqa_decode", **name, batch=batch, context=context, heads=heads, kv_heads=kv_heads, dim=dim, cache=cache, ragged=ragged, window=window,
                 softcap=softcap, page=page, query=query, append=append)


def _gqa_prefill(rows, prefix, heads, kv_heads, dim, cache="q8", window=0, softcap=0.0, page=16, **name):
    return _case("gqa_prefill", **name, rows=rows, prefix=prefix, heads=heads, kv_heads=kv_heads, dim=dim, cache=cache, window=window, softcap=softcap,
                 page=page)


def _mla_decode(batch, context, heads, nope=128, value=128, weights=16, ragged=False, page=64, append=False, **name):
    return _case("mla_decode", **name, batch=batch, context=context, heads=heads, nope=nope, value=value, weights=weights, ragged=ragged, page=page,
                 append=append)


def _mla_prefill(rows, prefix, heads, nope=128, value=128, weights=16, page=64, **name):
    return _case("mla_prefill", **name, rows=rows, prefix=prefix, heads=heads, nope=nope, value=value, weights=weights, page=page)


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_heads(rng):
    """Query heads, KV heads, head dimension and cache format that are met together."""
    return rng.choice([(64, 8, 128, "q8"), (32, 8, 128, "q8"), (16, 4, 128, "q8"), (24, 8, 128, "q8"), (8, 1, 128, "q8"), (32, 8, 64, "q8"),
                       (16, 2, 256, "q8"), (16, 8, 256, "f16"), (16, 8, 256, "f16"), (32, 8, 128, "f16")])


def _row_bytes(cache, kv_heads, dim):
    return 4 * kv_heads * dim if cache == "f16" else 2 * (kv_heads * dim + kv_heads * dim // 64 * 2)


def _lengths(case):
    """The batch's context lengths: all `context`, or spread evenly over [context / 32, context] in a shuffled order."""
    if not case["ragged"]:
        return [case["context"]] * case["batch"]
    low = case["context"] // 32 + 1
    return [low + int((case["context"] - low) * ((i + 1) * _GOLDEN % 1.0)) for i in range(case["batch"])]


def _segment_lengths(case):
    """`rows` cut into `segments` unequal parts (ratio of the longest to the shortest about three)."""
    weight = [0.5 + (i + 1) * _GOLDEN % 1.0 for i in range(case["segments"])]
    ends = [int(round(case["rows"] * sum(weight[: i + 1]) / sum(weight))) for i in range(case["segments"])]
    return [end - begin for begin, end in zip([0] + ends[:-1], ends)]


# ---- inputs -------------------------------------------------------------------------------------------------------------


def _randn(gen, *shape, dtype=torch.bfloat16):
    return torch.randn(*shape, generator=gen, device=_DEV, dtype=dtype)


def _tables(gen, lengths, page):
    """Block tables [sequences, pages of the longest] and the pool's rows: pages in random order, without replacement."""
    pages = [(n + page - 1) // page for n in lengths]
    pool = sum(pages) + sum(pages) // 4 + 1
    order = torch.randperm(pool, generator=gen, device=_DEV).to(torch.int32)
    tables = torch.zeros(len(lengths), max(pages), dtype=torch.int32, device=_DEV)
    at = 0
    for b, n in enumerate(pages):
        tables[b, :n] = order[at : at + n]
        at += n
    return tables, pool * page


def _channel_gain(gen, cols):
    gain = torch.ones(cols, device=_DEV, dtype=torch.bfloat16)
    gain[torch.randperm(cols, generator=gen, device=_DEV)[: max(1, cols // 100)]] = 8.0
    return gain


def _gqa_planes(case, gen, lengths):
    """K and V planes of the pool with every sequence's rows written: (planes, tables, gains)."""
    cols, page = case["kv_heads"] * case["dim"], case["page"]
    tables, rows = _tables(gen, lengths, page)
    planes, gains = {}, {}
    for name in ("k", "v"):
        gains[name] = _channel_gain(gen, cols)
        if case["cache"] == "f16":
            planes[name] = torch.zeros(rows, cols, dtype=torch.float16, device=_DEV)
        else:
            planes[name] = torch.zeros(rows, cols, dtype=torch.int8, device=_DEV)
            planes[name + "_scales"] = torch.zeros(rows, cols // 64, dtype=torch.int16, device=_DEV)
        for b, length in enumerate(lengths):
            if length == 0:
                continue
            x = _randn(gen, length, cols) * gains[name]
            if case["cache"] == "f16":
                ops.half_append(x, planes[name], tables[b], 0, page)
            else:
                ops.q8g64_append(x, planes[name], planes[name + "_scales"], tables[b], 0, page, capi.QUANT_METAL_GQA)
    return planes, tables, gains


def _rope_tables(rows, dim):
    angle = torch.arange(rows, device=_DEV, dtype=torch.float64)[:, None] / 10000.0 ** (torch.arange(dim // 2, device=_DEV, dtype=torch.float64) * 2 / dim)
    return angle.cos().float(), angle.sin().float()


def _new_rows(case, gen, rows, gains, dtype):
    """Projections of `rows` new tokens, head-norm weights and rotary tables."""
    heads, kv_heads, dim = case["heads"], case["kv_heads"], case["dim"]
    new = {"q": _randn(gen, rows, heads * dim, dtype=dtype)}
    for name in ("k", "v"):
        new[name] = _randn(gen, rows, kv_heads * dim, dtype=dtype) * gains[name].to(dtype)
        new[name + "_norm"] = _randn(gen, dim, dtype=torch.float32) * 0.1
    new["q_norm"] = _randn(gen, dim, dtype=torch.float32) * 0.1
    return new


def _append(s, case, new, position, q_dtype):
    """What precedes the attention call of a layer: the new rows' K and V into the pages, and the query."""
    planes, table, page = s["planes"], s["tables"][0], case["page"]
    if case["cache"] == "f16":
        ops.half_append(new["k"], planes["k"], table, position, page)
        ops.half_append(new["v"], planes["v"], table, position, page)
        return new["q"]
    return ops.gqa_prologue(new["q"], new["k"], new["v"], new["q_norm"], new["k_norm"], s["cos"], s["sin"], planes["k"], planes["k_scales"], planes["v"],
                            planes["v_scales"], table, position, case["heads"], case["kv_heads"], case["dim"], case["dim"], page, q_out_dtype=q_dtype)


def _cache_args(case, planes):
    f16 = case["cache"] == "f16"
    return (planes["k"], planes.get("k_scales"), planes["v"], planes.get("v_scales")), dict(kv_format=capi.KV_F16 if f16 else capi.KV_Q8G64)


# ---- GQA decode ---------------------------------------------------------------------------------------------------------


def _prepare_gqa_decode(case, gen):
    lengths = _lengths(case)
    planes, tables, gains = _gqa_planes(case, gen, lengths)
    dtype = _DTYPES[case["query"]]
    s = {"case": case, "planes": planes, "tables": tables, "run": _run_gqa_decode, "lengths": torch.tensor(lengths, dtype=torch.int32, device=_DEV)}
    s["new"] = _new_rows(case, gen, case["batch"], gains, dtype)
    if case["append"]:
        s["cos"], s["sin"] = _rope_tables(case["context"], case["dim"])
    s["layers"] = [dict(max_kv_len=max(lengths), total_kv_tokens=sum(lengths))]
    if case["window"]:
        seen = [min(n, case["window"]) for n in lengths]
        s["layers"].append(dict(max_kv_len=max(lengths), total_kv_tokens=sum(seen),
                                first_visible=torch.tensor([n - v for n, v in zip(lengths, seen)], dtype=torch.int32, device=_DEV)))
    need = 0
    for layer in s["layers"]:
        args, _, _ = _gqa_decode_call(s, s["new"]["q"], layer, ops.gqa_decode_args, workspace=False)
        need = max(need, capi.load().zllm_attn_gqa_decode_workspace_bytes(args))
    s["workspace"] = torch.empty(need, dtype=torch.uint8, device=_DEV)
    return s


def _gqa_decode_call(s, q, layer, call, workspace):
    case = s["case"]
    planes, how = _cache_args(case, s["planes"])
    return call(q, *planes, s["tables"], s["lengths"], case["heads"], case["kv_heads"], case["dim"], case["page"], case["dim"] ** -0.5,
                softcap=case["softcap"], workspace=workspace, **how, **layer)


def _run_gqa_decode(s):
    case, new = s["case"], s["new"]
    q = _append(s, case, new, case["context"] - 1, _DTYPES[case["query"]]) if case["append"] else new["q"]
    outs = [_gqa_decode_call(s, q, layer, ops.gqa_decode, s["workspace"]) for layer in s["layers"]]
    return {"attention": outs, "cache": s["planes"]} if case["append"] else {"attention": outs}


# ---- GQA prefill --------------------------------------------------------------------------------------------------------


def _prepare_gqa_prefill(case, gen):
    total = case["prefix"] + case["rows"]
    planes, tables, gains = _gqa_planes(case, gen, [total])
    s = {"case": case, "planes": planes, "tables": tables, "run": _run_gqa_prefill, "new": _new_rows(case, gen, case["rows"], gains, torch.bfloat16)}
    s["cos"], s["sin"] = _rope_tables(total, case["dim"])
    return s


def _run_gqa_prefill(s):
    case = s["case"]
    q = _append(s, case, s["new"], case["prefix"], torch.bfloat16)
    planes, how = _cache_args(case, s["planes"])
    outs = [ops.gqa_prefill_chunk(q, *planes, s["tables"][0], case["prefix"], case["heads"], case["kv_heads"], case["dim"], case["page"],
                                  case["dim"] ** -0.5, window=window, softcap=case["softcap"], **how)
            for window in ([0, case["window"]] if case["window"] else [0])]
    return {"attention": outs, "cache": s["planes"]}


# ---- packed segments ----------------------------------------------------------------------------------------------------


def _prepare_block(case, gen):
    rows, cols = case["rows"], case["kv_heads"] * case["dim"]
    lens = torch.tensor(_segment_lengths(case), device=_DEV)
    ends = torch.cumsum(lens, 0)
    padded = (rows + 63) // 64 * 64
    return {"case": case, "run": _run_block, "q": _randn(gen, rows, case["heads"] * case["dim"]), "k": _randn(gen, rows, cols), "v": _randn(gen, rows, cols),
            "k_plane": torch.zeros(padded, cols, dtype=torch.float16, device=_DEV), "v_plane": torch.zeros(padded, cols, dtype=torch.float16, device=_DEV),
            "table": torch.arange(padded // 64, dtype=torch.int32, device=_DEV),
            "starts": torch.repeat_interleave(ends - lens, lens).to(torch.int32), "ends": torch.repeat_interleave(ends, lens).to(torch.int32)}


def _run_block(s):
    case = s["case"]
    ops.half_append(s["k"], s["k_plane"], s["table"], 0, 64)
    ops.half_append(s["v"], s["v_plane"], s["table"], 0, 64)
    return ops.gqa_prefill_chunk(s["q"], s["k_plane"], None, s["v_plane"], None, s["table"], 0, case["heads"], case["kv_heads"], case["dim"], 64,
                                 case["dim"] ** -0.5, kv_format=capi.KV_F16, visible_starts=s["starts"], visible_ends=s["ends"])


# ---- MLA ----------------------------------------------------------------------------------------------------------------


def _quantized(weight, bits, group):
    """kv_b as packed codes, low bits first, and a bf16 scale per row and `group` columns."""
    top, half = (127, 128) if bits == 8 else (7, 8)
    w = weight.view(weight.shape[0], -1, group)
    scale = (w.abs().amax(dim=2) / top).to(torch.bfloat16)
    codes = ((w / scale.float()[:, :, None]).round().clamp(-top, top) + half).to(torch.int64).view(weight.shape[0], -1, 32 // bits)
    words = (codes << (torch.arange(32 // bits, device=_DEV) * bits)).sum(dim=2)
    return torch.where(words >= 2**31, words - 2**32, words).to(torch.int32), scale


def _prepare_mla(case, gen):
    chunk = case["kind"] == "mla_prefill"
    lengths = [case["prefix"] + case["rows"]] if chunk else _lengths(case)
    rows, heads, page = (case["rows"] if chunk else case["batch"]), case["heads"], case["page"]
    tables, pool = _tables(gen, lengths, page)
    s = {"case": case, "run": _run_mla, "tables": tables, "lengths": torch.tensor(lengths, dtype=torch.int32, device=_DEV), "longest": max(lengths),
         "total": sum(lengths), "codes": torch.zeros(pool, _LATENT, dtype=torch.int8, device=_DEV),
         "scales": torch.zeros(pool, _LATENT // 64, dtype=torch.int16, device=_DEV), "rope": torch.zeros(pool, _ROPE, dtype=torch.int16, device=_DEV)}
    for b, length in enumerate(lengths):
        ops.mla_append(_randn(gen, length, _LATENT, dtype=torch.float32), _randn(gen, length, _ROPE, dtype=torch.float32), s["codes"], s["scales"],
                       s["rope"], tables[b], 0, page)
    s["appends"] = case["rows"] if chunk else int(case["append"])
    if s["appends"]:
        s["latent"], s["k_rope"] = (_randn(gen, s["appends"], n, dtype=torch.float32) for n in (_LATENT, _ROPE))
        s["cos"], s["sin"] = _rope_tables(max(lengths), _ROPE)
    weight = _randn(gen, heads * (case["nope"] + case["value"]), _LATENT, dtype=torch.float32) / _LATENT**0.5
    if case["weights"] == 16:
        s["kv_b"], s["form"] = weight.to(torch.bfloat16), {}
    else:
        s["kv_b"], scale = _quantized(weight, case["weights"], 128)
        s["form"] = dict(kv_b_bits=case["weights"], kv_b_scales=scale, kv_b_group=128, kv_b_scale_dtype=capi.SCALE_BF16)
    s["q"] = _randn(gen, rows, heads * (case["nope"] + _ROPE))
    s["out"] = torch.empty(rows, heads * case["value"], dtype=torch.bfloat16 if chunk else torch.float32, device=_DEV)
    args, _, s["workspace"] = _mla_call(s, ops.mla_decode_args, None)
    return s


def _mla_call(s, call, workspace):
    case = s["case"]
    return call(s["q"], s["kv_b"], s["codes"], s["scales"], s["rope"], s["tables"], s["lengths"], case["heads"], case["nope"] + _ROPE,
                case["nope"] + case["value"], _LATENT, _ROPE, case["page"], s["longest"], out_dtype=s["out"].dtype, out=s["out"], workspace=workspace,
                query_rows=case["rows"] if case["kind"] == "mla_prefill" else 1, total_ctx_tokens=s["total"], **s["form"])


def _run_mla(s):
    case = s["case"]
    if s["appends"]:
        position = s["longest"] - s["appends"]
        ops.mla_append(s["latent"], s["k_rope"], s["codes"], s["scales"], s["rope"], s["tables"][0], position, case["page"], cos=s["cos"], sin=s["sin"],
                       rotary_dim=_ROPE, rope_position=position)
    out = _mla_call(s, ops.mla_decode, s["workspace"])
    return {"attention": out, "cache": [s["codes"], s["scales"], s["rope"]]} if s["appends"] else {"attention": out}
