"""The measured workloads of the HQMQ KV-cache path: what a serving loop or an evaluation script calls, over the sizes
this repository's configurations name.

A case is a dict of plain values:
  kind    decode   one new token per sequence attends over the packed cache (one layer of a decode step)
          step     append of that token's K and V, then the same attention (a whole decode step of one layer)
          append   a prompt's K and V quantized into the packed cache
          chunk    Tq prompt tokens attend, causally, over a packed cache of T tokens that ends with them
          fake     quantize_K and quantize_V of the cache hook of the evaluation scripts (same shape and type out)
          encode   the unpacked integer codes of K and V
          fused    fused_attention on unpacked codes (Tq == T: causal prefill, Tq == 1: decode)
          dense    decode_dequant: unpacked codes to a dense K
  B, Hq, Hkv, d, T, Tq   sequences, query heads, KV heads, head size, tokens per sequence, query tokens
  S, bits                secondary codebook size and radius bits
  dtype                  float16, bfloat16 or float32
  med3x                  outlier extraction (C = 3) with the verbatim sideband
  ragged                 sequences of different lengths (T / 16 .. T), started longest first
  data                   normal: N(0, 1); channels: a lognormal(0, 0.5) scale per channel; spikes: 2 % of the K chunks
                         scaled by 50 - 200 (with d = 64: 1 % of the K and V chunks scaled by 100)
"""
import torch

import hqmq
from hqmq import kernels
from hqmq_amd import ops

DEV = "cuda:0"
NEW_TOKENS = 64           # a step case generates this many tokens, then rolls back to the prompt for the next continuation
SHAPES = ((32, 8, 128), (28, 4, 128), (64, 8, 64))             # (query heads, KV heads, head size)
BOOKS = ((24, 3), (96, 4), (192, 6), (192, 4))                 # (secondary size, radius bits)


def _case(name, kind, B, shape, T, book, dtype, Tq=1, med3x=False, ragged=False, data="normal"):
    Hq, Hkv, d = shape
    c = dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, d=d, T=T, Tq=Tq, S=book[0], bits=book[1], dtype=dtype, med3x=med3x, ragged=ragged, data=data)
    return dict(c, name=name) if name else c


def listed():
    llama, qwen25, oss = SHAPES
    s24, s96, s192, s192r4 = BOOKS
    return [
        # a chat's first answers: a few hundred tokens in the cache, launches and host work count
        _case("decode_300", "decode", 1, llama, 300, s96, "float16"),
        # long-context decode of one user
        _case("decode_32k", "decode", 1, llama, 32768, s96, "float16"),
        # batched long-context decode with outlier-heavy keys
        _case("decode_b8_32k_spikes", "decode", 8, qwen25, 32768, s192, "float16", med3x=True, data="spikes"),
        # very long contexts, small heads
        _case("decode_b4_131k_d64", "decode", 4, oss, 131072, s96, "bfloat16", med3x=True, data="spikes"),
        # the whole decode step of a layer, one user
        _case("step_4k", "step", 1, llama, 4096, s96, "float16"),
        # the whole decode step of a layer, a server's ragged batch
        _case("step_b64_ragged", "step", 64, llama, 16384, s24, "bfloat16", med3x=True, ragged=True, data="channels"),
        # a long prompt into the cache
        _case("append_32k", "append", 1, llama, 32768, s96, "float16"),
        # a batch of ordinary prompts, of no round length, with outlier extraction, into recycled cache slots
        _case("append_b4_4001", "append", 4, llama, 4001, s24, "bfloat16", med3x=True, data="channels"),
        # the evaluation scripts' cache hook on one layer's prompt
        _case("fake_2048", "fake", 1, llama, 2048, s192, "float16", med3x=True, data="channels"),
        # one chunk of a chunked prefill deep in a long prompt
        _case("chunk_1024_of_32k", "chunk", 1, llama, 32768, s96, "float16", Tq=1024),
        # the drop-in kernel call on unpacked codes, square causal prefill
        _case("fused_2048", "fused", 1, llama, 2048, s192r4, "float16", Tq=2048),
        # dense decode of unpacked codes
        _case("dense_4096", "dense", 1, llama, 4096, s192, "float16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(("decode", "decode", "step", "append", "chunk", "fake", "encode", "fused", "dense"))
    shape = rng.choice(SHAPES)
    Hq, Hkv, d = shape
    book = rng.choice(BOOKS)
    dtype = rng.choice(("float16", "bfloat16"))
    data = rng.choice(("normal", "channels", "spikes"))
    med3x = rng.random() < 0.5
    B = _log_int(rng, 1, 64)
    row = Hkv * d
    if kind in ("decode", "step"):
        T = _log_int(rng, 100, min(131072, 250_000_000 // (B * row)))
        return _case(None, kind, B, shape, T, book, dtype, med3x=med3x, ragged=B > 1 and rng.random() < 0.5, data=data)
    if kind in ("append", "fake", "encode", "dense"):
        if kind in ("fake", "encode") and rng.random() < 0.25:
            dtype = "float32"
        most = 4_000_000 if dtype == "float32" else 16_000_000
        B = min(B, 16)
        T = _log_int(rng, 16, max(17, most // (B * row)))
        return _case(None, kind, B, shape, T, book, dtype, med3x=med3x and kind != "dense", data=data)
    B = min(B, 8)
    if kind == "fused":
        Tq = T = _log_int(rng, 64, 2048 // B)
        if rng.random() < 0.3:
            Tq = 1
        return _case(None, kind, B, shape, T, book, dtype, Tq=Tq, data=data)
    T = _log_int(rng, 200, 32768 // B)
    Tq = _log_int(rng, 8, max(9, min(T, 1024, 7_000_000 // (B * T))))
    return _case(None, kind, B, shape, T, book, dtype, Tq=Tq, med3x=med3x, data=data)


def _values(case, which, g, tokens):
    """K (which = 0) or V (which = 1) activations of `tokens` tokens, on the GPU."""
    dt = getattr(torch, case["dtype"])
    B, H, d = case["B"], case["Hkv"], case["d"]
    x = torch.randn(B, H, tokens, d, generator=g, device=DEV, dtype=dt)
    if case["data"] == "channels":
        x *= torch.exp(0.5 * torch.randn(H, 1, d, generator=g, device=DEV)).to(dt)
    elif case["data"] == "spikes" and (which == 0 or d == 64):
        share, lo, hi = (0.01, 100.0, 100.0) if d == 64 else (0.02, 50.0, 200.0)
        hit = torch.rand(B, H, tokens, d // 4, 1, generator=g, device=DEV) < share
        gain = lo + (hi - lo) * torch.rand(B, H, tokens, d // 4, 1, generator=g, device=DEV)
        x.view(B, H, tokens, d // 4, 4).mul_(torch.where(hit, gain, torch.ones_like(gain)).to(dt))
    return x


def prepare(case, seed):
    kind, B, Hq, Hkv, d, T, Tq = (case[k] for k in ("kind", "B", "Hq", "Hkv", "d", "T", "Tq"))
    dt = getattr(torch, case["dtype"])
    g = torch.Generator(device=DEV).manual_seed(seed)
    q = hqmq.HQMQ(n_layers=1, n_heads=Hkv, secondary_size=case["S"], radius_bits=case["bits"], device=DEV)
    w = hqmq.with_outlier_extraction(q, C=3.0) if case["med3x"] else q
    s = {"kind": kind, "w": w}
    k, v = _values(case, 0, g, T), _values(case, 1, g, T)
    if kind in ("decode", "step", "chunk", "fused"):
        s["Q"] = torch.randn(B, Hq, Tq, d, generator=g, device=DEV, dtype=dt)
    if kind in ("fake", "encode"):
        # a model in use has called its quantizer before: the codebooks of the layer are there
        for call in (q.quantize_K, q.quantize_V):
            call(k[:, :, :1], 0)
        return dict(s, k=k, v=v)
    if kind in ("fused", "dense"):
        r_qmax = (1 << case["bits"]) - 1
        ck = q.encode_K(k, 0)
        if kind == "dense":
            return dict(s, args=(ck["idx"], ck["rq"], ck["r_max"], ck["joint"], r_qmax))
        cv = q.encode_V(v, 0)
        args = (s.pop("Q"), ck["idx"], ck["rq"], ck["r_max"], ck["joint"], cv["idx"], cv["rq"], cv["r_max"], cv["joint"], r_qmax)
        return dict(s, args=args, causal=Tq > 1)
    cache = w.new_cache(B, T + (NEW_TOKENS if kind == "step" else 0), d, dt, 0)
    s["cache"] = cache
    planes = ("main", "aux", "scale", "flags", "sideband", "sb_coord", "sb_tile_off", "sb_count")
    s["planes"] = {"%s.%s" % (n, p): getattr(t, p) for n, t in (("K", cache.K), ("V", cache.V)) for p in planes}
    if kind == "append":
        return dict(s, k=k, v=v)
    w.append(cache, k, v, 0)
    del k, v
    s["lens"] = s["order"] = None
    if case["ragged"]:
        lens = torch.randint(max(1, T // 16), T + 1, (B,), generator=g, device=DEV, dtype=torch.int32)
        lens[0] = T
        cache.crop_(lens)
        s["lens"], s["order"] = lens, ops.longest_first(lens)
    if kind == "chunk":
        s["offset"] = T - Tq
    if kind == "step":
        s.update(k=_values(case, 0, g, NEW_TOKENS), v=_values(case, 1, g, NEW_TOKENS), done=0, prompt=T)
        if case["ragged"]:
            s["pos"] = s["lens"].clone()
    return s


def run(s):
    kind = s["kind"]
    if kind == "decode":
        if s["lens"] is None:
            return hqmq.fused_attention_packed(s["Q"], s["cache"])
        return hqmq.fused_attention_packed(s["Q"], s["cache"], kv_lens=s["lens"], batch_order=s["order"])
    if kind == "step":
        w, cache, i = s["w"], s["cache"], s["done"]
        if i == NEW_TOKENS:                 # the next continuation of the same prompts
            i = 0
            if s["lens"] is None:
                cache.crop_(s["prompt"])
            else:
                cache.crop_(s["lens"])
                s["pos"].copy_(s["lens"])
        s["done"] = i + 1
        k, v = s["k"][:, :, i:i + 1], s["v"][:, :, i:i + 1]
        if s["lens"] is None:
            w.append(cache, k, v, 0)
            return {"O": hqmq.fused_attention_packed(s["Q"], cache), **s["planes"]}
        w.append(cache, k, v, 0, pos=s["pos"])
        s["pos"].add_(1)
        return {"O": hqmq.fused_attention_packed(s["Q"], cache, kv_lens=s["pos"], batch_order=s["order"]), **s["planes"]}
    if kind == "append":
        s["cache"].crop_(0)                 # the slot's last request is gone
        s["w"].append(s["cache"], s["k"], s["v"], 0)
        return s["planes"]
    if kind == "chunk":
        return hqmq.fused_attention_packed(s["Q"], s["cache"], causal=True, causal_offset=s["offset"])
    if kind == "fake":
        return s["w"].quantize_K(s["k"], 0), s["w"].quantize_V(s["v"], 0)
    if kind == "encode":
        return s["w"].encode_K(s["k"], 0), s["w"].encode_V(s["v"], 0)
    if kind == "fused":
        return hqmq.fused_attention(*s["args"], causal=s["causal"])
    return kernels.decode_dequant(*s["args"])


def work(case):
    """Bytes: every input read once and every output written once (packed rows at their stored width, sideband entries
    left out: a few per cent of the chunks).  Flops: the two products of attention; quantizing has none that it could
    not do without."""
    kind, B, Hq, Hkv, d, T, Tq, S, bits = (case[k] for k in ("kind", "B", "Hq", "Hkv", "d", "T", "Tq", "S", "bits"))
    e = 4 if case["dtype"] == "float32" else 2
    n = d // 4
    tokens = B * T * ((1 + 1 / 16) / 2 if case["ragged"] else 1)
    code_bits = (24 * S - 1).bit_length() + bits
    row = n * code_bits / 8 + e + (n / 8 if case["med3x"] else 0)
    tables = 2 * Hkv * 24 * S * 4 * e
    dense, unpacked = d * e, 8 * n + e
    qo = 2 * B * Hq * Tq * d * e
    pairs = B * Hq * (Tq * T - (Tq * (Tq - 1) // 2 if Tq > 1 else 0)) * (tokens / (B * T))
    attn = {"bytes": 2 * tokens * Hkv * row + qo + tables, "flops": 4 * d * pairs}
    if kind in ("decode", "chunk"):
        return attn
    if kind == "step":
        return {"bytes": attn["bytes"] + 2 * B * Hkv * (dense + row), "flops": attn["flops"]}
    if kind == "fused":
        return {"bytes": 2 * tokens * Hkv * unpacked + qo + tables, "flops": attn["flops"]}
    both = 2 * tokens * Hkv
    if kind == "append":
        return {"bytes": both * (dense + row), "flops": 0}
    if kind == "fake":
        return {"bytes": both * 2 * dense, "flops": 0}
    if kind == "encode":
        return {"bytes": both * (dense + unpacked + (n if case["med3x"] else 0)), "flops": 0}
    return {"bytes": tokens * Hkv * (unpacked + dense) + tables // 2, "flops": 0}


def tolerance(case):
    # codes, masks, packed bytes and decoded values are defined to the bit; attention outputs are rounded to 16 bits and
    # their sums run in another order from one split of the work to the next
    if case["kind"] in ("append", "fake", "encode", "dense"):
        return "exact"
    return {"rel": 1e-2 if case["dtype"] == "bfloat16" else 2e-3}
