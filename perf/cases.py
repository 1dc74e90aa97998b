"""Timing cases of the library: what a serving program has it do, over the range of sizes it is used at.

Three kinds of case, each through the public entry points:

  decode    one attention step of a batch over packed caches: `fwd_kvcache_int`, or a `DecodePlan` that the program
            keeps ("entry": call / plan)
  pack      quantize-pack of prompt K/V, or of one full window per sequence behind what is packed already:
            `kvcache_pack_int`
  generate  one request batch from its prompt to its last token with `BitKVCache`: ragged prefill, then a token per
            pass, either with `step` (one launch) or with `append` + `decode`

Inputs are N(0,1) with three of 128 K channels ten times as large (outlier channels), as in bench.py.
"""
from __future__ import annotations

import math
import random

import torch

from bitladder_amd import BitKVCache, fwd_kvcache_int, kvcache_pack_int, plan_fwd_kvcache_int

D = 128                 # head dimension
BLOCK = 128             # tokens per packed block
SCALE = 1.0 / math.sqrt(D)


# ------------------------------------------------------------------------------------------------ the cases
def _decode(name, b, h, hk, tokens, window, bits, gs, *, dtype="fp16", mode="k-channel", entry="plan", rows=1,
            ragged=False, page=0):
    """tokens: packed tokens per sequence (the longest one's, if ragged); window: fp16 tokens behind them; rows: query
    rows per sequence; page: tokens per page of a paged cache, 0 = contiguous."""
    c = dict(kind="decode", b=b, h=h, hk=hk, tokens=tokens, window=window, bits=bits, gs=gs, dtype=dtype, mode=mode,
             entry=entry, rows=rows, ragged=ragged, page=page)
    return c if name is None else dict(c, name=name)


def _pack(name, b, hk, tokens, bits, gs, *, dtype="fp16", mode="k-channel", held=0):
    """held: tokens of every sequence that are packed already; the new ones go behind them, by device-side offsets."""
    c = dict(kind="pack", b=b, hk=hk, tokens=tokens, bits=bits, gs=gs, dtype=dtype, mode=mode, held=held)
    return c if name is None else dict(c, name=name)


def _generate(name, b, h, hk, lo, hi, steps, bits, gs, *, dtype="fp16", mode="k-channel", loop="step"):
    """Prompts of lo to hi tokens, then `steps` tokens per sequence."""
    c = dict(kind="generate", b=b, h=h, hk=hk, lo=lo, hi=hi, steps=steps, bits=bits, gs=gs, dtype=dtype, mode=mode,
             loop=loop)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a short chat turn of one user: nothing but latency
        _decode("decode-1k", 1, 32, 8, 1024, 37, 4, 128, entry="call"),
        # one user, 4K context, one kv head per query head
        _decode("decode-4k-mha", 1, 32, 32, 4096, 128, 4, 128, entry="call"),
        # one user, long document, grouped heads: the benchmark's default shape
        _decode("decode-32k", 1, 32, 8, 32768, 128, 4, 128),
        # one user, very long context, 2-bit codes in small groups
        _decode("decode-128k-2bit", 1, 32, 8, 131072, 128, 2, 64),
        # eight long sequences of a model with eight query heads per kv head, bf16
        _decode("decode-64k-b8-2bit", 8, 64, 8, 65536, 128, 2, 128, dtype="bf16"),
        # a batch of unequal sequences, lengths on the device
        _decode("decode-ragged-b16", 16, 32, 8, 7936, 128, 4, 128, ragged=True),
        # a batch that is no power of two, paged cache, the smallest groups
        _decode("decode-paged-b6", 6, 32, 8, 10112, 77, 4, 32, dtype="bf16", page=256, entry="call"),
        # eight query rows per sequence at once (verification of drafted tokens)
        _decode("decode-rows", 2, 32, 8, 8192, 64, 4, 128, entry="call", rows=8),
        # prompt of one long document
        _pack("pack-32k", 1, 8, 32768, 4, 128),
        # full windows of 16 sequences move behind what is packed
        _pack("pack-block-b16", 16, 8, 128, 4, 128, held=3968),
        # small request batch, one launch per token
        _generate("generate-step", 4, 32, 8, 700, 2000, 16, 4, 128),
        # larger ragged request batch, append and decode as two calls
        _generate("generate-append", 8, 32, 8, 1024, 8192, 8, 4, 128, loop="append"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(("decode",) * 6 + ("pack",) * 2 + ("generate",) * 2)
    mode = "k-tensor" if rng.random() < 0.15 else "k-channel"
    bits = 4 if mode == "k-tensor" else rng.choice((4, 4, 2))
    gs = rng.choice((32, 64, 128, 128))
    dtype = rng.choice(("fp16", "fp16", "bf16"))
    hk = rng.choice((1, 2, 4, 8, 8, 8, 16, 32))
    g = rng.choice([x for x in (1, 2, 4, 4, 8) if hk * x <= 64])
    per_token = hk * D * 2 * (bits / 8 + 4 / gs)        # packed bytes of a token
    if kind == "decode":
        while True:
            b = _log_int(rng, 1, 32)
            tokens = BLOCK * _log_int(rng, 2, 1024)
            if b * tokens * per_token < 280e6:
                break
        rows = rng.randint(2, 8) if rng.random() < 0.15 else 1
        return _decode(None, b, g * hk, hk, tokens, rng.randint(0, 128), bits, gs, dtype=dtype, mode=mode, rows=rows,
                       entry="call" if rows > 1 else rng.choice(("call", "plan")),
                       ragged=b > 1 and rows == 1 and rng.random() < 0.4, page=rng.choice((0, 0, 0, 256)))
    if kind == "pack":
        while True:
            b = _log_int(rng, 1, 32)
            tokens = BLOCK * _log_int(rng, 1, 256)
            if b * tokens * hk * D * 4 < 280e6:
                break
        return _pack(None, b, hk, tokens, bits, gs, dtype=dtype, mode=mode, held=BLOCK * rng.choice((0, 0, 1, 7)))
    while True:
        b = rng.randint(1, 8)
        lo = _log_int(rng, 100, 4000)
        hi = lo + _log_int(rng, 1, 4000)
        if b * hi * hk * D * 4 < 200e6:
            break
    return _generate(None, b, g * hk, hk, lo, hi, rng.randint(4, 16), bits, gs, dtype=dtype, mode=mode,
                     loop=rng.choice(("step", "append")))


# ------------------------------------------------------------------------------------------------ inputs
def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float16


def _kv(case, g, tokens):
    """K and V [b, tokens, hk, 128] of the prompt."""
    shape = (case["b"], tokens, case["hk"], D)
    k = torch.randn(shape, generator=g, device="cuda", dtype=_dtype(case))
    v = torch.randn(shape, generator=g, device="cuda", dtype=_dtype(case))
    for head in range(case["hk"]):
        k[:, :, head, torch.randperm(D, generator=g, device="cuda")[:3]] *= 10.0
    return k, v


def _cache(case, pages, tokens):
    """Packed tensors of `pages` sequences (or pages) of `tokens` tokens, as the caller allocates them."""
    hk, bits, gs = case["hk"], case["bits"], case["gs"]
    pn = 16 // bits
    v_params = torch.zeros((pages, D // gs, hk, tokens), dtype=torch.float32, device="cuda")
    k_params = torch.zeros_like(v_params) if case["mode"] == "k-tensor" else \
        torch.zeros((pages, tokens // gs, hk, D), dtype=torch.float32, device="cuda")
    return (torch.zeros((pages, tokens // pn, hk, D), dtype=torch.uint16, device="cuda"), k_params,
            torch.zeros((pages, tokens, hk, D // pn), dtype=torch.uint16, device="cuda"), v_params)


def _lengths(case, lo, hi, shuffle=None):
    """Sequence lengths from lo to hi, the same ones for every seed; `shuffle` deals them out."""
    r = random.Random(case["b"] * 1000003 + hi)
    n = [r.randint(lo, hi) for _ in range(case["b"])]
    if shuffle is not None:
        random.Random(shuffle).shuffle(n)
    return n


def _decode_lengths(case, shuffle=None):
    """(packed, window) tokens of every sequence: an eighth of the longest up to the longest, if ragged."""
    if not case["ragged"]:
        return [case["tokens"]] * case["b"], [case["window"]] * case["b"]
    blocks = _lengths(case, max(1, case["tokens"] // BLOCK // 8), case["tokens"] // BLOCK, shuffle)
    w = case["window"]
    return [BLOCK * n for n in blocks], [w - (7 * n) % (w + 1) for n in blocks]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return {"decode": _prepare_decode, "pack": _prepare_pack, "generate": _prepare_generate}[case["kind"]](case, seed, g)


def _prepare_decode(case, seed, g):
    b, tokens, page = case["b"], case["tokens"], case["page"]
    q = torch.randn((b, case["rows"], case["h"], D), generator=g, device="cuda", dtype=_dtype(case))
    k, v = _kv(case, g, tokens + case["window"])
    table = None
    if page:
        per_seq = -(-tokens // page)
        table = torch.randperm(b * per_seq, generator=g, device="cuda").to(torch.int32).reshape(b, per_seq)
        cache = _cache(case, b * per_seq, page)
    else:
        cache = _cache(case, b, tokens)
    kvcache_pack_int(k[:, :tokens], cache[0], cache[1], v[:, :tokens], cache[2], cache[3], table, None, tokens,
                     case["mode"], case["gs"], case["bits"])
    options = {}
    if page and not case["ragged"]:
        options["seqlen_k"] = tokens
    if case["window"]:
        options.update(k_residual=k[:, tokens:].contiguous(), v_residual=v[:, tokens:].contiguous())
    if case["ragged"]:
        packed, window = _decode_lengths(case, seed)
        options.update(seqlens_k=torch.tensor(packed, dtype=torch.int32, device="cuda"), max_seqlen_k=max(packed))
        if case["window"]:
            options.update(residual_len=torch.tensor(window, dtype=torch.int32, device="cuda"),
                           max_residual_len=max(window))
    args = (q, *cache, table, SCALE, case["mode"], case["gs"], case["bits"])
    if case["entry"] == "plan":
        return {"run": "plan", "plan": plan_fwd_kvcache_int(*args, **options)}
    return {"run": "decode", "args": args, "options": options}


def _prepare_pack(case, seed, g):
    k, v = _kv(case, g, case["tokens"])
    cache = _cache(case, case["b"], case["held"] + case["tokens"])
    options = {}
    if case["held"]:
        options["dst_offsets"] = torch.full((case["b"],), case["held"], dtype=torch.int32, device="cuda")
    return {"run": "pack", "args": (k, cache[0], cache[1], v, cache[2], cache[3], None, None, case["tokens"],
                                    case["mode"], case["gs"], case["bits"]), "options": options,
            "out": [t.view(torch.int16) for t in cache]}


def _prepare_generate(case, seed, g):
    b, hk, steps = case["b"], case["hk"], case["steps"]
    lengths = _lengths(case, case["lo"], case["hi"])
    k, v = _kv(case, g, case["hi"])
    new = [[torch.randn((b, 1, n, D), generator=g, device="cuda", dtype=_dtype(case)) for n in (case["h"], hk, hk)]
           for _ in range(steps)]
    cache = BitKVCache(b, hk, case["hi"] + steps, num_bits=case["bits"], group_size=case["gs"], dtype=_dtype(case),
                       quant_mode=case["mode"])
    # what the cache holds at the end: of every sequence the packed blocks (a region per sequence and head, block
    # after block) and the live rows of its window
    blocks = cache.capacity // BLOCK
    held = []
    packed = [t.view(torch.int16).reshape(b, hk, blocks, -1) for t in (cache.k_pack, cache.k_params, cache.v_pack,
                                                                       cache.v_params)]
    for i, n in enumerate(n + steps for n in lengths):
        held += [t[i, :, :n // BLOCK] for t in packed]
        held += [t[i, :n % BLOCK] for t in (cache.k_res, cache.v_res)]
    return {"run": "generate", "cache": cache, "k": k, "v": v, "lengths": lengths, "new": new, "loop": case["loop"],
            "held": held + [cache.total]}


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    if state["run"] == "plan":
        return state["plan"].run()
    if state["run"] == "decode":
        return fwd_kvcache_int(*state["args"], **state["options"])
    if state["run"] == "pack":
        kvcache_pack_int(*state["args"], **state["options"])
        return state["out"]
    cache = state["cache"]
    cache.prefill(state["k"], state["v"], state["lengths"])
    outs = []
    for q, k_new, v_new in state["new"]:
        if state["loop"] == "step":
            outs.append(cache.step(q, k_new, v_new, SCALE))
        else:
            cache.append(k_new, v_new)
            outs.append(cache.decode(q, SCALE))
    return {"out": torch.cat(outs, 1), "held": state["held"]}


# ------------------------------------------------------------------------------------------------ work, tolerance
def _token_bytes(case):
    """(fp16, packed) bytes of one token's K and V."""
    return case["hk"] * D * 4, case["hk"] * D * 2 * (case["bits"] / 8 + 4 / case["gs"])


def work(case):
    wide, packed = _token_bytes(case)
    b = case["b"]
    if case["kind"] == "decode":
        in_cache, in_window = (sum(x) for x in _decode_lengths(case))
        rows = b * case["rows"] * case["h"]
        return {"bytes": in_cache * packed + in_window * wide + rows * D * 4,
                "flops": 4 * D * case["rows"] * case["h"] * (in_cache + in_window)}
    if case["kind"] == "pack":
        return {"bytes": b * case["tokens"] * (wide + packed), "flops": 0}
    total, flops = 0.0, 0.0
    for n in _lengths(case, case["lo"], case["hi"]):
        total += n // BLOCK * BLOCK * (wide + packed) + n % BLOCK * 2 * wide
        for t in range(n, n + case["steps"]):       # read what is held, take the new token, write the output
            total += t // BLOCK * BLOCK * packed + t % BLOCK * wide + 2 * wide + case["h"] * D * 4
            total += BLOCK * (wide + packed) if t % BLOCK == BLOCK - 1 else 0
            flops += 4 * D * case["h"] * (t + 1)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Packed bytes are the same for everybody.  An attention output differs from dequantize-then-attend in 64 bits by
    what its rounding adds (fp16 2.1e-4 of its norm, bf16 1.7e-3) and by the splits and the fp16 probabilities: measured
    over these sizes 3e-4 to 5e-4 of the norm in fp16 (1.1e-3 where one wave works through many thousand 2-bit tokens)
    and 1.7e-3 in bf16, at worst 3e-3 and 6e-3 of a single value.  Four times that."""
    if case["kind"] == "pack":
        return "exact"
    return {"rel": 7e-3, "max": 2.5e-2} if case["dtype"] == "bf16" else {"rel": 2e-3, "max": 1.2e-2}
