"""Performance cases of the compressed-KV path: what a program that keeps its KV cache in DartKV pages
has the framework do, through the public entry points.

Four kinds of work:

* ``decode``: attention of one query token (or a few, as in speculative decoding) over a packed cache;
* ``generate``: a new prompt is packed, then tokens are appended one at a time, each followed by its
  attention call (one layer of a generation loop, the first decode after a prefill included);
* ``materialize``: the cache read back as dense K and V (the attention backends that do not read packed
  pages), from a kept cache or right after the prompt is packed (``update``);
* ``quantize``: the tensor-level API, quantize along tokens (keys) and along channels (values), and back.

Keys are N(0, 1) with a sixteenth of the channels of each KV head scaled by 10, values N(0, 1), queries
N(0, 1): the distribution the quantizer's channel promotion is made for.
"""

import math

import torch

import dartkv_amd as dart

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
PAGE = 128

# One sequence and layer of the usual cache: 2-bit pages of 128 tokens, a quarter of the key channels
# promoted to 4 bits, 32 full-precision sink tokens, the newest partial page held dense.
DART = dict(bits=2, promote=0.25, kgroup=128, vgroup=64, sink=32, held=True)


def _case(name, kind, B, H, G, T, D, dtype, **over):
    case = dict(name=name, kind=kind, B=B, H=H, G=G, T=T, D=D, dtype=dtype, Q=1, steps=0, **DART)
    case.update(over)
    return case


def listed():
    return [
        # a single interactive sequence: one layer's attention for one token, launch and latency bound
        _case("decode_single", "decode", 1, 8, 4, 1024, 128, "bf16"),
        # long-context serving at full batch: the bandwidth case
        _case("decode_long_batch", "decode", 64, 8, 4, 32768, 128, "bf16"),
        # the 4-bit uniform cache (no promotion), a large ordinary batch, eight query heads per KV head
        _case("decode_uniform4", "decode", 16, 8, 8, 16384, 128, "bf16", bits=4, promote=0.0),
        # the configuration's own default groups (64 tokens, 64 channels) in fp16
        _case("decode_group64", "decode", 8, 8, 4, 4096, 128, "fp16", promote=0.0, kgroup=64, sink=0),
        # a model whose heads do not split into a power of two per KV head, ragged prompt length
        _case("decode_gqa6", "decode", 8, 8, 6, 8011, 128, "bf16"),
        # a small model's heads: 64 channels
        _case("decode_head64", "decode", 16, 8, 4, 4000, 64, "bf16"),
        # speculative decoding: four query tokens per head over one cache
        _case("decode_tokens4", "decode", 8, 8, 4, 8192, 128, "bf16", Q=4),
        # a batch of long prompts packed, then the first token of each
        _case("prefill_long", "generate", 8, 8, 4, 16384, 128, "bf16", steps=1),
        # a short chat turn: a ragged prompt, then 64 tokens across a page boundary, default groups
        _case("generate_short", "generate", 1, 8, 4, 1000, 128, "fp16", promote=0.0, kgroup=64, sink=0, steps=64),
        # the smallest prompt, full precision source, packed and read back at once
        _case("update_small", "materialize", 1, 8, 1, 256, 128, "fp32", promote=0.0, kgroup=32, vgroup=32, sink=2,
              held=False, fresh=True),
        # the dense read-back of a kept cache that an attention backend without packed pages does every step
        _case("materialize", "materialize", 8, 8, 1, 4096, 128, "bf16", fresh=False),
        # the tensor-level API: keys along tokens, values along channels, and both back
        _case("quantize_tensors", "quantize", 4, 8, 1, 4096, 128, "bf16", bits=4, promote=0.0, kgroup=64, sink=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges, sizes spread over their logarithm."""
    kind = rng.choice(["decode", "decode", "decode", "generate", "materialize", "quantize"])
    D = rng.choice([64, 128, 128])
    H = rng.choice([2, 4, 8])
    G = rng.randint(1, 8)
    dtype = rng.choice(["bf16", "fp16"])
    promote = rng.choice([0.0, 0.125, 0.25, 0.25, 0.5])
    bits = 2 if promote else rng.choice([2, 4, 8])
    kgroup = rng.choice([64, 128, 128])
    vgroup = rng.choice([32, 64, 64])
    sink = rng.choice([0, 32, 32])
    if kind == "decode":
        T = _log_int(rng, 200, 32768)
        top = max(1, min(64, (1 << 28) // (H * T * D)))
        c = _case("", kind, _log_int(rng, 1, top), H, G, T, D, dtype, Q=rng.choice([1, 1, 1, 2, 4]))
    elif kind == "generate":
        T = _log_int(rng, 200, 16384)
        top = max(1, min(8, (1 << 27) // (H * T * D)))
        c = _case("", kind, _log_int(rng, 1, top), H, G, T, D, dtype, steps=rng.choice([1, 16, 64]))
    elif kind == "materialize":
        T = _log_int(rng, 256, 8192)
        top = max(1, min(8, (1 << 25) // (H * T * D)))
        c = _case("", kind, _log_int(rng, 1, top), H, 1, T, D, rng.choice(["bf16", "fp16", "fp32"]),
                  held=rng.random() < 0.5, fresh=rng.random() < 0.5)
        kgroup = rng.choice([32, 64, 128])
    else:
        T = _log_int(rng, 128, 8192)
        top = max(1, min(8, (1 << 25) // (H * T * D)))
        c = _case("", kind, _log_int(rng, 1, top), H, 1, T, D, rng.choice(["bf16", "fp16", "fp32"]))
        promote, bits, sink = 0.0, rng.choice([2, 4, 8]), 0
    c.update(bits=bits, promote=promote, kgroup=kgroup, vgroup=vgroup, sink=sink)
    del c["name"]
    return c


def _config(case):
    return dart.DartKVCacheConfig(bits=case["bits"], page_size=PAGE, key_group_size=case["kgroup"],
                                  value_group_size=case["vgroup"], sink_tokens=case["sink"],
                                  hold_partial_pages=case["held"], promote_ratio=case["promote"],
                                  metadata_dtype=torch.float16)


def _inputs(case, seed):
    """K and V [B, H, T + steps, D] and the queries [max(steps, 1)] x [B, H * G, Q, D], from the seed."""
    B, H, D, dtype = case["B"], case["H"], case["D"], DTYPES[case["dtype"]]
    T = case["T"] + case["steps"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    keys = torch.randn(B, H, T, D, generator=gen, dtype=dtype, device="cuda")
    values = torch.randn(B, H, T, D, generator=gen, dtype=dtype, device="cuda")
    host = torch.Generator().manual_seed(seed + 1)
    factor = torch.ones(H, D)
    for h in range(H):
        factor[h, torch.randperm(D, generator=host)[: D // 16]] = 10.0
    keys.mul_(factor.to(device="cuda", dtype=dtype).view(1, H, 1, D))
    queries = torch.randn(max(case["steps"], 1), B, H * case["G"], case["Q"], D, generator=gen, dtype=dtype,
                          device="cuda")
    return keys, values, queries


def prepare(case, seed):
    keys, values, queries = _inputs(case, seed)
    state = {"kind": case["kind"], "config": _config(case)}
    if case["kind"] == "decode" or (case["kind"] == "materialize" and not case["fresh"]):
        cache = dart.DartKVCache(state["config"])
        cache.append(keys, values)
        state.update(cache=cache, query=queries[0])
    elif case["kind"] == "generate":
        T, steps = case["T"], case["steps"]
        state.update(keys=keys[:, :, :T].contiguous(), values=values[:, :, :T].contiguous(),
                     new=[(keys[:, :, T + i:T + i + 1].contiguous(), values[:, :, T + i:T + i + 1].contiguous(),
                           queries[i]) for i in range(steps)])
    else:
        state.update(keys=keys, values=values, bits=case["bits"], kgroup=case["kgroup"], vgroup=case["vgroup"],
                     cache=None)
    return state


def run(state):
    kind = state["kind"]
    if kind == "decode":
        return dart.fused_dart_attention(state["query"], state["cache"])
    if kind == "generate":
        cache = dart.DartKVCache(state["config"])
        cache.append(state["keys"], state["values"])
        outs = []
        for key, value, query in state["new"]:
            cache.append(key, value)
            outs.append(dart.fused_dart_attention(query, cache))
        return outs
    if kind == "materialize":
        if state["cache"] is not None:
            return state["cache"].get()
        return dart.DartKVCache(state["config"]).update(state["keys"], state["values"])
    bits = state["bits"]
    k = dart.quantize(state["keys"], bits=bits, group_size=state["kgroup"], metadata_dtype=torch.float16, axis=-2)
    v = dart.quantize(state["values"], bits=bits, group_size=state["vgroup"], metadata_dtype=torch.float16)
    return [k.values, k.scale, k.zero_point, v.values, v.scale, v.zero_point, k.dequantize(), v.dequantize()]


# ---- what a pass cannot do without ----

def _split(case, tokens):
    """(sink, packed, held) tokens of a cache that has seen ``tokens`` tokens."""
    sink = min(case["sink"], tokens)
    rest = tokens - sink
    packed = rest // PAGE * PAGE if case["held"] else rest
    return sink, packed, rest - packed


def _packed_bytes(case, tokens):
    """Bytes of a cache of ``tokens`` tokens: packed pages, their fp16 metadata, dense sink and tail."""
    B, H, D = case["B"], case["H"], case["D"]
    sink, packed, held = _split(case, tokens)
    esize = DTYPES[case["dtype"]].itemsize
    pages = packed / PAGE
    kgroups = -(-PAGE // case["kgroup"])
    K = int(D * case["promote"] + 1e-6)
    key = D * PAGE * case["bits"] / 8 + K * PAGE * 2 / 8 + 4 * K + 4 * D * kgroups
    value = PAGE * (D * case["bits"] / 8 + 4 * -(-D // case["vgroup"]))
    return B * H * (pages * (key + value) + (sink + held) * 2 * D * esize)


def work(case):
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    esize = DTYPES[case["dtype"]].itemsize
    heads = B * H * case["G"] * case["Q"]
    qo = 2 * heads * D * esize
    dense = 2 * B * H * T * D * esize
    kind = case["kind"]
    if kind == "decode":
        return {"bytes": _packed_bytes(case, T) + qo, "flops": 4 * heads * T * D}
    if kind == "generate":
        total = dense + _packed_bytes(case, T)
        flops = 4 * B * H * T * D
        for i in range(case["steps"]):
            total += _packed_bytes(case, T + i + 1) + qo
            flops += 4 * heads * (T + i + 1) * D
        return {"bytes": total, "flops": flops}
    if kind == "materialize":
        packed = _packed_bytes(case, T)
        return {"bytes": (2 * packed + 2 * dense if case["fresh"] else packed + dense), "flops": 4 * B * H * T * D}
    packed = 2 * B * H * T * D * case["bits"] / 8 + 4 * B * H * (D * -(-T // case["kgroup"]) + T * -(-D // case["vgroup"]))
    return {"bytes": dense + 2 * packed + dense, "flops": 8 * B * H * T * D}


def tolerance(case):
    if case["kind"] in ("materialize", "quantize"):
        return "exact"
    # 16-bit outputs: one rounding of the result over attention sums whose weights may be 16-bit (1e-4);
    # against the 64-bit result that is 1.7e-3 for bf16 and 2.1e-4 to 2.6e-4 for fp16
    return {"rel": 7e-3} if case["dtype"] == "bf16" else {"rel": 1e-3}


# ---- the same in plain torch: the quantizer's chain in the source dtype, attention in 64 bits ----

def _range_scale(mn, mx, qmax):
    eps = torch.tensor(1e-6 if mn.dtype == torch.float32 else 1e-4, dtype=mn.dtype, device=mn.device)
    return torch.maximum(mx - mn, eps) / qmax


def _requantized(x, qmax):
    """x [..., group, n] quantized along dim -2 in its own dtype and back through fp16 metadata: (values,
    scale, zero point).  ``qmax`` broadcasts against x's group minimum [..., 1, n]."""
    mn, mx = x.amin(dim=-2, keepdim=True), x.amax(dim=-2, keepdim=True)
    qmax = qmax.to(x.dtype).expand(mn.shape)
    scale = _range_scale(mn, mx, qmax)
    code = torch.minimum(((x - mn) / scale).round().clamp_min(0), qmax)
    scale16, zero16 = scale.to(torch.float16), mn.to(torch.float16)
    out = (code.to(torch.float16) * scale16 + zero16).to(x.dtype)
    return out, scale16, zero16


def _grouped(x, group):
    """[..., T, n] -> [..., G, group, n], the last group filled with copies of the last row."""
    short = -x.shape[-2] % group
    if short:
        x = torch.cat((x, x[..., -1:, :].expand(*x.shape[:-2], short, x.shape[-1])), dim=-2)
    return x.unflatten(-2, (-1, group))


def _token_means(x):
    """Mean of |x| over dim -2 of [..., n, D], in fp32, summed as CPU reductions sum it (runs of 16, then
    the runs in order, the remainder first), rounded to the source dtype."""
    n = x.shape[-2]
    a = x.abs().float()
    total = torch.zeros_like(a[..., 0, :])
    for start in range(0, n // 16 * 16, 16):
        run = torch.zeros_like(total)
        for i in range(start, start + 16):
            run = run + a[..., i, :]
        total = total + run
    rest = torch.zeros_like(total)
    for i in range(n // 16 * 16, n):
        rest = rest + a[..., i, :]
    return ((rest + total) / torch.full_like(total, float(n))).to(x.dtype)


def _key_pages(x, case):
    """Key pages [..., n, D] through the quantizer: one group run per ``kgroup`` tokens, promoted channels
    in 4 bits."""
    D, n = x.shape[-1], x.shape[-2]
    K = int(D * case["promote"] + 1e-6)
    qmax = torch.full((*x.shape[:-2], 1, 1, D), float(2 ** case["bits"] - 1), device=x.device)
    if K:
        score = _token_means(x).float().cpu()
        top = torch.topk(score, K, dim=-1, largest=True, sorted=True).indices.to(x.device)
        qmax.view(*x.shape[:-2], D).scatter_(-1, top, 15.0)
    return _requantized(_grouped(x, case["kgroup"]), qmax)[0].flatten(-3, -2)[..., :n, :]


def _value_rows(x, group, bits):
    T, D = x.shape[-2:]
    g = _grouped(x.transpose(-1, -2).contiguous(), group)
    qmax = torch.full((1, 1), float(2 ** bits - 1), device=x.device)
    out, scale, zero = _requantized(g, qmax)
    return (out.flatten(-3, -2)[..., :D, :].transpose(-1, -2).contiguous(),
            scale.squeeze(-2).transpose(-1, -2), zero.squeeze(-2).transpose(-1, -2))


def _cached(k, v, case, tokens):
    """What a cache that was given k, v [H, tokens, D] of one sequence holds, dequantized."""
    sink, packed, _ = _split(case, tokens)
    k, v = k.clone(), v.clone()
    full = packed // PAGE * PAGE
    for start, count, n in ((sink, full // PAGE, PAGE), (sink + full, 1, packed - full)):
        if count and n:
            rows = slice(start, start + count * n)
            k[:, rows] = _key_pages(k[:, rows].unflatten(1, (count, n)), case).flatten(1, 2)
    if packed:
        rows = slice(sink, sink + packed)
        v[:, rows] = _value_rows(v[:, rows], case["vgroup"], case["bits"])[0]
    return k, v


def _attention(q, k, v):
    """q [H * G, Q, D] over k, v [H, T, D] in 64 bits, every query token to every cached token."""
    H, _, D = k.shape
    q = q.double().view(H, -1, D)
    weights = torch.softmax(torch.matmul(q, k.double().transpose(-1, -2).contiguous()) / math.sqrt(D), dim=-1)
    return torch.matmul(weights, v.double())


def exact(case, seed):
    keys, values, queries = _inputs(case, seed)
    kind, B = case["kind"], case["B"]
    if kind == "decode":
        outs = [_attention(queries[0, b], *_cached(keys[b], values[b], case, case["T"])) for b in range(B)]
        return torch.stack(outs).view(queries[0].shape)
    if kind == "generate":
        outs = [torch.empty(queries[0].shape, dtype=torch.float64, device="cuda") for _ in range(case["steps"])]
        for b in range(B):
            total = case["T"] + case["steps"]
            k, v = _cached(keys[b], values[b], case, total)
            for i in range(case["steps"]):
                seen = case["T"] + i + 1
                sink, packed, _ = _split(case, seen)
                ki, vi = k[:, :seen].clone(), v[:, :seen].clone()
                ki[:, sink + packed:], vi[:, sink + packed:] = (t[b, :, sink + packed:seen] for t in (keys, values))
                outs[i][b] = _attention(queries[i, b], ki, vi).view(outs[i][b].shape)
        return outs
    if kind == "materialize":
        pairs = [_cached(keys[b], values[b], case, case["T"]) for b in range(B)]
        return tuple(torch.stack(t).double() for t in zip(*pairs))
    # quantize: packed codes have no value of their own
    qmax = torch.full((1, 1, 1), float(2 ** case["bits"] - 1), device="cuda")
    k, kscale, kzero = _requantized(_grouped(keys, case["kgroup"]), qmax)
    v, vscale, vzero = _value_rows(values, case["vgroup"], case["bits"])
    kscale, kzero = (t.squeeze(-2).transpose(-1, -2) for t in (kscale, kzero))
    return [None, kscale.double(), kzero.double(), None, vscale.double(), vzero.double(),
            k.flatten(-3, -2)[:, :, :case["T"]].double(), v.double()]
