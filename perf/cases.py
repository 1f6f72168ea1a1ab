"""The measured cases: decoder layers run through the op adapter (`ops`), as a serving program runs them.

A case is one pass over one or more layers, in one of three shapes:

  prefill     packed prompts: norm, stacked QKV projection, rotary embedding, K and V into the paged pool, causal
              attention, output projection, gated FFN
  decode      one new token for each of `batch` sequences whose K and V lie in a paged pool
  primitives  the layer as model code without fused ops writes it: every step a primitive aten op

`calls` says which entry points carry it: "fused" is this backend's own (rotary embedding and silu * mul in the
projections, residuals through addmm, one-pass decode attention), "plain" the ones the reference binds (separate
rotary, silu, mul and add, the two-call decode attention). `weights` is "dense" (the activations' type) or "int8"
(weight-only int8 with a scale for each channel). `launch` is "calls" (one by one) or "graph": recorded once into a
HIP graph and replayed, as a serving loop does with its decode step.

Sequence lengths are drawn from [min_len, max_len] by the case's own `mix`, so that all seeds of a case do the same
work; everything else that a state holds comes from the seed.
"""
import math
import random

import torch

from __graft_entry__ import load_package

pkg = load_package()
ops = pkg.ops

EPS = 1e-5
THETA = 10000.0
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# hidden size, query heads, K/V heads, FFN width
SMALL = (512, 8, 8, 1376)
MEDIUM = (1024, 8, 8, 2816)
BASE = (4096, 32, 32, 11008)
GROUPED = (4096, 32, 8, 14336)
WIDE = (5120, 40, 40, 13824)
LARGE = (8192, 64, 8, 28672)


def _case(path, size, batch, min_len, max_len, dtype, calls="fused", weights="dense", launch="calls", layers=1, mix=0, **more):
    hidden, heads, kv_heads, ffn = size
    return dict(path=path, hidden=hidden, heads=heads, kv_heads=kv_heads, ffn=ffn, batch=batch, min_len=min_len,
                max_len=max_len, dtype=dtype, calls=calls, weights=weights, launch=launch, layers=layers, mix=mix, **more)


def listed():
    return [
        # the block of the fp32 parity configuration: every kernel is a few microseconds, calls and launches are what counts
        _case("prefill", SMALL, 2, 128, 128, "fp32", calls="plain", name="tiny_fp32_2x128"),
        # one user waiting for a token, called op by op: the latency of small batches
        _case("decode", BASE, 1, 1777, 1777, "bf16", name="decode_1_calls"),
        # a small batch on grouped K/V heads through the calls that the reference binds
        _case("decode", GROUPED, 16, 64, 2048, "fp16", calls="plain", mix=1, name="decode_16_plain_fp16"),
        # the throughput end of decoding: 64 sequences of 512 to 4096 tokens, a replayed graph
        _case("decode", BASE, 64, 512, 4096, "bf16", launch="graph", layers=2, mix=2, name="decode_64_graph"),
        # the same on grouped K/V heads, where projections and attention weigh alike
        _case("decode", GROUPED, 48, 512, 4096, "bf16", launch="graph", layers=2, mix=3, name="decode_48_grouped_graph"),
        # int8 weights: decoding for a few users from a model that would be slow to stream in 16 bits
        _case("decode", WIDE, 8, 256, 2048, "bf16", weights="int8", launch="graph", layers=2, mix=4, name="decode_8_int8_graph"),
        # a chat turn: one prompt of a few hundred tokens, the time to the first token
        _case("prefill", BASE, 1, 203, 203, "bf16", name="prefill_1x203"),
        # prompts of very different lengths packed into one batch, through the calls that the reference binds
        _case("prefill", GROUPED, 7, 17, 900, "fp16", calls="plain", mix=5, name="prefill_7_ragged_fp16"),
        # prompts against int8 weights: the weights are read once, the matrix cores do the work
        _case("prefill", WIDE, 3, 100, 500, "bf16", weights="int8", mix=6, name="prefill_3_ragged_int8"),
        # the benchmark's layer: a full batch of prompts
        _case("prefill", BASE, 4, 2048, 2048, "bf16", name="prefill_4x2048"),
        # one long document of an odd length on grouped K/V heads: attention has its largest share here
        _case("prefill", GROUPED, 1, 6001, 6001, "bf16", name="prefill_1x6001_grouped"),
        # a model not rewritten for the fused ops: forty primitive calls with materialised scores
        _case("primitives", BASE, 2, 777, 777, "bf16", calls="plain", name="primitives_2x777"),
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], even over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["tiny", "decode", "decode", "decode", "decode_plain", "decode_int8", "prefill", "prefill", "prefill_plain",
                       "prefill_int8", "primitives"])
    mix = rng.randrange(1 << 20)
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "tiny":
        return _case("prefill", rng.choice([SMALL, MEDIUM]), rng.randint(1, 4), *[_spread(rng, 16, 256)] * 2, "fp32", calls="plain", mix=mix)
    if kind == "primitives":
        size = rng.choice([MEDIUM, BASE])
        return _case("primitives", size, rng.randint(1, 2), *[_spread(rng, 100, 1000)] * 2, half, calls="plain", mix=mix)
    if kind.startswith("decode"):
        int8 = kind == "decode_int8"
        size = rng.choice([MEDIUM, BASE, GROUPED, WIDE, LARGE])
        low = _spread(rng, 32, 2048)
        graph = rng.random() < 0.6
        return _case("decode", size, _spread(rng, 1, 64), low, min(4096, low * rng.randint(1, 8)), half,
                     calls="plain" if kind == "decode_plain" else "fused", weights="int8" if int8 else "dense",
                     launch="graph" if graph else "calls", layers=2 if graph else 1, mix=mix)
    int8 = kind == "prefill_int8"
    size = rng.choice([MEDIUM, BASE, GROUPED, WIDE, LARGE])
    # no more work than the largest listed case: 8192 tokens through BASE
    most = min(8192, int(8192 * 202.4e6 / _weights(*size)))
    batch = rng.randint(1, 8)
    high = _spread(rng, 24, most // batch)
    low = high if rng.random() < 0.3 else max(8, high // rng.randint(2, 16))
    return _case("prefill", size, batch, low, high, half, calls="plain" if kind == "prefill_plain" else "fused",
                 weights="int8" if int8 else "dense", mix=mix)


def _weights(hidden, heads, kv_heads, ffn):
    """Weight elements of a layer."""
    d = hidden // heads
    return hidden * (heads + 2 * kv_heads) * d + hidden * hidden + 3 * hidden * ffn


def _size(case):
    return case["hidden"], case["heads"], case["kv_heads"], case["ffn"]


def _lens(case):
    """Tokens of each sequence (decode: after the new token)."""
    rng = random.Random(case["mix"])
    lens = [rng.randint(case["min_len"], case["max_len"]) for _ in range(case["batch"])]
    return [n + 1 for n in lens] if case["path"] == "decode" else lens


# ------------------------------------------------------------------ what a program holds before the call
def _layer_weights(case, rnd, gen, dev, dt):
    """The weights of one layer as a loader leaves them: q, k and v stacked; for the fused calls the q and k rows in the
    adjacent-pair order and gate and up interleaved (all of them random matrices here)."""
    hidden, heads, kv_heads, ffn = _size(case)
    d = hidden // heads
    shapes = {"wqkv": ((heads + 2 * kv_heads) * d, hidden), "wo": (hidden, hidden), "wdown": (hidden, ffn)}
    if case["path"] == "primitives" or (case["calls"] == "plain" and case["weights"] == "dense"):
        shapes.update(wgate=(ffn, hidden), wup=(ffn, hidden))
    else:
        shapes["wgu"] = (2 * ffn, hidden)
    p = {"norm1": 1 + 0.1 * rnd(hidden), "norm2": 1 + 0.1 * rnd(hidden)}
    for name, (n, k) in shapes.items():
        if case["weights"] == "int8":
            p[name] = torch.randint(-127, 128, (n, k), generator=gen, device=dev, dtype=torch.int8)
            spread = 0.5 + torch.rand(n, generator=gen, device=dev)          # 73: the standard deviation of the int8 values
            p[name + "_scale"] = (spread / (73 * math.sqrt(k))).to(torch.float16)
        else:
            p[name] = rnd(n, k).mul_(1 / math.sqrt(k))
    return p


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    rnd = lambda *shape: torch.randn(*shape, generator=gen, device=dev, dtype=dt)
    hidden, heads, kv_heads, ffn = _size(case)
    d = hidden // heads
    lens = _lens(case)
    batch, total = len(lens), sum(lens)
    decode = case["path"] == "decode"
    rows = batch if decode else total
    s = {"case": case, "x": rnd(rows, hidden), "layers": [_layer_weights(case, rnd, gen, dev, dt) for _ in range(case["layers"])]}
    if case["path"] == "primitives":
        s["x"] = s["x"].view(batch, lens[0], hidden)
        return s
    # rotary tables: by position, one row per token; equal prompts share the rows of one
    cos, sin = pkg.workloads.rotary_tables(d, max(lens), theta=THETA)
    if decode:
        at = torch.tensor(lens) - 1
    elif min(lens) == max(lens):
        at = torch.arange(lens[0])
    else:
        at = torch.cat([torch.arange(n) for n in lens])
    s["cos"], s["sin"] = cos[at].to(dev, dt), sin[at].to(dev, dt)
    # the paged pool: every sequence owns slots scattered over it, an eighth of it is free
    slots = total + total // 8 + 16
    perm = torch.randperm(slots, generator=gen, device=dev).to(torch.int32)[:total]
    starts = [0]
    for n in lens[:-1]:
        starts.append(starts[-1] + n)
    s["b_seq_len"] = torch.tensor(lens, dtype=torch.int32, device=dev)
    s["b_start_loc"] = torch.tensor(starts, dtype=torch.int32, device=dev)
    s["max_len"], s["tokens"] = max(lens), total
    make = rnd if decode else lambda *shape: torch.zeros(*shape, device=dev, dtype=dt)
    s["pools"] = [(make(slots, kv_heads, d), make(slots, kv_heads, d)) for _ in range(case["layers"])]
    if decode:
        owner = torch.repeat_interleave(torch.arange(batch), torch.tensor(lens))
        column = torch.cat([torch.arange(max(lens) - n, max(lens)) for n in lens])      # the table is right-aligned
        s["b_loc"] = torch.zeros(batch, max(lens), dtype=torch.int32, device=dev)
        s["b_loc"][owner.to(dev), column.to(dev)] = perm
        s["dest"] = s["b_loc"][:, -1].contiguous()
    else:
        s["dest"] = perm
    if case["launch"] == "graph":
        _record(s)
    return s


def _record(s):
    """The pass as a HIP graph. Recording may not allocate device memory, so the passes before it fill the cache of the
    recording stream's workspace."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(6):
            before = pkg.runtime.cachingStats()["num_device_malloc"]
            warm = ops.WorkspaceScope()
            with warm:
                _layers(s)
            side.synchronize()
            warm.close()
            if pkg.runtime.cachingStats()["num_device_malloc"] == before:
                break
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"], stream=side):
        s["scope"] = ops.WorkspaceScope()
        with s["scope"]:
            s["out"] = _layers(s)
    torch.cuda.synchronize()


# ------------------------------------------------------------------ the pass
def run(state):
    if state["case"]["path"] == "primitives":
        return _primitives_layer(state, state["x"], state["layers"][0])
    if state["case"]["launch"] == "graph":
        state["graph"].replay()
        return state["out"]
    return _layers(state)


def _layers(s):
    x, new = s["x"], []
    for p, (k_pool, v_pool) in zip(s["layers"], s["pools"]):
        x, k, v = _layer(s, x, p, k_pool, v_pool)
        new.append((k, v))
    return {"hidden": x, "new_kv": new, "pools": s["pools"]}


def _layer(s, x, p, k_pool, v_pool):
    case = s["case"]
    hidden, heads, kv_heads, ffn = _size(case)
    d = hidden // heads
    rows = x.shape[0]
    plain, int8 = case["calls"] == "plain", case["weights"] == "int8"
    if int8:
        linear = lambda t, name: ops.weight_only_int8_linear(t, p[name], p[name + "_scale"])
    else:
        linear = lambda t, name: ops.linear(t, p[name])
    h = ops.rms_norm(x, p["norm1"], EPS)
    if plain or int8:
        qkv = linear(h, "wqkv").view(rows, heads + 2 * kv_heads, d)
        q = ops.rotary_emb(qkv[:, :heads], s["cos"], s["sin"])
        k = ops.rotary_emb(qkv[:, heads:heads + kv_heads], s["cos"], s["sin"])
    else:
        qkv = ops.linear_rotary(h, p["wqkv"], s["cos"], s["sin"], (heads + kv_heads) * d, d).view(rows, heads + 2 * kv_heads, d)
        q, k = qkv[:, :heads], qkv[:, heads:heads + kv_heads]
    v = qkv[:, heads + kv_heads:]
    if plain:
        ops.dest_index_copy_kv(k, s["dest"], k_pool)
        ops.dest_index_copy_kv(v, s["dest"], v_pool)
    else:
        ops.dest_index_copy_kv_pair(k, v, s["dest"], k_pool, v_pool)
    if case["path"] == "prefill":
        att = torch.empty(rows, heads, d, dtype=x.dtype, device=x.device)
        ops.context_attention(q, k, v, s["b_start_loc"], s["b_seq_len"], s["max_len"], out=att)
    else:
        att = torch.empty(rows, heads, d, dtype=x.dtype, device=x.device)
        paged = (s["b_loc"], s["b_start_loc"], s["b_seq_len"], s["max_len"])
        if plain:
            scores = torch.empty(heads, s["tokens"], dtype=torch.float32, device=x.device)
            ops.token_attention(q, k_pool, scores, *paged)
            ops.token_softmax_reducev(scores, v_pool, att, *paged)
        else:
            ops.token_decode_attention(q, k_pool, v_pool, *paged, out=att)
    att = att.view(rows, hidden)
    x1 = ops.add(x, linear(att, "wo")) if plain or int8 else ops.addmm(x, att, p["wo"].t())
    h = ops.rms_norm(x1, p["norm2"], EPS)
    if int8:
        gate_up = linear(h, "wgu")
        return ops.add(x1, linear(ops.silu_mul(gate_up[:, :ffn], gate_up[:, ffn:]), "wdown")), k, v
    if plain:
        act = ops.mul(ops.silu(linear(h, "wgate")), linear(h, "wup"))
        return ops.add(x1, linear(act, "wdown")), k, v
    return ops.addmm(x1, ops.linear_silu_mul(h, p["wgu"]), p["wdown"].t()), k, v


def _primitives_layer(s, x, p):
    case = s["case"]
    b, seq, hidden = x.shape
    heads = case["heads"]
    d = hidden // heads
    dev, dt = x.device, x.dtype

    def rms(t, w):
        return ops.mul(ops.mul(t, ops.rsqrt(ops.add(ops.mean(ops.pow(t, 2), [-1], keepdim=True), EPS))), w)

    def copied(t):
        return ops.copy_(torch.empty(t.shape, dtype=dt, device=dev), t)

    index = ops.arange(0, d, 2, dtype=torch.float32, device=dev)
    inverse = ops.exp(ops.mul(index, -math.log(THETA) / d))
    angle = ops.mul(ops.arange(0, seq, 1, dtype=torch.float32, device=dev)[:, None], inverse[None, :])
    cos, sin = copied(ops.cos(angle))[None, :, None, :], copied(ops.sin(angle))[None, :, None, :]

    def rotated(t):
        a, c = t[..., :d // 2], t[..., d // 2:]
        return ops.cat([ops.sub(ops.mul(a, cos), ops.mul(c, sin)), ops.add(ops.mul(a, sin), ops.mul(c, cos))], dim=-1)

    q, k, v = (t.view(b, seq, heads, d) for t in ops.linear(rms(x, p["norm1"]), p["wqkv"]).split(hidden, dim=-1))
    q, k, v = (copied(t.permute(0, 2, 1, 3)).view(b * heads, seq, d) for t in (rotated(q), rotated(k), v))
    scores = ops.div(ops.bmm(q, copied(k.transpose(1, 2))), math.sqrt(d))
    at = ops.arange(0, seq, 1, dtype=torch.int64, device=dev)
    probs = ops.softmax(ops.masked_fill(scores, ops.gt(at[None, :], at[:, None]), float("-inf")), -1)
    att = copied(ops.bmm(probs, v).view(b, heads, seq, d).permute(0, 2, 1, 3)).view(b, seq, hidden)
    x1 = ops.add(x, ops.linear(att, p["wo"]))
    h = rms(x1, p["norm2"])
    act = ops.mul(ops.silu(ops.linear(h, p["wgate"])), ops.linear(h, p["wup"]))
    return {"hidden": ops.add(x1, ops.linear(act, p["wdown"])), "k": k, "v": v}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    hidden, heads, kv_heads, ffn = _size(case)
    d = hidden // heads
    e = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    lens = _lens(case)
    total = sum(lens)
    rows = len(lens) if case["path"] == "decode" else total
    elements = _weights(*_size(case))
    row = kv_heads * d * e                                                  # a token's K, or its V, in one layer
    if case["weights"] == "int8":
        weight_bytes = elements + 2 * ((heads + 2 * kv_heads) * d + hidden + 2 * ffn + hidden)
    else:
        weight_bytes = elements * e
    flops = 2 * rows * elements
    if case["path"] == "decode":
        # the K and V rows of every cached token and the table of their slots; one query a sequence
        kv_bytes = 2 * total * row + 4 * total
        flops += 4 * total * heads * d
    else:
        # the new K and V rows; every query meets itself and the keys before it
        kv_bytes = 2 * total * row
        flops += sum(2 * n * (n + 1) for n in lens) * heads * d
    layer = weight_bytes + 2 * hidden * e + kv_bytes + (2 * rows * row if case["path"] == "decode" else 0)
    return {"bytes": case["layers"] * layer + 2 * rows * hidden * e, "flops": case["layers"] * flops}


def tolerance(case):
    # Measured against the same pass in float64 without any rounding between the steps, over the listed cases and fourteen
    # drawn ones: bf16 at most 5.3e-3 (2-norm) and 3.0e-2 (largest), fp16 5.7e-4 and 3.8e-3, fp32 5.1e-7 and 3.6e-6. Two
    # passes that round at other places are that far from it each; a larger model or a second layer adds to it.
    return {"bf16": {"rel": 1.2e-2, "max": 1.2e-1}, "fp16": {"rel": 2e-3, "max": 1.5e-2}, "fp32": {"rel": 2e-6, "max": 1.5e-5}}[case["dtype"]]
