"""The work that a program built on this library has it do, as cases that can be timed and compared.

The sizes are those of the model the kernels are written for: 10 full-attention layers (16 q heads, 2 kv heads,
head dim 256, rotary dims 64, theta 1e7) and 30 Gated DeltaNet layers (16 key heads, 32 value heads of 128, conv
kernel 4), caches that hold halves or 8/4-bit codes, prompts taken in chunks of up to 4096 tokens.  A case names
one kind of work:

  token      one generated token (rows 1) or one verify step of drafted tokens (rows 2..8) in the attention layers:
             per layer, the norms, RoPE and the store of the new keys and values, then attention over the cache
  prefill    a chunk of a prompt in one attention layer: its keys and values appended to the cache, then causal
             attention over what the cache holds
  gemm       the same chunk through AttGemm, the route with the scores in blocks of keys
  deltanet   one generated token (rows 1) or a verify step (rows 2..8, with the states after every row kept, so
             that rejected rows can be undone) in the Gated DeltaNet layers
  chunk      a chunk of a prompt in one Gated DeltaNet layer: the conv, the delta rule and the gated norm
"""
import importlib
import math

import torch

saetta = importlib.import_module("saetta-macqwen_amd")

HEADS, KV_HEADS, DIM = 16, 2, 256
VALUES = KV_HEADS * DIM
ROPE_DIMS, ROPE_THETA, EPS = 64, 1e7, 1e-6
ATTENTION_LAYERS, DELTANET_LAYERS = 10, 30
K_HEADS, V_HEADS, K_DIM, V_DIM, CONV = 16, 32, 128, 128, 4
CHANNELS = 2 * K_HEADS * K_DIM + V_HEADS * V_DIM
CHUNK = 4096        # tokens of a prompt taken at a time
LONGEST = 262144    # tokens of the longest context
CACHE_START = 8192  # a cache starts here and doubles when it is full
MOST_PAIRS = 2048 * (118784 + 2049 / 2)  # (query, key) pairs of the largest listed case
OUTLIERS = [7, 101, 230, 333, 460]       # 1 % of the key and value channels are larger, as in real layers
KINDS = {16: saetta.KvBits.Half, 8: saetta.KvBits.Eight, 4: saetta.KvBits.Four}


def listed():
    return [
        # one layer, a short context in halves, launched call by call: nothing but latency and launches
        {"name": "token-half-4k-eager", "kind": "token", "bits": 16, "rows": 1, "context": 4096, "capacity": 8192,
         "layers": 1, "graph": False},
        # the headline: a generated token at 32k tokens over 8-bit codes, all attention layers
        {"name": "token-8bit-32k", "kind": "token", "bits": 8, "rows": 1, "context": 32768, "capacity": 32896,
         "layers": 10, "graph": True},
        # a long conversation over 4-bit codes, in a cache that has grown by doubling
        {"name": "token-4bit-150k", "kind": "token", "bits": 4, "rows": 1, "context": 150000, "capacity": 262144,
         "layers": 10, "graph": True},
        # two drafted tokens and the one before them, at 32k tokens
        {"name": "verify3-8bit-32k", "kind": "token", "bits": 8, "rows": 3, "context": 32768, "capacity": 32896,
         "layers": 10, "graph": True},
        # a longer draft over a half cache, an odd length
        {"name": "verify6-half-57k", "kind": "token", "bits": 16, "rows": 6, "context": 57123, "capacity": 65536,
         "layers": 10, "graph": True},
        # the DeltaNet layers' part of a generated token, and of a verify step
        {"name": "deltanet-token", "kind": "deltanet", "rows": 1, "layers": 30, "graph": True},
        {"name": "deltanet-verify4", "kind": "deltanet", "rows": 4, "layers": 30, "graph": True},
        # a full chunk of a prompt in a DeltaNet layer
        {"name": "deltanet-chunk-4096", "kind": "chunk", "tokens": 4096},
        # a short first prompt over halves
        {"name": "prefill-half-166", "kind": "prefill", "bits": 16, "tokens": 166, "pos": 0},
        # the headline chunk: 4096 tokens behind 4096, 8-bit codes
        {"name": "prefill-8bit-4096-at-4k", "kind": "prefill", "bits": 8, "tokens": 4096, "pos": 4096},
        # the next turn of a long conversation over 4-bit codes, an odd number of tokens
        {"name": "prefill-4bit-1237-at-60k", "kind": "prefill", "bits": 4, "tokens": 1237, "pos": 60007},
        # the matrix-product route near the end of a long prompt, in chunks of 2048
        {"name": "gemm-half-2048-at-116k", "kind": "gemm", "bits": 16, "tokens": 2048, "pos": 118784},
    ]


def _between(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["token", "token", "token", "verify", "verify", "deltanet", "chunk", "prefill", "prefill", "prefill",
                       "gemm"])
    if kind in ("token", "verify"):
        bits = rng.choice([16, 8, 4])
        rows = 1 if kind == "token" else rng.randint(2, 8)
        context = _between(rng, 16, LONGEST - 8)
        capacity = CACHE_START
        while capacity < context + rows:
            capacity *= 2
        if rng.random() < 0.5:  # a cache made for a known length instead of one that has grown
            capacity = -(-(context + rows) // 128) * 128
        graph = rng.random() < 0.8
        return {"kind": "token", "bits": bits, "rows": rows, "context": context, "capacity": capacity,
                "layers": ATTENTION_LAYERS if graph or rng.random() < 0.5 else 1, "graph": graph}
    if kind == "deltanet":  # the layers of a part of the model, to all of them
        return {"kind": "deltanet", "rows": rng.randint(1, 8), "layers": rng.randint(8, DELTANET_LAYERS),
                "graph": rng.random() < 0.8}
    if kind == "chunk":
        return {"kind": "chunk", "tokens": _between(rng, 16, CHUNK - 1)}
    tokens = _between(rng, 7 if kind == "prefill" else 64, CHUNK)
    most = int(min(LONGEST / 2 - tokens, MOST_PAIRS / tokens - tokens / 2))
    pos = 0 if rng.random() < 0.2 else _between(rng, 16, most)
    return {"kind": kind, "bits": rng.choice([16, 8, 4]), "tokens": tokens, "pos": pos}


class _Maker:
    """Tensors of a seed, made on the GPU."""

    def __init__(self, seed):
        self.generator = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        return torch.randn(*shape, generator=self.generator, device="cuda") * scale

    def kv(self, tokens):
        x = self.normal(tokens, VALUES)
        x[:, OUTLIERS] *= 8.0
        return x

    def fill(self, cache, tokens):
        """Keys and values of `tokens` tokens into a cache."""
        for start in range(0, tokens, 8192):
            n = min(8192, tokens - start)
            for half, rows in zip((cache.keys, cache.values), cache.quant or (None, None)):
                x = self.kv(n).view(-1)
                if rows is None:
                    half[start * VALUES:(start + n) * VALUES] = x.to(torch.float16)
                else:
                    rows.encode(x, start, n)


def _new_rows(cache, start, n):
    """The rows start .. start + n of every buffer of a cache."""
    return [b[start * (b.numel() // cache.capacity):(start + n) * (b.numel() // cache.capacity)] for b in cache.buffers()]


def _prepare_token(case, make):
    layers, rows, context, bits = case["layers"], case["rows"], case["context"], case["bits"]
    qg = make.normal(layers, rows, HEADS, 2 * DIM)
    k, v = make.kv(layers * rows).view(layers, rows, VALUES), make.kv(layers * rows).view(layers, rows, VALUES)
    norms = 1.0 + make.normal(layers, 2, DIM, scale=0.1)
    q = torch.zeros(layers, rows, HEADS, DIM, device="cuda")
    out = torch.zeros(layers, rows, HEADS, DIM, device="cuda")
    params = saetta.PrepParams(HEADS, KV_HEADS, DIM, ROPE_DIMS, ROPE_THETA, EPS)
    caches = [saetta.GpuKvCache.with_bits(HEADS, KV_HEADS, DIM, case["capacity"], KINDS[bits]) for _ in range(layers)]
    capacity = caches[0].capacity
    verify = saetta.AttentionRows(HEADS, KV_HEADS, capacity, rows) if rows > 1 else None
    plan = saetta.Plan()
    for i, cache in enumerate(caches):
        make.fill(cache, context)
        keys, values = cache.quant or (cache.keys, cache.values)
        saetta.record_store(plan, qg[i], k[i], v[i], norms[i, 0], norms[i, 1], q[i], keys, values, params, capacity, rows=rows)
        if verify is None:
            record = cache.decode.record if bits == 16 else cache.decode.record_quant
            record(plan, q[i], keys, values, qg[i], out[i])
        else:
            record = verify.record if bits == 16 else verify.record_quant
            record(plan, rows, q[i], keys, values, qg[i], out[i], [plan.params] * rows)
    plan.set_params(saetta.TokenParams(0, context))
    outputs = {"out": out, "q": q, "new": [_new_rows(c, context, rows) for c in caches]}
    return {"plan": plan, "built": plan.build(graph=case["graph"]), "params": saetta.TokenParams(0, context),
            "outputs": outputs, "keep": caches}


def _prepare_prefill(case, make):
    tokens, pos, bits = case["tokens"], case["pos"], case["bits"]
    cache = saetta.GpuKvCache.with_bits(HEADS, KV_HEADS, DIM, pos + tokens, KINDS[bits])
    make.fill(cache, pos)
    flash = saetta.FlashParams(HEADS, KV_HEADS, pos, tokens, 1.0 / math.sqrt(DIM))
    state = {"cache": cache, "flash": flash, "k": make.kv(tokens).view(-1), "v": make.kv(tokens).view(-1),
             "q": make.normal(tokens, HEADS, DIM).to(torch.float16), "qg": make.normal(tokens, HEADS, 2 * DIM),
             "out": torch.zeros(tokens, HEADS, DIM, device="cuda"), "new": _new_rows(cache, pos, tokens)}
    if case["kind"] == "gemm":
        state["gemm"] = saetta.attention_gemm.AttGemm(tokens, KV_HEADS)
    else:
        need = saetta.attention_prefill.workspace_bytes(flash)
        state["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    return state


def _layer(make):
    """The weights of a DeltaNet layer."""
    return {"w": make.normal(CHANNELS * CONV, scale=0.5), "a_log": make.normal(V_HEADS), "dt_bias": make.normal(V_HEADS),
            "norm": 1.0 + make.normal(V_DIM, scale=0.1)}


def _prepare_deltanet(case, make):
    layers, rows = case["layers"], case["rows"]
    x, z = make.normal(layers, rows, CHANNELS), make.normal(layers, rows, V_HEADS * V_DIM)
    a, b = make.normal(layers, rows, V_HEADS), make.normal(layers, rows, V_HEADS)
    outputs = {"y": torch.zeros(layers, rows, V_HEADS * V_DIM, device="cuda"),
               "conv": make.normal(layers, CONV - 1, CHANNELS),
               "state": make.normal(layers, V_HEADS, V_DIM, K_DIM, scale=0.1)}
    if rows > 1:
        outputs["conv_snaps"] = torch.zeros(layers, rows, CONV - 1, CHANNELS, device="cuda")
        outputs["state_snaps"] = torch.zeros(layers, rows, V_HEADS, V_DIM, K_DIM, device="cuda")
    plan = saetta.Plan()
    for i in range(layers):
        n = _layer(make)
        buffers = (x[i], n["w"], outputs["conv"][i], a[i], b[i], n["a_log"], n["dt_bias"], outputs["state"][i], z[i], n["norm"],
                   outputs["y"][i])
        if rows == 1:
            saetta.deltanet_token(plan, *buffers, K_HEADS, V_HEADS, V_DIM, CONV, EPS)
        else:
            saetta.deltanet_rows_fused(plan, *buffers, K_HEADS, V_HEADS, V_DIM, CONV, rows, EPS, outputs["conv_snaps"][i],
                                       outputs["state_snaps"][i])
    return {"plan": plan, "built": plan.build(graph=case["graph"]), "params": None, "outputs": outputs}


def _prepare_chunk(case, make):
    tokens, n = case["tokens"], _layer(make)
    x, z = make.normal(tokens, CHANNELS), make.normal(tokens, V_HEADS * V_DIM)
    a, b = make.normal(tokens, V_HEADS), make.normal(tokens, V_HEADS)
    mixed = torch.zeros(tokens, CHANNELS, device="cuda")
    conv, state = make.normal(CONV - 1, CHANNELS), make.normal(V_HEADS, V_DIM, K_DIM, scale=0.1)
    y = torch.zeros(tokens, V_HEADS * V_DIM, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_conv_rows(plan, x, n["w"], conv, mixed, CHANNELS, CONV, tokens)
    saetta.deltanet_rows(plan, mixed, a, b, n["a_log"], n["dt_bias"], state, z, n["norm"], y, K_HEADS, V_HEADS, V_DIM, tokens, EPS)
    return {"plan": plan, "built": plan.build(), "params": None,
            "outputs": {"mixed": mixed, "y": y, "conv": conv, "state": state}}


def prepare(case, seed):
    make = _Maker(seed)
    kind = case["kind"]
    state = {"token": _prepare_token, "prefill": _prepare_prefill, "gemm": _prepare_prefill, "deltanet": _prepare_deltanet,
             "chunk": _prepare_chunk}[kind](case, make)
    state["kind"] = kind
    return state


def run(state):
    if state["kind"] in ("prefill", "gemm"):
        cache, flash, k, v, out = state["cache"], state["flash"], state["k"], state["v"], state["out"]
        pos, tokens = flash.pos, flash.tokens
        if cache.quant:
            cache.quant[0].encode(k, pos, tokens)
            cache.quant[1].encode(v, pos, tokens)
        else:
            saetta.to_half(k, cache.keys[pos * VALUES:(pos + tokens) * VALUES])
            saetta.to_half(v, cache.values[pos * VALUES:(pos + tokens) * VALUES])
        if state["kind"] == "gemm":
            state["gemm"].encode(state["q"], cache.keys, cache.values, cache.quant, state["qg"], out, flash)
        elif cache.quant:
            saetta.attention_prefill.encode_quant(state["q"], *cache.quant, state["qg"], out, flash, workspace=state["workspace"])
        else:
            saetta.attention_prefill.encode(saetta.attention_prefill.DEFAULT, state["q"], cache.keys, cache.values, state["qg"],
                                            out, flash, workspace=state["workspace"])
        return {"out": out, "new": state["new"]}
    if state["params"] is not None:
        state["plan"].set_params(state["params"])  # the token's position, as before every token
    state["built"].run()
    return state["outputs"]


def _deltanet_work(tokens, rows_kept):
    """Bytes and operations of `tokens` tokens in one DeltaNet layer, without the conv's output."""
    state, conv = 4 * V_HEADS * V_DIM * K_DIM, 4 * (CONV - 1) * CHANNELS
    values = V_HEADS * V_DIM
    nbytes = 4 * (tokens * (CHANNELS + 2 * values + 2 * V_HEADS) + CHANNELS * CONV + 2 * V_HEADS + V_DIM)
    nbytes += (2 + rows_kept) * (state + conv)
    return nbytes, tokens * (7.0 * values * K_DIM + 2.0 * CHANNELS * CONV)


def work(case):
    kind = case["kind"]
    if kind == "deltanet":
        rows = case["rows"]
        nbytes, flops = _deltanet_work(rows, rows if rows > 1 else 0)
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}
    if kind == "chunk":
        nbytes, flops = _deltanet_work(case["tokens"], 0)
        return {"bytes": nbytes + 2 * 4 * case["tokens"] * CHANNELS, "flops": flops}
    token_bytes = 2 * VALUES * KINDS[case["bits"]].bytes_per_value()  # the key and the value of a token in the cache
    if kind == "token":
        rows, context = case["rows"], case["context"]
        nbytes = (context + rows) * token_bytes                              # the cache
        nbytes += 4 * rows * (2 * HEADS * DIM + 2 * VALUES) + 4 * 2 * DIM    # q, gates, the new keys and values, the norms
        nbytes += 4 * rows * 2 * HEADS * DIM                                 # q after the norm, and the result
        pairs = sum(context + r + 1 for r in range(rows))
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * 4.0 * HEADS * DIM * pairs}
    tokens, pos = case["tokens"], case["pos"]
    nbytes = (pos + tokens) * token_bytes + tokens * (4 * 2 * VALUES)        # the cache, the new keys and values
    nbytes += tokens * HEADS * DIM * (2 + 4 + 4)                             # q, gates, the result
    return {"bytes": nbytes, "flops": 4.0 * HEADS * DIM * (tokens * pos + tokens * (tokens + 1) / 2)}


def tolerance(case):
    if case["kind"] in ("prefill", "gemm"):
        return {"rel": 1e-3, "max": 2e-2}  # halves go into the products and the probabilities are halves; codes are equal
    return {"rel": 1e-5, "max": 1e-3}      # 32-bit sums, in another order; codes are equal
