"""Chunked causal prefill attention on the GPU against the oracle.

Restates tests/attention_prefill.rs (spread data; (pos, tokens) = (0,1), (0,7), (5,8), (70,100),
(1000,64), (0,300), (4093,37); finite and max abs diff < 2e-3) with the oracle's token-by-token
f32 CPU attention as the other side (src/prefill.rs:2489-2495 defines the chunk that way), over a
half cache and over 8/4-bit caches read in place; bar of this build: rel-RMS <= 1e-3.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

from gpu_common import D, H, KV, VALUES, dev, host, oracle, saetta

pytestmark = pytest.mark.gpu
KINDS = [saetta.KvBits.Half, saetta.KvBits.Eight, saetta.KvBits.Four]
SHAPES = [(0, 1), (0, 7), (5, 8), (70, 100), (1000, 64), (0, 300), (4093, 37)]
REL_RMS = 1e-3
MAX_ABS = 2e-3  # tests/attention_prefill.rs:56-59


def make_cache(kind, k, v, capacity, chunk_from=None):
    """Cache holding k, v [n, 512].  Rows from chunk_from on are appended on the device
    (to_half / kv_quantize), the others come from the host; rows past n hold NaN patterns."""
    n = k.shape[0]
    first = n if chunk_from is None else chunk_from
    if kind is saetta.KvBits.Half:
        kc = torch.full((capacity, VALUES), float("nan"), dtype=torch.float16, device="cuda")
        vc = torch.full((capacity, VALUES), float("nan"), dtype=torch.float16, device="cuda")
        kc[:first], vc[:first] = dev(k[:first].astype(np.float16)), dev(v[:first].astype(np.float16))
        if first < n:
            saetta.to_half(dev(k[first:].reshape(-1)), kc[first:n].view(-1))
            saetta.to_half(dev(v[first:].reshape(-1)), vc[first:n].view(-1))
        kf = k.astype(np.float16).astype(np.float32)
        vf = v.astype(np.float16).astype(np.float32)
        return kc, vc, kf, vf
    bits = kind.value
    kc, vc = saetta.QuantRows(kind, VALUES, capacity), saetta.QuantRows(kind, VALUES, capacity)
    for c, x in ((kc, k), (vc, v)):
        c.scales[:], c.biases[:], c.data[:] = float("nan"), float("inf"), -1
        if first:
            data, scales, biases = oracle.quantize(x[:first], bits)
            c.data[:data.size] = dev(data.view(np.int32))
            c.scales[:scales.size] = dev(scales.view(np.float16))
            c.biases[:biases.size] = dev(biases.view(np.float16))
        if first < n:
            c.encode(dev(x[first:].reshape(-1)), first, n - first)  # quantize-on-append
    return kc, vc, oracle.round_trip_as_half(k, bits), oracle.round_trip_as_half(v, bits)


def run(kind, q16, kc, vc, qg, pos, tokens):
    out = torch.full((tokens, H, D), float("nan"), device="cuda")
    p = saetta.FlashParams(H, KV, pos, tokens, 1.0 / math.sqrt(D))
    if kind is saetta.KvBits.Half:
        saetta.attention_prefill.encode(saetta.attention_prefill.DEFAULT, dev(q16), kc, vc, dev(qg), out, p)
    else:
        saetta.attention_prefill.encode_quant(dev(q16), kc, vc, dev(qg), out, p)
    return host(out)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos,tokens", SHAPES)
def test_matches_cpu_on_spread_data(kind, pos, tokens):
    n = pos + tokens
    capacity = -(-n // 64) * 64 + 64
    q16 = oracle.spread(tokens * H * D, 1).reshape(tokens, H, D)
    k = oracle.spread(n * VALUES, 2).astype(np.float32).reshape(n, VALUES)
    v = oracle.spread(n * VALUES, 3).astype(np.float32).reshape(n, VALUES)
    qg = ((np.arange(tokens * H * 2 * D) % 7) - 3).astype(np.float32).reshape(tokens, H, 2 * D)
    kc, vc, kf, vf = make_cache(kind, k, v, capacity, chunk_from=pos)
    got = run(kind, q16, kc, vc, qg, pos, tokens)
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() < MAX_ABS, f"{kind} pos {pos} tokens {tokens}"
    assert oracle.rel_rms(got, want) < REL_RMS


@pytest.mark.parametrize("kind", KINDS)
def test_gaussian_chunk_with_cached_prefix(kind):
    # a chunk behind a prefix of its length, scaled to what the CPU finishes in seconds: bf16-exact N(0,1) q, a cached
    # prefix quantized on the host, the chunk's K/V quantized on the device, gate N(0,1).
    rng = np.random.default_rng(12)
    pos, tokens = 300, 200
    n = pos + tokens
    q = rng.standard_normal((tokens, H, D)).astype(np.float32)
    q16 = torch.from_numpy(q).to(torch.bfloat16).to(torch.float16).numpy()
    k = rng.standard_normal((n, VALUES)).astype(np.float32)
    v = rng.standard_normal((n, VALUES)).astype(np.float32)
    qg = rng.standard_normal((tokens, H, 2 * D)).astype(np.float32)
    kc, vc, kf, vf = make_cache(kind, k, v, n, chunk_from=pos)
    got = run(kind, q16, kc, vc, qg, pos, tokens)
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    assert oracle.rel_rms(got, want) < REL_RMS
    assert np.abs(got - want).max() < MAX_ABS


def test_causality_at_full_size():
    # The 4096 + 4096 shape: a token's output must not change when later keys change, and the
    # first token of the chunk must equal single-token decode attention over pos + 1 keys.
    rng = np.random.default_rng(3)
    pos = tokens = 4096
    n = pos + tokens
    kind = saetta.KvBits.Eight
    gen = torch.Generator(device="cuda").manual_seed(5)
    kx = torch.randn(n, VALUES, generator=gen, device="cuda")
    vx = torch.randn(n, VALUES, generator=gen, device="cuda")
    q16 = torch.randn(tokens, H, D, generator=gen, device="cuda").to(torch.float16)
    qg = torch.randn(tokens, H, 2 * D, generator=gen, device="cuda")
    kc, vc = saetta.QuantRows(kind, VALUES, n), saetta.QuantRows(kind, VALUES, n)
    kc.encode(kx.view(-1), 0, n), vc.encode(vx.view(-1), 0, n)
    p = saetta.FlashParams(H, KV, pos, tokens, 1.0 / 16)
    out = torch.empty(tokens, H, D, device="cuda")
    saetta.attention_prefill.encode_quant(q16, kc, vc, qg, out, p)
    a = host(out).copy()
    assert np.isfinite(a).all()
    # overwrite the last 1000 tokens' keys and values: rows before them must stay bit-equal
    kc.encode(vx[-1000:].contiguous().view(-1), n - 1000, 1000)
    vc.encode(kx[-1000:].contiguous().view(-1), n - 1000, 1000)
    saetta.attention_prefill.encode_quant(q16, kc, vc, qg, out, p)
    b = host(out)
    assert np.array_equal(a[:tokens - 1000], b[:tokens - 1000])
    assert not np.array_equal(a[tokens - 1000:], b[tokens - 1000:])
    # token 0 of the chunk against decode attention (itself checked against the oracle)
    kc.encode(kx[-1000:].contiguous().view(-1), n - 1000, 1000)
    vc.encode(vx[-1000:].contiguous().view(-1), n - 1000, 1000)
    att = saetta.DecodeAttention(H, KV, D, n)
    one = torch.empty(H, D, device="cuda")
    plan = saetta.Plan()
    att.record_quant(plan, q16[0].float().contiguous(), kc, vc, qg[0].contiguous(), one)
    plan.set_params(saetta.TokenParams(0, pos))
    plan.build().run()
    assert oracle.rel_rms(a[0], host(one)) < REL_RMS
    # a sample of rows against the oracle
    groups = n * 8
    kf = oracle.dequantize(host(kc.data).view(np.uint32), host(kc.scales).view(np.uint16), host(kc.biases).view(np.uint16), 8)
    vf = oracle.dequantize(host(vc.data).view(np.uint32), host(vc.scales).view(np.uint16), host(vc.biases).view(np.uint16), 8)
    kf = kf.astype(np.float16).astype(np.float32)
    vf = vf.astype(np.float16).astype(np.float32)
    qh, qgh = host(q16).astype(np.float32), host(qg)
    # Workgroups take 16-token tiles heaviest first, the second half of the tiles in a second
    # round: rows from both rounds, tile edges included; every row covers both kv heads.
    for i in (0, 1, 15, 16, 777, 1234, 2047, 2048, 2500, 3333, 4080, 4095):
        want = oracle.attend(qh[i], kf, vf, pos + i + 1, q_and_gate=qgh[i], threads=8)
        assert oracle.rel_rms(a[i], want) < REL_RMS


def test_shape_and_argument_checks():
    q = torch.zeros(1, H, D, dtype=torch.float16, device="cuda")
    kc = torch.zeros(64, VALUES, dtype=torch.float16, device="cuda")
    qg = torch.zeros(1, H, 2 * D, device="cuda")
    out = torch.zeros(1, H, D, device="cuda")
    with pytest.raises(ValueError):
        saetta.attention_prefill.encode("attention_fa16", q, kc, kc, qg, out, saetta.FlashParams(H, KV, 0, 1, 0.0625))
    with pytest.raises(ValueError):
        saetta.attention_prefill.encode("attention_fa8", q, kc, kc, qg, out, saetta.FlashParams(H, 4, 0, 1, 0.0625))
    # zero tokens: nothing to do
    saetta.attention_prefill.encode("attention_fa8", q, kc, kc, qg, out, saetta.FlashParams(H, KV, 0, 0, 0.0625))


def test_spread_rows2_and_bench_mirror_the_reference():
    # spread (src/attention_prefill.rs:102-108) against the oracle's restatement
    got = host(saetta.attention_prefill.spread(5000, 3)).astype(np.float32)
    assert np.array_equal(got, oracle.spread(5000, 3).astype(np.float32))
    # encode_rows2 is the same computation as encode
    pos, tokens = 40, 24
    n = pos + tokens
    q16 = oracle.spread(tokens * H * D, 1).reshape(tokens, H, D)
    k = torch.from_numpy(oracle.spread(n * VALUES, 2)).cuda()
    v = torch.from_numpy(oracle.spread(n * VALUES, 3)).cuda()
    qg = dev(((np.arange(tokens * H * 2 * D) % 7) - 3).astype(np.float32))
    q = torch.from_numpy(q16).cuda()
    a, b = torch.empty(tokens, H, D, device="cuda"), torch.empty(tokens, H, D, device="cuda")
    p = saetta.FlashParams(H, KV, pos, tokens, 1 / 16)
    saetta.attention_prefill.encode("attention_fa4", q, k, v, qg, a, p)
    saetta.attention_prefill.encode_rows2(q, k, v, qg, b, p)
    assert torch.equal(a, b)
    # bench of both modules on toy sizes: shapes and sanity of what they report
    rows = saetta.attention_prefill.bench([100], 64, 2)
    assert rows[0]["context"] == 128 and rows[0]["last_TFLOP/s"] > 0 and rows[0]["mid_TFLOP/s"] > 0
    for bits in (saetta.KvBits.Half, saetta.KvBits.Eight):
        rows = saetta.bench([256, 1000], 2, 3, bits)
        assert [r["tokens"] for r in rows] == [256, 1000] and all(r["GB/s"] > 0 and r["reduce_ms"] > 0 for r in rows)


@pytest.mark.parametrize("pos,tokens", [(4096, 4096), (0, 1000), (37, 3001), (100, 9000)])
def test_equal_keys_give_running_means_at_full_size(pos, tokens):
    # A closed form for every one of the 4096 x 16 rows of the headline shape: with the same key in every cache
    # row all scores of a token are equal, so token i's output is the mean of the first pos + i + 1 value rows
    # (as the half values the cache is read through) times sigmoid(gate), whatever q is.  A key block skipped,
    # taken twice or masked at the wrong place, or a wrong merge of the two waves of a row group, moves it.
    # The other shapes are the other ways the tiles reach the workgroups (one workgroup per CU takes tiles until
    # none are left, the ones past its first by asking a counter): 126 tiles, fewer than workgroups; 376, between
    # one and two each; 1126, more than four each, the chunk and its position ragged against tiles and key blocks.
    n = pos + tokens
    kind = saetta.KvBits.Eight
    gen = torch.Generator(device="cuda").manual_seed(17)
    krow = torch.randn(VALUES, generator=gen, device="cuda") * 2.0
    kx = krow.repeat(n, 1).contiguous()
    vx = torch.randn(n, VALUES, generator=gen, device="cuda")
    vx[:, 7] += 2.0
    q16 = torch.randn(tokens, H, D, generator=gen, device="cuda").to(torch.float16)
    qg = torch.randn(tokens, H, 2 * D, generator=gen, device="cuda")
    kc, vc = saetta.QuantRows(kind, VALUES, n), saetta.QuantRows(kind, VALUES, n)
    kc.encode(kx.view(-1), 0, n), vc.encode(vx.view(-1), 0, n)
    p = saetta.FlashParams(H, KV, pos, tokens, 1.0 / 16)
    out = torch.full((tokens, H, D), float("nan"), device="cuda")
    saetta.attention_prefill.encode_quant(q16, kc, vc, qg, out, p)
    got = host(out)
    vf = oracle.dequantize(host(vc.data).view(np.uint32), host(vc.scales).view(np.uint16), host(vc.biases).view(np.uint16), 8)
    vf = vf.reshape(n, VALUES).astype(np.float16).astype(np.float64)
    sums = np.cumsum(vf[pos:], axis=0) + vf[:pos].sum(axis=0)          # [tokens, 512]
    assert np.isfinite(got).all()
    means = (sums / (pos + 1 + np.arange(tokens))[:, None]).reshape(tokens, KV, D)
    gate = 1.0 / (1.0 + np.exp(-host(qg).reshape(tokens, H, 2 * D)[:, :, D:].astype(np.float64)))
    want = np.repeat(means, H // KV, axis=1) * gate
    worst = np.abs(got - want).max()
    assert worst < 2e-5, worst


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos", [1, 2, 3, 5, 17, 30, 31])
def test_chunk_from_a_position_that_splits_a_row_group(kind, pos):
    # A chunk that starts at a position that is no multiple of 4, early in the cache: in the row group whose
    # tokens see 30 .. 33 keys some rows end inside key block 0 and others reach block 1, so the wave that
    # takes the odd blocks meets rows for which its first block is masked whole.
    rng = np.random.default_rng(600 + pos)
    tokens = 70
    n = pos + tokens
    k = rng.standard_normal((n, VALUES)).astype(np.float32)
    v = rng.standard_normal((n, VALUES)).astype(np.float32)
    q16 = rng.standard_normal((tokens, H, D)).astype(np.float16)
    qg = rng.standard_normal((tokens, H, 2 * D)).astype(np.float32)
    kc, vc, kf, vf = make_cache(kind, k, v, n + 9, chunk_from=pos)
    got = run(kind, q16, kc, vc, qg, pos, tokens)
    assert np.isfinite(got).all()
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    assert oracle.rel_rms(got, want) < REL_RMS
    assert np.abs(got - want).max() < MAX_ABS


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos,tokens", [(250, 16), (1018, 20), (2040, 33), (5000, 7), (9985, 50)])
def test_keys_in_parts(kind, pos, tokens):
    # Few tokens behind a long prefix: a tile's keys go to several workgroups and a second kernel joins the parts.
    # (250, 16) is next to the smallest split, (1018, 20) and (2040, 33) have tiles whose tokens cross a key block where
    # parts end (rows that see nothing of the last part), (9985, 50) the most parts and a ragged last tile.
    rng = np.random.default_rng(pos)
    n = pos + tokens
    k = rng.standard_normal((n, VALUES)).astype(np.float32)
    v = rng.standard_normal((n, VALUES)).astype(np.float32)
    q16 = rng.standard_normal((tokens, H, D)).astype(np.float16)
    qg = rng.standard_normal((tokens, H, 2 * D)).astype(np.float32)
    kc, vc, kf, vf = make_cache(kind, k, v, n + 5, chunk_from=pos)
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    p = saetta.FlashParams(H, KV, pos, tokens, 1.0 / math.sqrt(D))
    images = saetta.ffi.lib().saetta_prefill_workspace_bytes(0, -(-n // 32) * 32, KV)  # of one tile-aligned chunk: no parts
    for nbytes in (saetta.attention_prefill.workspace_bytes(p), images):  # and a workspace that holds no parts
        ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device="cuda")
        out = torch.full((tokens, H, D), float("nan"), device="cuda")
        if kind is saetta.KvBits.Half:
            saetta.attention_prefill.encode(saetta.attention_prefill.DEFAULT, dev(q16), kc, vc, dev(qg), out, p, workspace=ws)
        else:
            saetta.attention_prefill.encode_quant(dev(q16), kc, vc, dev(qg), out, p, workspace=ws)
        got = host(out)
        assert np.isfinite(got).all()
        assert oracle.rel_rms(got, want) < REL_RMS
        assert np.abs(got - want).max() < MAX_ABS


def attention_64(q16, k, v, qg, pos):
    """out [tokens][heads][256] in 64 bits, k and v [pos + tokens][kv][256] as the cache stands for them."""
    tokens, heads, kv = q16.shape[0], q16.shape[1], k.shape[1]
    q = q16.double().view(tokens, kv, 8, D).permute(1, 2, 0, 3).reshape(kv, 8 * tokens, D)
    s = torch.matmul(q, k.double().permute(1, 2, 0).contiguous()) / 16
    sees = torch.arange(pos + tokens, device="cuda")[None] <= pos + torch.arange(tokens, device="cuda")[:, None]
    p = torch.softmax(s.view(kv, 8, tokens, -1).masked_fill(~sees, float("-inf")), -1).view(kv, 8 * tokens, -1)
    o = torch.matmul(p, v.double().permute(1, 0, 2).contiguous()).view(kv, 8, tokens, D).permute(2, 0, 1, 3).reshape(tokens, heads, D)
    return o * torch.sigmoid(qg.double().view(tokens, heads, 2 * D)[:, :, D:])


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos,tokens,kv", [(505, 1, 1), (767, 2, 2), (1020, 9, 2), (1279, 30, 3), (1800, 64, 2), (2047, 130, 2), (3000, 250, 2), (6100, 33, 1),
                                           (9000, 7, 5), (20001, 30, 2), (50000, 5, 2), (32510, 1, 2), (33998, 49, 5)])
def test_row_groups_with_their_keys_in_parts(kind, pos, tokens, kv):
    # A part is a multiple of 8 blocks of 32 keys: a row group that sees no key of a part that its tile has (1020, 1279, 2047),
    # one block of the last, parts of one round and of many, two rounds of workgroups (33998, halves), as many as 64 parts
    # (32510), kv heads that an eighth of the workgroups does not divide; in a workspace of NaN of just the size, and in one with
    # room for the images, which holds the parts too where there are few rows to a key (767, 1020, from 9000 on) and elsewhere
    # makes it the layout without them.
    heads, n = 8 * kv, pos + tokens
    gen = torch.Generator(device="cuda").manual_seed(pos)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    k, v, q16, qg = normal(n, kv * D), normal(n, kv * D), normal(tokens, heads, D).half(), normal(tokens, heads, 2 * D)
    if kind is saetta.KvBits.Half:
        kc, vc = k.half(), v.half()
        kf, vf = kc, vc
    else:
        kc, vc = saetta.QuantRows(kind, kv * D, n), saetta.QuantRows(kind, kv * D, n)
        kc.encode(k.view(-1), 0, n), vc.encode(v.view(-1), 0, n)
        kf, vf = (saetta.dequantize(*c.tensors(), kind) for c in (kc, vc))
    want = attention_64(q16, kf.view(n, kv, D), vf.view(n, kv, D), qg, pos)
    p = saetta.FlashParams(heads, kv, pos, tokens, 1.0 / 16)
    for nbytes in (saetta.attention_prefill.workspace_bytes(p), -(-n // 32) * kv * 32768 + 256):
        ws, out = torch.full((nbytes,), 0xff, dtype=torch.uint8, device="cuda"), torch.full((tokens, heads, D), float("nan"), device="cuda")
        if kind is saetta.KvBits.Half:
            saetta.attention_prefill.encode(saetta.attention_prefill.DEFAULT, q16, kc, vc, qg, out, p, workspace=ws)
        else:
            saetta.attention_prefill.encode_quant(q16, kc, vc, qg, out, p, workspace=ws)
        off = (out.double() - want).norm() / want.norm()
        assert float(off) < REL_RMS, float(off)
        assert float((out - want).abs().max()) < MAX_ABS


def chunk(kind, pos, tokens, kv):
    """Inputs of a chunk, what the cache stands for in 64 bits, and the C call of it in a workspace (address, bytes)."""
    heads, n = 8 * kv, pos + tokens
    gen = torch.Generator(device="cuda").manual_seed(n)
    normal = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    k, v, q16, qg = normal(n, kv * D), normal(n, kv * D), normal(tokens, heads, D).half(), normal(tokens, heads, 2 * D)
    lib, p, out = saetta.ffi.lib(), saetta.FlashParams(heads, kv, pos, tokens, 1.0 / 16), torch.empty(tokens, heads, D, device="cuda")
    if kind is saetta.KvBits.Half:
        keys, values = k.half(), v.half()
        kf, vf = keys, values
        call = lambda ws, size: lib.saetta_attn_prefill(saetta.host._stream(), q16.data_ptr(), keys.data_ptr(), values.data_ptr(), qg.data_ptr(),  # noqa: E731
                                                        out.data_ptr(), p, ws, size)
    else:
        keys, values = saetta.QuantRows(kind, kv * D, n), saetta.QuantRows(kind, kv * D, n)
        keys.encode(k.view(-1), 0, n), values.encode(v.view(-1), 0, n)
        kf, vf = (saetta.dequantize(*c.tensors(), kind) for c in (keys, values))
        call = lambda ws, size: lib.saetta_attn_prefill_quant(saetta.host._stream(), kind.value, q16.data_ptr(), keys.c(), values.c(),  # noqa: E731
                                                              qg.data_ptr(), out.data_ptr(), p, ws, size)
    return call, out, p, attention_64(q16, kf.view(n, kv, D), vf.view(n, kv, D), qg, pos)


@pytest.mark.parametrize("kind,pos,tokens,kv", [(saetta.KvBits.Half, 1166, 1, 1), (saetta.KvBits.Half, 1166, 85, 1), (saetta.KvBits.Half, 1203, 183, 1),
                                                (saetta.KvBits.Half, 315, 1317, 1), (saetta.KvBits.Eight, 981, 134, 1), (saetta.KvBits.Four, 759, 638, 1),
                                                (saetta.KvBits.Eight, 95, 1401, 1), (saetta.KvBits.Half, 767, 2, 2), (saetta.KvBits.Four, 200, 30, 2)])
def test_short_chunks_are_recorded_without_a_workspace(kind, pos, tokens, kv):
    # what the row groups take without parts needs none; sizes at the line to the tiles, which a recorded call without a
    # workspace is refused
    call, out, _, want = chunk(kind, pos, tokens, kv)
    lib, results = saetta.ffi.lib(), []
    assert lib.saetta_plan_begin() == 0
    results.append(call(None, 0))
    plan = ctypes.c_void_p(lib.saetta_plan_end())
    try:
        assert results == [0], lib.saetta_last_error()
        out.fill_(float("nan"))
        assert lib.saetta_plan_run(saetta.host._stream(), plan) == 0
        assert float((out.double() - want).norm() / want.norm()) < REL_RMS
        assert float((out - want).abs().max()) < MAX_ABS
    finally:
        torch.cuda.synchronize()
        lib.saetta_plan_free(plan)


@pytest.mark.parametrize("kind,pos,tokens,kv", [(saetta.KvBits.Half, 767, 2, 2), (saetta.KvBits.Half, 1020, 9, 2), (saetta.KvBits.Half, 961, 139, 2),
                                                (saetta.KvBits.Eight, 767, 2, 2), (saetta.KvBits.Four, 767, 2, 2), (saetta.KvBits.Half, 2300, 4, 2),
                                                (saetta.KvBits.Half, 200, 30, 2)])
def test_no_workspace_is_as_good_as_one(kind, pos, tokens, kv):
    # the library's own holds the parts of a chunk that could do without too: the same bits as in a workspace of just the size;
    # one that does not hold the images is refused
    call, out, p, want = chunk(kind, pos, tokens, kv)
    size = saetta.attention_prefill.workspace_bytes(p)
    ws, results = torch.full((size,), 0xff, dtype=torch.uint8, device="cuda"), []
    for args in ((ws.data_ptr(), size), (None, 0)):
        out.fill_(float("nan"))
        assert call(*args) == 0, saetta.ffi.lib().saetta_last_error()
        results.append(host(out))
        assert float((out.double() - want).norm() / want.norm()) < REL_RMS
    assert np.array_equal(*results)
    for nbytes in (0, 1, -(-(pos + tokens) // 32) * kv * 32768):
        assert call(ws.data_ptr(), nbytes) == -6  # SAETTA_E_SCRATCH


@pytest.mark.parametrize("kind,pos,tokens,kv,split", [(saetta.KvBits.Half, 379, 5, 2, False), (saetta.KvBits.Half, 380, 5, 2, True), (saetta.KvBits.Eight, 314, 6, 2, False),
                                                      (saetta.KvBits.Four, 315, 6, 2, True), (saetta.KvBits.Half, 480, 152, 2, True), (saetta.KvBits.Half, 480, 153, 2, False),
                                                      (saetta.KvBits.Eight, 400, 152, 2, True), (saetta.KvBits.Four, 400, 153, 2, False), (saetta.KvBits.Eight, 511, 1, 1, True)])
def test_few_row_groups_over_some_hundred_keys(kind, pos, tokens, kv, split):
    # at the lines of the rule: the blocks from which keys go to parts, 76 row groups and 78 (256 CUs); recorded without a workspace
    # the same chunk takes all of its keys in one workgroup a row group
    call, out, p, want = chunk(kind, pos, tokens, kv)
    size = saetta.attention_prefill.workspace_bytes(p)
    ws = torch.full((size,), 0xff, dtype=torch.uint8, device="cuda")
    lib, results = saetta.ffi.lib(), []
    assert lib.saetta_plan_begin() == 0
    results.append(call(None, 0))
    plan = ctypes.c_void_p(lib.saetta_plan_end())
    assert results == [0], lib.saetta_last_error()
    try:
        for run_it in (lambda: call(ws.data_ptr(), size), lambda: lib.saetta_plan_run(saetta.host._stream(), plan)):
            out.fill_(float("nan"))
            assert run_it() == 0, lib.saetta_last_error()
            assert float((out.double() - want).norm() / want.norm()) < REL_RMS
            assert float((out - want).abs().max()) < MAX_ABS
        assert bool((ws != 0xff).any()) == split
    finally:
        torch.cuda.synchronize()
        lib.saetta_plan_free(plan)


@pytest.mark.parametrize("pos,tokens", [(2045, 3), (2300, 4), (4200, 3), (8186, 5), (8200, 4), (16300, 2)])
def test_many_parts_are_merged_by_teams(pos, tokens):
    # 8 parts of 8 blocks and one team, 9 and more and four: teams without a part, one batch each and two, a last batch of one
    test_row_groups_with_their_keys_in_parts(saetta.KvBits.Half, pos, tokens, 2)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos,tokens", [(0, 4), (31, 1), (32, 2), (125, 3), (126, 5), (253, 3), (254, 5), (300, 17), (500, 30)])
def test_short_chunks_over_short_contexts(kind, pos, tokens):
    # A workgroup per 4 tokens, its 8 waves on alternate blocks of 32 keys: one block, two, four and five (the waves'
    # parts are joined in one pass or two), eight and nine (a wave with two blocks), 17; ragged last tokens.
    rng = np.random.default_rng(1000 * pos + tokens)
    n = pos + tokens
    k = rng.standard_normal((n, VALUES)).astype(np.float32)
    v = rng.standard_normal((n, VALUES)).astype(np.float32)
    q16 = rng.standard_normal((tokens, H, D)).astype(np.float16)
    qg = rng.standard_normal((tokens, H, 2 * D)).astype(np.float32)
    kc, vc, kf, vf = make_cache(kind, k, v, n + 7, chunk_from=pos)
    got = run(kind, q16, kc, vc, qg, pos, tokens)
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    assert np.isfinite(got).all()
    assert oracle.rel_rms(got, want) < REL_RMS
    assert np.abs(got - want).max() < MAX_ABS


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos,tokens", [(255, 1), (256, 1), (509, 3), (510, 6), (640, 9), (150, 600), (0, 701), (740, 7), (900, 150)])
def test_short_chunks_whose_scores_grow(kind, pos, tokens):
    # Rounds of 8 blocks, one a wave: one round and two (8 and 9 blocks), 16 and 17 blocks, a row group with a block more
    # than the one before it, more row groups than CUs (two of them past the line of codes, before that of halves).  The
    # keys grow with the square of their position, so that later rounds raise a wave's maximum by more than the slack of 8
    # powers of two (scores to +-11; rounding keys of codes to halves moves those by 4e-4, their standard deviation, and an
    # output by a quarter of that times the 4 or 5 between two values: within the tolerance of the other tests).
    rng = np.random.default_rng(1000 * pos + tokens)
    n = pos + tokens
    k = (rng.standard_normal((n, VALUES)) * 3.0 * np.linspace(0.2, 1.0, n)[:, None] ** 2).astype(np.float32)
    v = rng.standard_normal((n, VALUES)).astype(np.float32)
    q16 = rng.standard_normal((tokens, H, D)).astype(np.float16)
    qg = rng.standard_normal((tokens, H, 2 * D)).astype(np.float32)
    kc, vc, kf, vf = make_cache(kind, k, v, n + 7, chunk_from=pos)
    got = run(kind, q16, kc, vc, qg, pos, tokens)
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    assert np.isfinite(got).all()
    assert oracle.rel_rms(got, want) < REL_RMS
    assert np.abs(got - want).max() < MAX_ABS


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pos,tokens,kv", [(0, 1, 3), (190, 34, 1), (193, 31, 2), (225, 31, 3), (226, 31, 2), (207, 512, 2), (208, 514, 1), (288, 512, 2), (289, 512, 2),
                                           (1, 900, 2), (4095, 1, 2), (4090, 12, 1), (20000, 12, 2), (1997, 64, 2), (40000, 7, 2), (3000, 120, 2)])
def test_short_chunks_whose_waves_share_their_blocks(kind, pos, tokens, kv):
    # one block; the last round with 6, 7 and 8 blocks (where the probabilities lie differs from the eighth on) and with the ninth
    # in a second round; the keys in the mean at which the rounds of 4-bit codes and of halves stop being shared, and one past them;
    # parts of 8, 16, 24 and 32 blocks; 1, 2 and 3 kv heads
    call, out, p, want = chunk(kind, pos, tokens, kv)
    out.fill_(float("nan"))
    size = saetta.attention_prefill.workspace_bytes(p)
    ws = torch.full((size,), 0xff, dtype=torch.uint8, device="cuda")
    assert call(ws.data_ptr(), size) == 0, saetta.ffi.lib().saetta_last_error()
    assert float((out.double() - want).norm() / want.norm()) < REL_RMS
    assert float((out - want).abs().max()) < MAX_ABS


PART_O, PART_ML = 16 * 8 * D * 4, 16 * 8 * 8  # bytes of a tile's part (16 tokens, 8 heads): its sums; its maxima and their sums


def parts_written(ws, plain, tokens, kv, parts):
    """[part][tile of 16 tokens]: whether a call left sums there, in a workspace of 0xff with `parts` parts behind `plain` bytes."""
    items = parts * -(-tokens // 16) * kv
    sums = ws[plain + items * PART_O:plain + items * (PART_O + PART_ML)].view(torch.int32).view(parts, -1, kv * 16 * 8 * 2)
    return (sums != -1).any(2)


@pytest.mark.parametrize("kind,pos,tokens,kv,blocks", [(saetta.KvBits.Half, 1000, 2100, 2, 50), (saetta.KvBits.Eight, 1003, 2113, 2, 50), (saetta.KvBits.Four, 9990, 2309, 2, 130),
                                                       (saetta.KvBits.Half, 2991, 4177, 1, 112), (saetta.KvBits.Half, 3000, 1441, 3, 36), (saetta.KvBits.Eight, 1000, 2112, 2, 50),
                                                       (saetta.KvBits.Four, 1005, 2080, 2, 50)])
def test_wide_tiles(kind, pos, tokens, kv, blocks):
    # tiles of 32 tokens, their keys in parts of `blocks` blocks: a last one with 20, 1, 5, 17, 1 tokens (its second half of no place, or of one
    # token), and whole; parts that begin between a tile's tokens; 1 and 3 kv heads
    call, out, p, want = chunk(kind, pos, tokens, kv)
    size, plain = saetta.attention_prefill.workspace_bytes(p), -(-(pos + tokens) // 32) * kv * 32768 + 256
    ws = torch.full((size,), 0xff, dtype=torch.uint8, device="cuda")
    out.fill_(float("nan"))
    assert call(ws.data_ptr(), size) == 0, saetta.ffi.lib().saetta_last_error()
    # a tile leaves the parts that its last token sees: the second half of a wide one is in the same as the first
    begins, tile = torch.arange(0, pos + tokens, 32 * blocks), torch.arange(-(-tokens // 16))
    left = lambda tq: pos + torch.clamp((16 * tile // tq + 1) * tq, max=tokens)[None] > begins[:, None]  # noqa: E731
    assert size == plain + len(begins) * len(tile) * kv * (PART_O + PART_ML)
    assert torch.equal(parts_written(ws, plain, tokens, kv, len(begins)).cpu(), left(32))
    assert torch.equal(left(32), left(16)) == (pos in (9990, 3000))  # (elsewhere tiles of 16 would leave fewer)
    got = out.clone()
    assert float((got.double() - want).norm() / want.norm()) < REL_RMS
    assert float((got - want).abs().max()) < MAX_ABS
    # without room for the parts: tiles of 16, the same to the rounding of the probabilities
    out.fill_(float("nan"))
    assert call(ws.data_ptr(), plain) == 0, saetta.ffi.lib().saetta_last_error()
    assert float((out.double() - want).norm() / want.norm()) < REL_RMS


@pytest.mark.parametrize("kind,pos,tokens,kv,wide,narrow", [(saetta.KvBits.Half, 5499, 1379, 3, 3, 2), (saetta.KvBits.Four, 36049, 1236, 1, 5, 3),
                                                            (saetta.KvBits.Eight, 5272, 2210, 2, 3, 2)])
def test_a_workspace_without_room_for_wide_tiles_parts(kind, pos, tokens, kv, wide, narrow):
    # wide tiles leave more parts than tiles of 16 would: in a workspace that holds only the latter's, those are made, and only
    # where it holds neither are the keys not split
    call, out, p, want = chunk(kind, pos, tokens, kv)
    plain = -(-(pos + tokens) // 32) * kv * 32768 + 256
    bytes_of = lambda n: plain + n * -(-tokens // 16) * kv * (PART_O + PART_ML)  # noqa: E731
    assert saetta.attention_prefill.workspace_bytes(p) == bytes_of(wide)
    ws = torch.empty(bytes_of(wide), dtype=torch.uint8, device="cuda")
    for size, parts in ((bytes_of(wide), wide), (bytes_of(wide) - 1, narrow), (bytes_of(narrow), narrow), (bytes_of(narrow) - 1, 0), (plain, 0)):
        ws.fill_(0xff), out.fill_(float("nan"))
        assert call(ws.data_ptr(), size) == 0, saetta.ffi.lib().saetta_last_error()
        assert float((out.double() - want).norm() / want.norm()) < REL_RMS
        assert float((out - want).abs().max()) < MAX_ABS
        assert bool((ws[plain:] == 0xff).all()) == (parts == 0)
        if parts:
            assert bool((ws[bytes_of(parts):] == 0xff).all()) and bool(parts_written(ws, plain, tokens, kv, parts)[0].all())


@pytest.mark.parametrize("kind,pos,tokens,kv", [(saetta.KvBits.Half, 2097, 2148, 2), (saetta.KvBits.Four, 5499, 1379, 3)])
def test_calls_without_room_for_their_parts(kind, pos, tokens, kv, monkeypatch):
    # 151 and 125 MB of workspace are wanted and 9 and 21 needed: a call that makes its own, and AttGemm, do with what there is
    _, out, p, want = chunk(kind, pos, tokens, kv)
    gen, heads, n = torch.Generator(device="cuda").manual_seed(pos + tokens), 8 * kv, pos + tokens  # (chunk's own inputs again)
    k, v = (torch.randn(n, kv * D, generator=gen, device="cuda") for _ in range(2))
    q16, qg = torch.randn(tokens, heads, D, generator=gen, device="cuda").half(), torch.randn(tokens, heads, 2 * D, generator=gen, device="cuda")
    if kind is saetta.KvBits.Half:
        keys, values = k.half(), v.half()
        flash = lambda: saetta.attention_prefill.encode(saetta.attention_prefill.DEFAULT, q16, keys, values, qg, out, p)  # noqa: E731
    else:
        keys, values = (saetta.QuantRows(kind, kv * D, n) for _ in range(2))
        keys.encode(k.view(-1), 0, n), values.encode(v.view(-1), 0, n)
        flash = lambda: saetta.attention_prefill.encode_quant(q16, keys, values, qg, out, p)  # noqa: E731
    gemm = saetta.attention_gemm.AttGemm(tokens, kv)
    quant = None if kind is saetta.KvBits.Half else (keys, values)
    empty, refused = torch.empty, []

    def limited(size, **options):
        if options.get("dtype") is torch.uint8 and size > 80e6:
            refused.append(size)
            raise torch.OutOfMemoryError
        return empty(size, **options)

    monkeypatch.setattr(torch, "empty", limited)
    encode = lambda: gemm.encode(q16, keys, values, quant, qg, out, p)  # noqa: E731
    for call in (flash, encode, encode):
        out.fill_(float("nan"))
        call()
        assert float((out.double() - want).norm() / want.norm()) < REL_RMS
    assert refused == [saetta.attention_prefill.workspace_bytes(p), gemm.workspace_bytes(p)]
    gemm.stages = 3  # the passes cannot do with less
    for _ in range(2):
        with pytest.raises(torch.OutOfMemoryError):
            encode()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("scale", [1e-3, 300.0])
def test_short_chunks_of_small_and_large_values(kind, scale):
    # Codes become halves in packed half arithmetic, with scales below the least normal half (8-bit: 1e-3 * 8 / 255 = 3e-5)
    # and values past 1000 as well.  A value is rounded to 2^-12 of itself, or to 2^-25 below 6e-5, a fiftieth of the values'
    # size here: outputs are as close, relative to theirs, as at scale 1.
    rng = np.random.default_rng(int(scale * 1000))
    pos, tokens = 300, 37
    n = pos + tokens
    k = rng.standard_normal((n, VALUES)).astype(np.float32)
    v = (scale * rng.standard_normal((n, VALUES))).astype(np.float32)
    q16 = rng.standard_normal((tokens, H, D)).astype(np.float16)
    qg = rng.standard_normal((tokens, H, 2 * D)).astype(np.float32)
    kc, vc, kf, vf = make_cache(kind, k, v, n + 7, chunk_from=pos)
    got = run(kind, q16, kc, vc, qg, pos, tokens)
    want = oracle.prefill(q16.astype(np.float32), kf, vf, pos, tokens, q_and_gate=qg, threads=8)
    assert np.isfinite(got).all()
    assert oracle.rel_rms(got, want) < REL_RMS
    assert np.abs(got - want).max() < MAX_ABS * scale
