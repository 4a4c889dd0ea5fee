"""The library's own plans (saetta_plan_*): calls recorded between begin and end launch nothing until the plan runs,
then give what the calls give, at the position in the record that saetta_token_params_set wrote (src/plan.rs:63-168)."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_common import VALUES, dev, host, oracle, saetta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [0, 1, 3])
def test_a_recorded_call_runs_when_the_plan_does(tokens):
    lib, ffi = saetta.ffi.lib(), saetta.ffi
    x = np.random.default_rng(tokens).standard_normal((tokens + 1, VALUES)).astype(np.float32)
    data, scales, _ = oracle.quantize(x[tokens:], 8)
    rows = saetta.QuantRows(saetta.KvBits.Eight, VALUES, 8)
    plan = saetta.Plan()
    p = ffi.KvQuantParamsC(rows.per_token, rows.per_token)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.saetta_plan_begin() == 0
    assert lib.saetta_plan_begin() != 0  # one at a time
    xt = dev(x[tokens])
    for _ in range(tokens):
        assert lib.saetta_kv_quantize(s, 8, xt.data_ptr(), rows.c(), p, plan.params.data_ptr(), 0) == 0
    assert lib.saetta_kv_quantize(s, 5, xt.data_ptr(), rows.c(), p, plan.params.data_ptr(), 0) != 0  # arguments are checked here
    made = ctypes.c_void_p(lib.saetta_plan_end())
    assert made and not lib.saetta_plan_end()
    assert lib.saetta_plan_launches(made) == tokens
    assert not host(rows.data).any()
    for pos in (2, 7):
        plan.set_params(saetta.TokenParams(0, pos))
        assert lib.saetta_plan_run(s, made) == 0
        if tokens:
            words = data.size
            assert np.array_equal(host(rows.data)[pos * words:(pos + 1) * words].view(np.uint32), data.reshape(-1))
            assert np.array_equal(host(rows.scales)[pos * 8:(pos + 1) * 8].view(np.uint16), scales.reshape(-1))
    assert host(rows.data)[:2 * data.size].any() == False  # noqa: E712
    lib.saetta_plan_free(made)


def test_a_plan_of_calls_and_other_ops_keeps_their_order():
    x = torch.ones(VALUES, device="cuda")
    rows = saetta.QuantRows(saetta.KvBits.Eight, VALUES, 2)
    seen = []
    plan = saetta.Plan()
    rows.record(plan, x)
    plan.op("look", lambda s: seen.append(rows.biases.clone()))
    plan.op("double", lambda s: x.mul_(2.0))
    rows.record(plan, x)
    plan.op("look", lambda s: seen.append(rows.biases.clone()))
    plan.set_params(saetta.TokenParams(0, 1))
    built = plan.build()
    for run in range(2):
        built.run()
    got = [float(t[8]) for t in seen]
    assert got == [1.0, 2.0, 2.0, 4.0]


def test_a_plan_recorded_on_a_busy_stream_first_runs_on_another():
    # The plan's own buffers (the position's record, the counters of the one-launch DeltaNet token) are zero whichever
    # stream reads them first: the fills must not stand behind the work of the stream the plan was recorded on.
    k_heads, v_heads, v_dim, conv = 16, 32, 128, 4
    channels = 2 * k_heads * 128 + v_heads * v_dim
    gen = torch.Generator(device="cuda").manual_seed(3)
    made = [torch.randn(n, generator=gen, device="cuda") for n in (channels, channels * conv, 3 * channels, v_heads, v_heads, v_heads, v_heads,
                                                                 v_heads * v_dim * 128, v_heads * v_dim, v_dim, v_heads * v_dim)]
    x, state = made[0], made[2]
    before = state.clone()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        used = [torch.full((n,), 7, dtype=torch.int32, device="cuda") for n in (4, 4096)]
        del used  # (memory that holds something else, for the allocator to hand out again)
        big = torch.ones(8192, 8192, device="cuda")
        for _ in range(20):
            big = big @ big  # a few ms at least
        plan = saetta.Plan()
        saetta.deltanet_token(plan, *made, k_heads, v_heads, v_dim, conv, 1e-6)
    built = plan.build()
    with torch.cuda.stream(b):
        params = plan.params.clone()
        built.run()
    torch.cuda.synchronize()
    assert not host(params).any()
    assert torch.equal(state, torch.cat([before[channels:], x]))


def test_build_records_and_refuses_what_a_call_does_not_accept():
    rows = saetta.QuantRows(saetta.KvBits.Eight, VALUES, 8)
    x = torch.ones(VALUES, device="cuda")
    plan = saetta.Plan()
    for _ in range(3):
        rows.record(plan, x)
    (part,) = plan.build()._parts
    assert saetta.ffi.lib().saetta_plan_launches(part.plan) == 3  # (before any run)
    y = torch.zeros(4096, device="cuda")
    saetta.deltanet_step(plan, *[y] * 11, 2, 3, 8, 1e-6)  # three value heads over two key heads
    with pytest.raises(saetta.ffi.SaettaError, match="value heads"):
        plan.build()
    assert saetta.ffi.lib().saetta_plan_begin() == 0  # (the recording that failed is over)
    saetta.ffi.lib().saetta_plan_free(saetta.ffi.lib().saetta_plan_end())
    assert not host(rows.data).any()
