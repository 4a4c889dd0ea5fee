"""Gated DeltaNet decode step on the GPU (deltanet_conv + deltanet_step) against the oracle.

The oracle is pinned by the reference's MLX golden vectors at dims 8 (tests/test_oracle_deltanet.py);
here the kernels run the real shape (16 key / 32 value heads of 128, conv kernel 4) and
smaller value dims over several tokens, with the states carried along on both sides.  Dot products
are summed in another order than on the CPU: 2e-5 relative on y and the state, 2e-6 on the conv.
"""
import numpy as np
import pytest
import torch

from gpu_common import dev, host, oracle, saetta

pytestmark = pytest.mark.gpu
K_DIM = 128


def run_tokens(k_heads, v_heads, v_dim, kernel, tokens, seed):
    rng = np.random.default_rng(seed)
    eps = 1e-6
    key, val = k_heads * K_DIM, v_heads * v_dim
    channels = 2 * key + val
    conv_w = (0.5 * rng.standard_normal((channels, kernel))).astype(np.float32)
    a_log = rng.uniform(-1, 1, v_heads).astype(np.float32)
    dt_bias = rng.standard_normal(v_heads).astype(np.float32)
    norm = (1 + 0.1 * rng.standard_normal(v_dim)).astype(np.float32)
    conv_cpu = np.zeros((kernel - 1, channels), np.float32)
    state_cpu = np.zeros(v_heads * v_dim * K_DIM, np.float32)
    conv_gpu, state_gpu = dev(conv_cpu.copy()), dev(state_cpu.copy())
    mixed, y = torch.empty(channels, device="cuda"), torch.empty(val, device="cuda")
    x_d, z_d = torch.empty(channels, device="cuda"), torch.empty(val, device="cuda")
    a_d, b_d = torch.empty(v_heads, device="cuda"), torch.empty(v_heads, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_conv(plan, x_d, dev(conv_w), conv_gpu, mixed, channels, kernel)
    saetta.deltanet_step(plan, mixed[:key], mixed[key:2 * key], mixed[2 * key:], a_d, b_d, dev(a_log), dev(dt_bias),
                         state_gpu, z_d, dev(norm), y, k_heads, v_heads, v_dim, eps)
    assert [n for n, _ in plan.ops] == ["deltanet_conv", "deltanet_step"]
    built = plan.build()
    for t in range(tokens):
        x = rng.standard_normal(channels).astype(np.float32)
        z = rng.standard_normal(val).astype(np.float32)
        a = rng.standard_normal(v_heads).astype(np.float32)
        b = rng.standard_normal(v_heads).astype(np.float32)
        for dst, src in ((x_d, x), (z_d, z), (a_d, a), (b_d, b)):
            dst.copy_(torch.from_numpy(src))
        built.run()
        want_mixed = oracle.deltanet_conv(conv_w, x, conv_cpu, kernel)
        want_y = oracle.deltanet_step(want_mixed[:key], want_mixed[key:2 * key], want_mixed[2 * key:], a, b, a_log,
                                      dt_bias, state_cpu, z, norm, k_heads, v_heads, K_DIM, v_dim, eps)
        assert np.abs(host(mixed) - want_mixed).max() <= 2e-6 * max(1.0, np.abs(want_mixed).max()), t
        assert np.array_equal(host(conv_gpu).reshape(kernel - 1, channels), conv_cpu), t
        assert np.abs(host(y) - want_y).max() <= 2e-5 * max(1.0, np.abs(want_y).max()), t
        assert np.abs(host(state_gpu) - state_cpu).max() <= 2e-5 * max(1.0, np.abs(state_cpu).max()), t


def test_real_shape_over_tokens():
    run_tokens(16, 32, 128, 4, 6, seed=1)


@pytest.mark.parametrize("v_dim", [1, 24, 33, 200, 256])
def test_other_value_dims(v_dim):
    run_tokens(2, 4, v_dim, 4, 3, seed=v_dim)


def test_step_with_vectors_apart():
    # q, k and v in buffers of their own take deltanet_step_kernel (one workgroup per value head);
    # as slices of the conv's output (the tests above) the same call runs the rows kernels.
    rng = np.random.default_rng(11)
    k_heads, v_heads, v_dim, eps = 16, 32, 128, 1e-6
    key, val = k_heads * K_DIM, v_heads * v_dim
    a_log = rng.uniform(-1, 1, v_heads).astype(np.float32)
    dt_bias = rng.standard_normal(v_heads).astype(np.float32)
    norm = (1 + 0.1 * rng.standard_normal(v_dim)).astype(np.float32)
    state_cpu = (0.1 * rng.standard_normal(v_heads * v_dim * K_DIM)).astype(np.float32)
    state_gpu = dev(state_cpu.copy())
    q, k = rng.standard_normal(key).astype(np.float32), rng.standard_normal(key).astype(np.float32)
    v, z = rng.standard_normal(val).astype(np.float32), rng.standard_normal(val).astype(np.float32)
    a, b = rng.standard_normal(v_heads).astype(np.float32), rng.standard_normal(v_heads).astype(np.float32)
    y = torch.empty(val, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_step(plan, dev(q), dev(k), dev(v), dev(a), dev(b), dev(a_log), dev(dt_bias), state_gpu, dev(z),
                         dev(norm), y, k_heads, v_heads, v_dim, eps)
    plan.build().run()
    want_y = oracle.deltanet_step(q, k, v, a, b, a_log, dt_bias, state_cpu, z, norm, k_heads, v_heads, K_DIM, v_dim, eps)
    assert np.abs(host(y) - want_y).max() <= 2e-5 * max(1.0, np.abs(want_y).max())
    assert np.abs(host(state_gpu) - state_cpu).max() <= 2e-5 * max(1.0, np.abs(state_cpu).max())


def test_conv_kernel_sizes_and_rejections():
    run_tokens(1, 1, 16, 2, 3, seed=5)
    run_tokens(1, 2, 16, 7, 9, seed=6)
    z = torch.zeros(4096, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_step(plan, z, z, z, z, z, z, z, torch.zeros(3 * 8 * 128, device="cuda"), z, z, z, 2, 3, 8, 1e-6)
    with pytest.raises(saetta.ffi.SaettaError, match="value heads"):
        plan.build().run()
    with pytest.raises(ValueError):
        saetta.deltanet_step(saetta.Plan(), z, z, z, z, z, z, z, torch.zeros(10, device="cuda"), z, z, z, 2, 4, 8, 1e-6)


@pytest.mark.parametrize("k_heads,v_heads,v_dim,kernel", [(16, 32, 128, 4), (2, 4, 24, 4), (1, 2, 200, 7), (1, 1, 1, 2)])
def test_token_call_matches_conv_then_step(k_heads, v_heads, v_dim, kernel):
    # saetta_deltanet_token: the same token step in two launches with the rows spread over more
    # workgroups; against the oracle over several tokens, states carried on both sides.
    rng = np.random.default_rng(v_dim + kernel)
    eps = 1e-6
    key, val = k_heads * K_DIM, v_heads * v_dim
    channels = 2 * key + val
    conv_w = (0.5 * rng.standard_normal((channels, kernel))).astype(np.float32)
    a_log = rng.uniform(-1, 1, v_heads).astype(np.float32)
    dt_bias = rng.standard_normal(v_heads).astype(np.float32)
    norm = (1 + 0.1 * rng.standard_normal(v_dim)).astype(np.float32)
    conv_cpu = np.zeros((kernel - 1, channels), np.float32)
    state_cpu = np.zeros(v_heads * v_dim * K_DIM, np.float32)
    conv_gpu, state_gpu = dev(conv_cpu.copy()), dev(state_cpu.copy())
    x_d, z_d, y = torch.empty(channels, device="cuda"), torch.empty(val, device="cuda"), torch.empty(val, device="cuda")
    a_d, b_d = torch.empty(v_heads, device="cuda"), torch.empty(v_heads, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_token(plan, x_d, dev(conv_w), conv_gpu, a_d, b_d, dev(a_log), dev(dt_bias), state_gpu, z_d,
                          dev(norm), y, k_heads, v_heads, v_dim, kernel, eps)
    built = plan.build(graph=True)
    for t in range(5):
        x = rng.standard_normal(channels).astype(np.float32)
        z = rng.standard_normal(val).astype(np.float32)
        a = rng.standard_normal(v_heads).astype(np.float32)
        b = rng.standard_normal(v_heads).astype(np.float32)
        for dst, src in ((x_d, x), (z_d, z), (a_d, a), (b_d, b)):
            dst.copy_(torch.from_numpy(src))
        built.run()
        m = oracle.deltanet_conv(conv_w, x, conv_cpu, kernel)
        want_y = oracle.deltanet_step(m[:key], m[key:2 * key], m[2 * key:], a, b, a_log, dt_bias, state_cpu, z, norm,
                                      k_heads, v_heads, K_DIM, v_dim, eps)
        assert np.array_equal(host(conv_gpu).reshape(kernel - 1, channels), conv_cpu), t
        assert np.abs(host(y) - want_y).max() <= 2e-5 * max(1.0, np.abs(want_y).max()), t
        assert np.abs(host(state_gpu) - state_cpu).max() <= 2e-5 * max(1.0, np.abs(state_cpu).max()), t


@pytest.mark.parametrize("rows", [1, 4])
def test_norm_of_outputs_whose_mean_square_is_below_the_normal_numbers(rows):
    # values of 1e-18 and no eps: outputs whose mean square is 1e-42 to 1e-38, which the hardware's reciprocal root takes for 0;
    # against the same in 64 bits, to half a step of 2^-149 of the 128 squares and of their mean
    rng = np.random.default_rng(rows)
    k_heads, v_heads, v_dim = 2, 4, 128
    key, val = k_heads * K_DIM, v_heads * v_dim
    x = rng.standard_normal((rows, 2 * key + val)).astype(np.float32)
    x[:, 2 * key:] *= 5e-18
    z, a, b = (rng.standard_normal((rows, n)).astype(np.float32) for n in (val, v_heads, v_heads))
    a_log, dt_bias, norm = rng.uniform(-1, 1, v_heads).astype(np.float32), rng.standard_normal(v_heads).astype(np.float32), np.ones(v_dim, np.float32)
    w = np.zeros((x.shape[1], 4), np.float32)
    w[:, 3] = 1
    conv, state, y = torch.zeros(3, x.shape[1], device="cuda"), torch.zeros(val * K_DIM, device="cuda"), torch.empty(rows, val, device="cuda")
    buffers = (dev(x), dev(w), conv, dev(a), dev(b), dev(a_log), dev(dt_bias), state, dev(z), dev(norm), y)
    plan = saetta.Plan()
    if rows == 1:
        saetta.deltanet_token(plan, *buffers, k_heads, v_heads, v_dim, 4, 0.0)
    else:
        saetta.deltanet_rows_fused(plan, *buffers, k_heads, v_heads, v_dim, 4, rows, 0.0)
    plan.build().run()
    sigmoid = lambda u: 1 / (1 + np.exp(-u.astype(np.float64)))  # noqa: E731
    m, s = x * sigmoid(x), np.zeros((v_heads, v_dim, K_DIM))
    for t in range(rows):
        for h in range(v_heads):
            q, k = (m[t, o + h // 2 * K_DIM:o + (h // 2 + 1) * K_DIM] for o in (0, key))
            q, k = q / np.linalg.norm(q) / np.sqrt(K_DIM), k / np.linalg.norm(k)
            g = np.exp(-np.exp(np.float64(a_log[h])) * np.logaddexp(0, np.float64(a[t, h]) + dt_bias[h]))
            v = m[t, 2 * key + h * v_dim:2 * key + (h + 1) * v_dim]
            s[h] = g * s[h]
            s[h] += np.outer((v - s[h] @ k) * sigmoid(b[t, h:h + 1]), k)
            o = s[h] @ q
            want = o / np.sqrt(np.mean(o * o)) * z[t, h * v_dim:(h + 1) * v_dim] * sigmoid(z[t, h * v_dim:(h + 1) * v_dim])
            got = host(y)[t, h * v_dim:(h + 1) * v_dim]
            assert np.mean(o * o) < 2.0 ** -120 and np.abs(got - want).max() < (1e-5 + 2.0 ** -149 / np.mean(o * o)) * np.abs(want).max(), (t, h)


def test_activation_over_the_whole_range():
    # the conv with a last tap of one is its activation, x / (1 + e^-x): two ulps of f32 (below 2^-119 see the next test), and the
    # limits
    x = np.concatenate([np.linspace(-100, 100, 2001), -np.logspace(-30, 2, 500), np.logspace(-30, 38, 500), [0.0, -87.0, -88.0, -89.0, -1e30]]).astype(np.float32)
    special = np.array([np.inf, -np.inf, np.nan], np.float32)
    xs = np.concatenate([x, special])
    w = np.zeros((xs.size, 4), np.float32)
    w[:, 3] = 1
    state, out = torch.zeros(3, xs.size, device="cuda"), torch.empty(xs.size, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_conv(plan, dev(xs), dev(w), state, out, xs.size, 4)
    plan.build().run()
    got, x64 = host(out), x.astype(np.float64)
    with np.errstate(over="ignore"):
        want = x64 / (1 + np.exp(-x64))
    assert (np.abs(got[:x.size] - want) <= 2.4e-7 * np.abs(want) + 2.0 ** -119).all()
    assert got[-3] == np.inf and np.isnan(got[-1]) and not got[-2] > 0


def test_activation_down_to_the_end_of_its_exponential():
    # up to where e^-x leaves f32 (x = -88.7228) two ulps, whatever its reciprocal; zero or the number it is from there on
    x = -np.concatenate([np.linspace(44, 130, 8001), [44.361419, 87.336544, 88.02969, 88.7227, 103.97208, 1e3, 1e30, 3.4e38]]).astype(np.float32)
    w = np.zeros((x.size, 4), np.float32)
    w[:, 3] = 1
    state, out = torch.zeros(3, x.size, device="cuda"), torch.empty(x.size, device="cuda")
    plan = saetta.Plan()
    saetta.deltanet_conv(plan, dev(x), dev(w), state, out, x.size, 4)
    plan.build().run()
    x64 = x.astype(np.float64)
    with np.errstate(over="ignore"):
        want = x64 / (1 + np.exp(-x64))
    allowed = np.where(x64 > -88.7228, 2.4e-7, 1.0) * np.abs(want) + 2.0 ** -149
    worst = (np.abs(host(out) - want) - allowed).argmax()
    assert abs(host(out)[worst] - want[worst]) <= allowed[worst], (x[worst], host(out)[worst], want[worst])
