"""A plan's token step: record_store, then decode or verify attention on the same buffers, which the library's plan
makes one launch less (the partial stage takes the store in, the new tokens get a partial result of their own).
Every result against the same ops launched one by one: the outputs to the decode tests' bound, q to rounding, what is
stored bit for bit."""
import numpy as np
import pytest
import torch

from gpu_common import D, H, KV, VALUES, dev, host, oracle, saetta

pytestmark = pytest.mark.gpu
KINDS = [saetta.KvBits.Half, saetta.KvBits.Eight, saetta.KvBits.Four]
PREP = saetta.PrepParams(H, KV, D, 64, 1e7, 1e-6)


def poison(rows):
    rows.fill_(float("nan") if rows.dtype == torch.float16 else -1)


class Step:
    def __init__(self, kind, capacity, rows, seed, rope_dims=64, lay=lambda step: None, theta=1e7, eps=1e-6):
        rng = np.random.default_rng(seed)
        self.rows, self.kind = rows, kind
        self.qg = dev(rng.standard_normal((rows, H, 2 * D)).astype(np.float32))
        self.k, self.v = (dev(rng.standard_normal((rows, VALUES)).astype(np.float32)) for _ in range(2))
        qn, kn = (dev((1 + 0.1 * rng.standard_normal(D)).astype(np.float32)) for _ in range(2))
        self.cache = saetta.GpuKvCache.with_bits(H, KV, D, capacity, kind)
        fill = dev(oracle.noise(self.cache.capacity * VALUES, seed).reshape(self.cache.capacity, VALUES))
        if kind is saetta.KvBits.Half:
            self.cache.keys.copy_(fill.flatten().half()), self.cache.values.copy_(fill.flatten().flip(0).half())
        else:
            for c, x in zip(self.cache.quant, (fill, fill.flip(0).contiguous())):
                c.encode(x, 0, self.cache.capacity)
        keys, values = self.cache.quant or (self.cache.keys, self.cache.values)
        self.q, self.out, self.back = (torch.zeros(rows, n, device="cuda") for n in (H * D, H * D, VALUES))
        self.k0, self.v0 = self.k.clone(), self.v.clone()
        self.clean = [b.clone() for b in self.cache.buffers()]
        self.att = saetta.AttentionRows(H, KV, self.cache.capacity, rows) if rows > 1 else None
        lay(self)  # (buffers over others)
        self.k.copy_(self.k0), self.v.copy_(self.v0)
        self.plan = saetta.Plan()
        saetta.record_store(self.plan, self.qg, self.k, self.v, qn, kn, self.q, keys, values, saetta.PrepParams(H, KV, D, rope_dims, theta, eps),
                            self.cache.capacity, rows=rows, k_back=self.back)
        if rows == 1:
            (self.cache.decode.record if kind is saetta.KvBits.Half else self.cache.decode.record_quant)(
                self.plan, self.q, keys, values, self.qg, self.out)
        else:
            (self.att.record if kind is saetta.KvBits.Half else self.att.record_quant)(
                self.plan, rows, self.q, keys, values, self.qg, self.out, [self.plan.params] * rows)

    def run(self, how, position, kv_len=None):
        # every run finds the cache as it was, with NaN (codes: all ones) where the step stores: what is there behind it is its own
        for buffer, was in zip(self.cache.buffers(), self.clean):
            buffer.copy_(was)
            poison(buffer.view(self.cache.capacity, -1)[position:position + self.rows])
        params = saetta.TokenParams(0, position)
        params.kv_len = position + 1 if kv_len is None else kv_len
        self.plan.set_params(params)
        self.q.fill_(float("nan")), self.out.fill_(float("nan")), self.back.fill_(float("nan"))
        self.k.copy_(self.k0), self.v.copy_(self.v0)
        how()
        return [host(t).copy() for t in (self.out, self.q, self.back)] + [host(b).copy() for b in self.cache.buffers()]


def launches(step):
    built = step.plan.build()
    built.run()
    return sum(saetta.ffi.lib().saetta_plan_launches(p.plan) for p in built._parts)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("capacity", [512, 8192, 40960])
def test_fused_step_equals_the_ops_one_by_one(kind, capacity, rows):
    # 512: four splits, three of them the context's; 8192: 63 of 64; 40960: 127 of 128, codes through the loader kernels
    step = Step(kind, capacity, rows, seed=capacity + 10 * rows + kind.value)
    assert launches(step) == (2 if rows <= 4 else 3)  # (five rows and more keep the store a launch of its own)
    built = step.plan.build()
    cap = step.cache.capacity
    # no context; one block and less; around a block's end; several rounds; the last rows; rows that do not fit
    for position in (0, 1, 15, 16, 100, cap // 2 + 3, cap - rows, cap - 1, cap + 2):
        want = step.run(step.plan.run_serial, position)
        got = step.run(built.run, position)
        if position == 0 or position <= cap - rows:
            assert np.isfinite(got[0]).all(), position
        ok = np.isfinite(want[0])
        assert np.array_equal(ok, np.isfinite(got[0]))
        assert np.abs(got[0] - want[0])[ok].max(initial=0.0) < 2e-5, position
        assert np.array_equal(got[1], want[1]), position
        assert np.array_equal(got[2], want[2]), position
        for a, b in zip(got[3:], want[3:]):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), position


@pytest.mark.parametrize("kind,capacity,rows", [(saetta.KvBits.Eight, 24576, 4), (saetta.KvBits.Eight, 49152, 2), (saetta.KvBits.Four, 49152, 2)])
def test_fused_step_by_another_kernel_than_the_ops(kind, capacity, rows):
    # rows over codes whose line between the loader kernels lies lower with the store taken in than for attention by itself
    test_fused_step_equals_the_ops_one_by_one(kind, capacity, rows)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows", [5, 6, 7, 8])
def test_many_rows_of_a_large_cache_take_the_store_in(rows, kind):
    step = Step(kind, 49152, rows, seed=rows)
    assert launches(step) == 2
    built = step.plan.build()
    for position in (0, 1, 17, 3000, 49152 - rows, 49152 - 1, 49152 + 2):
        want, got = step.run(step.plan.run_serial, position), step.run(built.run, position)
        ok = np.isfinite(want[0])
        assert ok.all() or position > 49152 - rows
        assert np.array_equal(ok, np.isfinite(got[0])), position
        assert np.abs(got[0] - want[0])[ok].max(initial=0.0) < 2e-5, position
        for a, b in zip(got[1:], want[1:]):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), position


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("capacity", [512, 8192, 40960])
def test_a_length_of_the_callers_own(kind, capacity):
    # A decode sees min(kv_len, capacity) tokens whatever the position is: without the new one, or with rows past it.
    step = Step(kind, capacity, 1, seed=capacity + kind.value)
    assert launches(step) == 2
    built = step.plan.build()
    for position in (0, 70, capacity - 3):
        for kv_len in (1, 20, position, position + 1, position + 2, position + 75, capacity + 9):
            want, got = step.run(step.plan.run_serial, position, kv_len), step.run(built.run, position, kv_len)
            ok = np.isfinite(want[0])  # (no token at all: no number)
            assert ok.all() or kv_len == 0
            assert np.array_equal(ok, np.isfinite(got[0])), (position, kv_len)
            assert np.abs(got[0] - want[0])[ok].max(initial=0.0) < 2e-5, (position, kv_len)
            for a, b in zip(got[1:], want[1:]):
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (position, kv_len)


@pytest.mark.parametrize("capacity,rows", [(128, 1), (128, 2), (128, 5), (128, 8), (256, 2), (256, 7), (384, 3), (384, 8)])
@pytest.mark.parametrize("kind", KINDS)
def test_a_small_cache_takes_one_launch(kind, capacity, rows):
    # Up to 128 tokens (two rows 256, more 384): a workgroup per (row, q head) does the whole step.  No context, around a pass of 32
    # tokens, the last rows that fit and rows that do not; a decode also without the new token and with rows past it.
    step = Step(kind, capacity, rows, seed=500 + 10 * rows + kind.value)
    assert launches(step) == 1
    built = step.plan.build()
    for position in (0, 1, 31, 32, 33, 100, 159, 160, 161, capacity - 60, capacity - rows, capacity - 1, capacity + 2):
        if position > capacity + 2:
            continue
        for kv_len in (None,) if rows > 1 else (None, 1, position, position + 2, position + 40, 200):
            if kv_len == 0:
                continue  # (no token at all: no number)
            want = step.run(step.plan.run_serial, position, kv_len)
            got = step.run(built.run, position, kv_len)
            assert np.isfinite(want[0]).all() and np.isfinite(got[0]).all(), (position, kv_len)
            assert np.abs(got[0] - want[0]).max() < 2e-5, (position, kv_len)
            for x, y in zip(got[1:], want[1:]):
                assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (position, kv_len)


@pytest.mark.parametrize("kind", KINDS)
def test_one_launch_where_its_buffers_lie_apart(kind):
    def result_over_the_key(step):
        step.k = step.out[:, :VALUES].view(step.rows, VALUES)
    for lay in (key_in_place, result_over_the_key):
        check_laid_over(Step(kind, 128, 1, seed=70 + kind.value, lay=lay), (0, 50, 127))


@pytest.mark.parametrize("capacity,rows", [(128, 1), (128, 3), (256, 2), (384, 3), (384, 8)])
@pytest.mark.parametrize("kind", KINDS)
def test_one_launch_drops_what_is_not_in_use(kind, capacity, rows):
    # NaN and codes of all ones in the rows past the context; a decode also without its last tokens and with rows past the new one
    step = Step(kind, capacity, rows, seed=90 + kind.value)
    assert launches(step) == 1
    built, clean = step.plan.build(), step.clean
    for kv_len in (None,) if rows > 1 else (None, 20, 38, 39, 75):
        step.clean = [b.clone() for b in clean]
        for buffer in step.clean:
            poison(buffer.view(capacity, -1)[kv_len or 37:])
        want, got = step.run(step.plan.run_serial, 37, kv_len), step.run(built.run, 37, kv_len)
        assert np.isfinite(got[0]).all() and np.abs(got[0] - want[0]).max() < 2e-5, kv_len
        for x, y in zip(got[1:], want[1:]):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), kv_len


@pytest.mark.parametrize("capacity,rows", [(128, 1), (256, 2), (384, 8)])
@pytest.mark.parametrize("kind", KINDS)
def test_one_launch_against_64_bits(kind, capacity, rows):
    # A few channels 8 times as large as the rest.  A score's terms (codes with the bias not yet taken off) add up to some 70 in units of
    # log2(e), half an ulp of which is 4e-6: a weight of the softmax, and so an output, is off by less than that of itself.
    step = Step(kind, capacity, rows, seed=150 + kind.value)
    assert launches(step) == 1
    rng = np.random.default_rng(rows)
    fill = rng.standard_normal((2, capacity, VALUES)).astype(np.float32)
    fill[:, :, [7, 101, 230, 333, 460]] *= 8
    for x, half, quant in zip(fill, (step.cache.keys, step.cache.values), step.cache.quant or (None, None)):
        half.copy_(dev(x).flatten().half()) if quant is None else quant.encode(dev(x), 0, capacity)
    step.clean, built = [b.clone() for b in step.cache.buffers()], step.plan.build()
    for position in (5, capacity // 2 + 3, capacity - rows):
        got = step.run(built.run, position)
        held = step.cache.quant and [host(saetta.dequantize(*c.tensors(), kind)) for c in step.cache.quant]
        keys, values = (x.reshape(capacity, VALUES) for x in held or [host(c.float()) for c in (step.cache.keys, step.cache.values)])
        want = oracle.rows(got[1], keys, values, position, rows, q_and_gate=host(step.qg), threads=8, f64=True).reshape(got[0].shape)
        error = np.linalg.norm(got[0] - want) / np.linalg.norm(want)
        assert error < 4e-6, (position, error)


@pytest.mark.parametrize("capacity,rows", [(128, 1), (128, 3), (256, 2), (384, 8)])
@pytest.mark.parametrize("kind", KINDS)
def test_one_launch_hides_no_nan(kind, capacity, rows):
    # NaN in one token that is in use, for one kv head: in its key (every output of its heads), in its value (dims of them), in
    # the new key, in the new value; the same outputs are numbers as by three launches.
    step = Step(kind, capacity, rows, seed=110 + rows + kind.value)
    assert launches(step) == 1
    built, position = step.plan.build(), capacity - 30
    spots = [(i, token) for i, b in enumerate(step.clean) if b.dtype == torch.float16 for token in (0, 33, position - 1)]  # halves, or scales and biases
    for spot, token in spots + [(x, position) for x in (step.k0, step.v0) if kind is saetta.KvBits.Half]:
        row = step.clean[spot].view(capacity, KV, -1)[token, 1] if isinstance(spot, int) else spot[0, D:]
        at, was = row.numel() // 4 + 1, row.clone()
        row[at] = float("nan")
        want, got = step.run(step.plan.run_serial, position), step.run(built.run, position)
        row.copy_(was)
        ok = np.isfinite(want[0]).reshape(rows, KV, -1)
        assert ok[:, 0].all() and not ok[:, 1].all(), (token, at)
        assert np.array_equal(ok, np.isfinite(got[0]).reshape(ok.shape)), (token, at)


@pytest.mark.parametrize("capacity,rows,count", [(128, 1, 1), (128, 8, 1), (256, 2, 1), (384, 3, 1), (512, 1, 2), (8192, 4, 2), (40960, 1, 2), (40960, 3, 2), (49152, 6, 2)])
@pytest.mark.parametrize("kind", KINDS)
def test_a_second_merge(kind, capacity, rows, count):
    # another reduce stage over the step's scratch, with a gate of its own, recorded behind it; and one more
    step = Step(kind, capacity, rows, seed=130 + rows + kind.value)
    att = step.att or step.cache.decode
    gates, out = dev(np.random.default_rng(rows).standard_normal((rows, H, 2 * D)).astype(np.float32)), torch.zeros(rows, H * D, device="cuda")
    keys, values = step.cache.quant or (step.cache.keys, step.cache.values)
    record = att.record if kind is saetta.KvBits.Half else att.record_quant
    if rows == 1:
        record(step.plan, step.q, keys, values, gates, out)
    else:
        record(step.plan, rows, step.q, keys, values, gates, out, [step.plan.params] * rows)
    step.plan.ops.pop(-2)  # (its partial stage)
    step.plan.ops.append(step.plan.ops[-1])
    assert launches(step) == count + 2
    built = step.plan.build()
    for position in (0, 50, capacity - rows):
        step.run(step.plan.run_serial, position)
        want = host(out).copy()
        for t in (out, att.part_o, att.part_ml):
            t.fill_(float("nan"))
        step.run(built.run, position)
        assert np.abs(host(out) - want).max() < 2e-5, position


def check_laid_over(step, positions):
    """A step with buffers over each other keeps its launches; outputs as the ops one by one, what is stored bit for bit."""
    assert launches(step) == 3
    built = step.plan.build()
    for position in positions:
        want, got = step.run(step.plan.run_serial, position), step.run(built.run, position)
        assert np.isfinite(got[0]).all()
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), position


def key_in_place(step):
    step.back = step.k


@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("capacity", [512, 8192, 40960])
def test_a_key_written_back_in_place(kind, capacity, rows):
    # Several workgroups make a new key; were one to write it back over what the others read, they would take a key
    # that is normed and rotated already.
    step = Step(kind, capacity, rows, seed=capacity + 7 * rows + kind.value, lay=key_in_place)
    check_laid_over(step, (100, step.cache.capacity - rows))


def partials_over_inputs(step):  # k and v, done with when the store has run, in front of part_o
    att = step.cache.decode if step.rows == 1 else step.att
    n = step.rows * VALUES
    step.k, step.v = (att.part_o[i * n:(i + 1) * n].view(step.rows, VALUES) for i in range(2))


def partial_sums_over_the_key(step):
    att = step.cache.decode if step.rows == 1 else step.att
    step.k = att.part_ml[:step.rows * VALUES].view(step.rows, VALUES)


def partials_over_the_key_written_back(step):  # which this program does not read
    att = step.cache.decode if step.rows == 1 else step.att
    step.back = att.part_o[:step.rows * VALUES].view(step.rows, VALUES)


@pytest.mark.parametrize("lay", [partials_over_inputs, partial_sums_over_the_key, partials_over_the_key_written_back])
@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("capacity", [8192, 40960])
def test_scratch_laid_over_what_is_done_with(kind, capacity, rows, lay):
    # The context's workgroups write partials while the new rows' workgroups still read k and v.
    step = Step(kind, capacity, rows, seed=capacity + 5 * rows + kind.value, lay=lay)
    check_laid_over(step, (100, step.cache.capacity - rows))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("rows", [1, 3])
def test_a_theta_below_one_keeps_its_launches(kind, rows):
    # angles of up to 2^31 times the position: the step that takes the store in is written for frequencies of at most 1
    step = Step(kind, 8192, rows, seed=rows, theta=2.0 ** -32)
    assert launches(step) == 3
    built = step.plan.build()
    for position in (0, 5, 3001, 8192 - rows):
        want, got = step.run(step.plan.run_serial, position), step.run(built.run, position)
        assert np.isfinite(want[0]).all() and np.abs(want[1]).max() < 20  # (a rotation keeps the norm)
        for a, b in zip(got, want):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), position


@pytest.mark.parametrize("rows", [1, 3])
@pytest.mark.parametrize("capacity", [8192, 40960])
def test_queries_whose_mean_square_is_below_the_normal_numbers(capacity, rows):
    # 1e-20 and no eps: the norm's root is of 1e-40 (with some 16 bits), which the hardware's reciprocal root takes for 0
    step, plain = (Step(saetta.KvBits.Eight, capacity, rows, seed=rows, eps=0.0) for _ in range(2))
    step.qg[:, :, :D] *= 1e-20
    built, ref = step.plan.build(), plain.plan.build()
    for position in (0, 100, 3001):
        got, want = step.run(built.run, position), plain.run(ref.run, position)
        assert np.isfinite(got[0]).all() and np.isfinite(got[1]).all(), position
        assert np.abs(got[0] - want[0]).max() < 1e-3 and np.abs(got[1] - want[1]).max() < 1e-3, position


def test_other_steps_keep_their_launches():
    assert launches(Step(saetta.KvBits.Eight, 256, 1, seed=1)) == 3                   # two splits only
    assert launches(Step(saetta.KvBits.Eight, 8192, 1, seed=1, rope_dims=32)) == 3    # other rotary dims
    step = Step(saetta.KvBits.Eight, 8192, 1, seed=1)
    step.plan.ops.insert(1, ("look", lambda s: None))                                # something between the store and the scores
    built = step.plan.build()
    built.run()
    assert [saetta.ffi.lib().saetta_plan_launches(p.plan) for p in built._parts if not callable(getattr(p, "__code__", None)) and hasattr(p, "plan")] == [1, 2]
