"""float32 attention of many rows with its operands in three bfloat16 parts: blocks of 128 rows in one part or several, against float64
attention at the edges of blocks, steps and parts; what is not finite; and the number of workgroups that a launch is given."""
import math

import pytest
import torch

from tests.test_attention_f32_gpu import batch, exact, run

CASES = [
    ([129], [0], 4, 2, None),  # a block of two rows behind whole ones
    ([97, 1, 5, 33, 64], [0, 40, 3, 70, 129], 8, 2, None),  # few rows and many in one launch
    ([31, 17, 200], [0, 250, 31], 3, 3, None),  # one query head a kv head: a block is 128 tokens
    ([70], [300], 10, 2, 16),  # a window of half a step, groups of five (a block ends inside a token)
    ([97, 1, 140], [60, 90, 10], 8, 2, 40),
    ([1, 33], [700, 480], 8, 1, None),
]


def in_parts(o, monkeypatch, steps):
    monkeypatch.setattr(o, "f32_attention_part_steps", lambda *a: steps)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,past,nq,nkv,window", CASES)
@pytest.mark.parametrize("steps", [1, 3, 4, 1 << 20])
def test_against_float64(lens, past, nq, nkv, window, steps, monkeypatch):
    from litellmengine_amd.csrc.ops import default_ops

    o = default_ops()
    args = batch(lens, past, nq, nkv, 128)
    want = exact(args, lens, past, nkv, window)
    monkeypatch.setattr(o, "f32_attention_splits", lambda *a: 1)  # (a row's keys in one chain of sums, which is as long as any here)
    in_parts(o, monkeypatch, 0)
    before = run(o, args, lens, past, window)
    in_parts(o, monkeypatch, steps)
    got = run(o, args, lens, past, window)
    # 128 products and as many sums of size |q| |k| / sqrt(128), then weights that add to 1 over at most 733 values of size 4: well
    # under 400 roundings of 4 * 2^-24, as for the float32 instruction; and all together no further off than it is (a quarter less, measured)
    off = lambda x: x.cpu().double() - want
    assert off(got).abs().max() < 400 * 4 * 2**-24
    assert off(got).norm() <= 1.05 * off(before).norm()


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 1 << 20])
def test_a_sink_is_a_place_without_a_value(steps, monkeypatch):
    from litellmengine_amd.csrc.ops import default_ops

    o, (nq, nkv) = default_ops(), (8, 2)
    args = batch([40, 90], [100, 0], nq, nkv, 128)
    sinks = torch.linspace(-2.0, 6.0, nq, device="cuda")
    call = lambda: o.paged_attention(*args, window=None, scale=128**-0.5, min_q_len=40, max_q_len=90, max_kv_len=140, sinks=sinks)
    before = call()
    in_parts(o, monkeypatch, steps)
    assert (call() - before).abs().max() < 400 * 4 * 2**-24 * 2


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 3, 1 << 20])
@pytest.mark.parametrize("value", [math.inf, math.nan, 3.4e38])
def test_what_is_not_finite(steps, value, monkeypatch):
    """Numbers without parts (the largest ones round to infinity in bfloat16) where the float32 instruction has them: rows that
    see them have its result, rows that do not are as they were."""
    from litellmengine_amd.csrc.ops import default_ops

    o, lens, past = default_ops(), [200], [50]
    q, kv, *rest = batch(lens, past, 8, 2, 128)
    page = lambda key: rest[0][0, key // 32].item()
    in_parts(o, monkeypatch, steps)
    clean = run(o, (q, kv, *rest), lens, past, None)
    kv[page(201), 1].view(2, 128, 32)[:, 5, 201 % 32] = value  # an element of a value, seen from token 151 on
    kv[page(230), 0, 1, 230 % 32, 7] = value  # one of a key, of the second head
    q[190, 2, 3] = value
    got = run(o, (q, kv, *rest), lens, past, None)
    in_parts(o, monkeypatch, 0)
    monkeypatch.setattr(o, "f32_attention_splits", lambda *a: 1)
    monkeypatch.setattr(o, "f32_attention_form", lambda *a: (2, 0, 1))  # (32 rows a wavefront, too: those beside a row that sees an infinite value get 0 times it)
    want = run(o, (q, kv, *rest), lens, past, None)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    assert (((got - want).abs() / want.abs().clamp(min=1.0))[fine] < 400 * 4 * 2**-24 * 2).all()
    assert torch.equal(got[:128], clean[:128])  # (blocks of 32 tokens: a block whose rows see none of them)


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [3, 1 << 20])
@pytest.mark.parametrize("q_size", [1.0, 1e-36, 1e-34, 1e-32, 1e30, 1e34, 1e36])
@pytest.mark.parametrize("v_size", [1.0, 1e-28, 1e-31, 1e-34, 1e-36])
def test_small_numbers(steps, q_size, v_size, monkeypatch):
    """Numbers whose last parts are below what bfloat16 has: no further off than with the float32 instruction, which takes such rows; keys are as
    small as q is large.  Some elements are 0, which is no small number."""
    from litellmengine_amd.csrc.ops import default_ops

    o, lens, past = default_ops(), [200], [50]
    q, kv, *rest = batch(lens, past, 8, 2, 128)
    q *= q_size
    kv[:, 0] /= q_size
    kv[:, 1] *= v_size
    q[:, :, 5], kv[:, 1].view(-1, 2, 128, 32)[:, :, 9] = 0.0, 0.0
    args = (q, kv, *rest)
    want = exact(args, lens, past, 2, None)
    monkeypatch.setattr(o, "f32_attention_splits", lambda *a: 1)
    in_parts(o, monkeypatch, 0)
    before = run(o, args, lens, past, None)
    in_parts(o, monkeypatch, steps)
    got = run(o, args, lens, past, None)
    off = lambda x: (x.cpu().double() - want).norm()
    assert off(got) <= 1.05 * off(before)


@pytest.mark.gpu
@pytest.mark.parametrize("steps", [1, 3, 1 << 20])
@pytest.mark.parametrize("value", [math.inf, 3e17])
@pytest.mark.parametrize("sink", [False, True])
def test_a_row_that_nothing_weighs_in(steps, value, sink, monkeypatch):
    """Every score of a row -inf, or finite and too low to count: NaN as from the float32 instruction in splits, 0 beside a sink, and never what the
    result's memory held before."""
    from litellmengine_amd.csrc import ops

    o, (nq, nkv) = ops.default_ops(), (8, 2)
    q, kv, *rest = batch([200], [50], nq, nkv, 128)
    kv[:, 0, 0, :, 3] = -1e16  # one channel of the first head's keys, all of one sign
    q[:, :4, 3] = 0.0
    q[190, 2] = 0.0
    q[190, 2, 3] = value
    sinks = torch.linspace(-2.0, 6.0, nq, device="cuda") if sink else None
    monkeypatch.setattr(ops, "_made", lambda shape, dtype, device: torch.full(shape, 5.0, dtype=dtype, device=device))
    call = lambda: o.paged_attention(q, kv, *rest, window=None, scale=128**-0.5, min_q_len=200, max_q_len=200, max_kv_len=250, sinks=sinks)
    in_parts(o, monkeypatch, steps)
    got = call()
    in_parts(o, monkeypatch, 0)
    monkeypatch.setattr(o, "f32_attention_splits", lambda *a: 3)
    want = call()
    row = got[190, 2 * 128 : 3 * 128]
    assert bool((row == 0.0).all()) if sink else bool(row.isnan().all())
    assert torch.equal(got.isnan(), want.isnan())
    assert (got - want)[want.isfinite()].abs().max() < 400 * 4 * 2**-24 * 2


@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 8, 40])
@pytest.mark.parametrize("window", [0, 16, 500])
def test_every_part_has_a_workgroup(group, window):
    """The launch's workgroups are enough for the parts of every request that fits its longest ones, and no block has more parts than the
    workspaces have places."""
    from litellmengine_amd.csrc.ops import HipOps

    for max_q in (17, 64, 129, 700, 2048):
        for max_past in (0, 15, 33, 900, 6000):
            max_kv = max_q + max_past
            span = min(max_kv, window + max_q) if window else max_kv
            for part_steps in (1, 4, 7, 32, 1 << 20):
                most, places = HipOps.f32_attention_parts(part_steps, max_q * group, group, max_kv, span)
                for q_len, past in ((max_q, max_past), (max_q, 0), (max(1, max_q // 3), max_kv - max(1, max_q // 3)), (max_q - 1, max_past)):
                    rows, total = q_len * group, 0
                    if rows <= 16:
                        total = most
                    else:
                        for r0 in range(0, rows, 128):  # (as the kernel cuts a block)
                            hi = past + (min(rows, r0 + 128) - 1) // group
                            lo = max(0, past + r0 // group - window + 1) if window else 0
                            total += min(most, -(-(hi // 32 + 1 - lo // 32) // part_steps))
                    assert total <= places, (group, window, max_q, max_past, part_steps, q_len, past)
