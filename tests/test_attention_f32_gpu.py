"""The float32 matrix-core attention's ways through a batch: one or two tiles of rows a wavefront,
row blocks longest first or paired, key splits or none.  Against float64 attention; and whatever the
form, a row's sums are the same sums, so without splits the forms agree to the last bit."""

import pytest
import torch

from litellmengine_amd.csrc.ops import default_ops

pytestmark = pytest.mark.gpu
PAGE = 32


def batch(lens, past, nq, nkv, d, seed=3):
    S, N = len(lens), sum(lens)
    kv_lens = [p + n for p, n in zip(past, lens)]
    pages = [-(-k // PAGE) for k in kv_lens]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(N, nq, d, device="cuda", generator=gen)
    kv = torch.randn(sum(pages), 2, nkv, PAGE, d, device="cuda", generator=gen)
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(seed)).tolist()
    table = torch.zeros(S, max(pages), dtype=torch.int32)
    for s, n in enumerate(pages):
        table[s, :n] = torch.tensor([order.pop() for _ in range(n)])
    ints = lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    seq = [s for s, n in enumerate(lens) for _ in range(n)]
    return q, kv, table.cuda(), ints(range(S)), ints(cu), ints(kv_lens), ints(seq)


def exact(args, lens, past, nkv, window):
    q, kv, table = args[0].cpu().double(), args[1].cpu().double(), args[2].cpu()
    nq, d = q.shape[1:]
    out, at = [], 0
    for s, (n, p) in enumerate(zip(lens, past)):
        used = table[s, : -(-(p + n) // PAGE)].long()
        k = kv[used, 0].transpose(0, 1).reshape(nkv, -1, d)[:, : p + n]
        v = kv[used, 1].reshape(len(used), nkv, d, PAGE).permute(1, 0, 3, 2).reshape(nkv, -1, d)[:, : p + n]
        k, v = (x.repeat_interleave(nq // nkv, 0) for x in (k, v))
        scores = q[at : at + n].transpose(0, 1) @ k.transpose(1, 2).contiguous() * d**-0.5
        i, j = torch.arange(p, p + n)[:, None], torch.arange(p + n)[None]
        hidden = (j > i) | (j <= i - window if window else torch.zeros_like(j > i))
        out.append((scores.masked_fill(hidden, float("-inf")).softmax(-1) @ v).transpose(0, 1).reshape(n, nq * d))
        at += n
    return torch.cat(out)


def run(o, args, lens, past, window):
    d = args[0].shape[2]
    return o.paged_attention(*args, window=window, scale=d**-0.5, min_q_len=min(lens), max_q_len=max(lens),
                             max_kv_len=max(p + n for p, n in zip(past, lens)))


CASES = [
    ([129], [0], 4, 2, 128, None),  # one row over a block of two tiles
    ([97, 1, 5, 33, 64], [0, 40, 3, 70, 129], 8, 2, 128, None),  # few rows and many, blocks that are not there
    ([97, 1, 5, 33, 64], [0, 40, 3, 70, 129], 8, 2, 64, 40),  # under a window the second tile starts later
    ([31, 17], [0, 250], 3, 3, 64, None),  # one query head a kv head
    ([70], [300], 10, 2, 128, 16),  # a window of one step
]


@pytest.mark.parametrize("lens,past,nq,nkv,d,window", CASES)
@pytest.mark.parametrize("splits", [1, 3])
def test_forms_agree(lens, past, nq, nkv, d, window, splits, monkeypatch):
    o = default_ops()
    args = batch(lens, past, nq, nkv, d)
    want = exact(args, lens, past, nkv, window)
    monkeypatch.setattr(o, "f32_attention_splits", lambda *a: splits)
    got = {}
    for form in ((1, 0, 1), (1, 1, 1), (2, 0, 1), (2, 1, 1)):
        monkeypatch.setattr(o, "f32_attention_form", lambda *a, form=form: form)
        got[form] = run(o, args, lens, past, window)
        # d products and as many sums of size sqrt(d) * |q| |k| / sqrt(d), then weights that add to 1 over
        # at most 400 values of size 4: well under 400 roundings of 4 * 2^-24
        assert (got[form].cpu().double() - want).abs().max() < 400 * 4 * 2**-24
    if splits == 1:
        assert all(torch.equal(x, got[1, 0, 1]) for x in got.values())


def test_a_later_row_is_not_seen():
    """What a row may not see does not reach it, also where its neighbour tile has a step of its own:
    the last token's key and value are infinite, and every row before its 16-key step stays as it was."""
    o = default_ops()
    lens, past = [49], [0]
    args = batch(lens, past, 8, 1, 128)  # a tile: 2 tokens; the last one starts a 16-key step of its own
    o_form, o_splits = o.f32_attention_form, o.f32_attention_splits
    try:
        o.f32_attention_splits = lambda *a: 1
        o.f32_attention_form = lambda *a: (2, 0, 1)
        before = run(o, args, lens, past, None)
        page = args[2][0, 48 // PAGE].item()
        args[1][page, 0, :, 48 % PAGE] = float("inf")
        args[1][page, 1].view(1, 128, PAGE)[:, :, 48 % PAGE] = float("inf")
        after = run(o, args, lens, past, None)
    finally:
        o.f32_attention_form, o.f32_attention_splits = o_form, o_splits
    assert torch.equal(before[:48], after[:48]) and not torch.isfinite(after[48]).any()


def test_rule():
    """What the rule chooses at the edges of its ranges (256 CUs)."""
    o = default_ops()
    if o.compute_units() != 256:
        pytest.skip("the numbers are for 256 CUs")
    form = o.f32_attention_form
    assert form(2048, 32, 8, 128, True, 2048, 2048) == (2, 1, 1)
    assert form(4096, 32, 8, 128, True, 4096, 4096) == (2, 0, 1)
    assert form(1024, 32, 8, 128, True, 1024, 1024) == (1, 1, 1)
    assert form(300, 32, 8, 128, True, 300, 4300) == (2, 0, 2)
    assert form(8, 32, 8, 128, True, 1, 4300) == (1, 0, 1)
    assert form(4096, 32, 8, 256, True, 4096, 4096)[0] == 1 and form(4096, 32, 8, 128, False, 4096, 4096)[0] == 1


@pytest.mark.parametrize("nq,nkv,tokens,past,want", [(32, 8, 64, 2000, (1, 0, 1)), (32, 8, 128, 2000, (2, 0, 1)), (32, 8, 200, 2000, (2, 0, 2)),
                                                     (32, 8, 300, 4000, (2, 0, 2)), (8, 1, 128, 2000, (1, 0, 1)), (8, 1, 64, 4000, (1, 0, 1)),
                                                     (8, 1, 300, 2000, (2, 0, 1)), (16, 8, 96, 12000, (1, 0, 1)), (8, 2, 400, 12000, (2, 0, 2))])
def test_splits_of_two_tiles_have_enough_keys(nq, nkv, tokens, past, want):
    """Two tiles in splits of a few steps took up to 1.4 times as long as one tile (8 / 1 heads, 128 tokens behind 2000: 40.4 and 28.9 us)."""
    o = default_ops()
    if o.compute_units() != 256:
        pytest.skip("the form follows the number of CUs")
    assert o.f32_attention_form(tokens, nq, nkv, 128, True, tokens, past + tokens) == want
    args = batch([tokens], [past], nq, nkv, 64)
    got = run(o, args, [tokens], [past], None)
    # a row's sums are chains of at most (12000 + 400) / 16 steps, rescaled and rounded, of weights that add to 1 over values up to 4
    # (and the weights are off by the scores' roundings): under 1000 roundings of 4 * 2^-24
    assert (got.cpu().double() - exact(args, [tokens], [past], nkv, None)).abs().max() < 1000 * 4 * 2**-24


def test_few_second_blocks_are_not_paired():
    """Up to four thirds of a block a CU the longest go first (600 and 60 tokens of 32 / 8 heads, a window of 256: 47 us, paired 68)."""
    o = default_ops()
    if o.compute_units() != 256:
        pytest.skip("the form follows the number of CUs")
    form = lambda n, nq: o.f32_attention_form(n, nq, 8, 128, True, n, n)
    assert form(660, 32) == form(1300, 16) == form(514, 32) == (1, 0, 1) and form(700, 32) == form(1024, 32) == (1, 1, 1)
    lens, past = [600, 60], [0, 0]
    args = batch(lens, past, 32, 8, 128)
    got = run(o, args, lens, past, 256)
    assert (got.cpu().double() - exact(args, lens, past, 8, 256)).abs().max() < 400 * 4 * 2**-24  # (as above)
