"""The delta rule in chunks of sixteen tokens (long requests where they are few) against the plain recurrence: the shortest request that goes in
chunks and the longest that is walked, last chunks of one and of fifteen tokens, value channels that are no sixteens, one decay
a head and one a channel, decays of zero and of one; more long requests than go in chunks; what is not finite."""
import math

import pytest
import torch

from .torch_ops import TorchOps

pytestmark = pytest.mark.gpu
REF = TorchOps()


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("dim,vdim,H,G,lens", [(64, 64, 2, 1, [161]), (64, 64, 4, 2, [1, 700, 160, 161, 3]), (64, 17, 3, 3, [223]), (64, 192, 2, 1, [176]),
                                               (128, 128, 2, 2, [175]), (128, 16, 2, 1, [5, 1, 650]), (64, 16, 130, 1, [165, 170, 400])])
def test_long_requests_in_chunks(dim, vdim, H, G, lens, channel):
    from litellmengine_amd.csrc.ops import HipOps

    o = HipOps()
    N, S, rand = sum(lens), len(lens), torch.Generator().manual_seed(dim + vdim)
    f = lambda *shape: torch.randn(shape, generator=rand).cuda()
    unit = lambda t: torch.nn.functional.normalize(t.view(N, G, dim), dim=-1).reshape(N, G * dim).contiguous()
    q, k, v, ba = unit(f(N, G * dim)), unit(f(N, G * dim)), f(N, H * vdim), f(N, 2 * H)
    k[N // 2] = k[N // 2 - 1]  # a key written twice
    a_log, dt_bias = (None, None) if channel else (f(H), f(H))
    decay = torch.sigmoid(3.0 * f(N, H * dim)) if channel else None
    if channel:
        decay[:, ::7], decay[:, 1::7] = 1.0, 0.0  # some channels never forget, some at once
        decay[::5] = 1.0
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    cu, slots = ints([sum(lens[:i]) for i in range(S + 1)]), ints(list(range(S, 0, -1)))
    start = 0.3 * f(S + 2, H * vdim * dim + 5)
    a, b = start.clone(), start.clone()
    want = REF.delta_scan(q, k, v, ba, a_log, dt_bias, a, H, G, dim, vdim, slots, cu, decay=decay)
    got = o.delta_scan(q, k, v, ba, a_log, dt_bias, b, H, G, dim, vdim, slots, cu, decay=decay)
    # values stay of the order of |v| + |S_0|, up to about 5 (unit keys, decays and betas up to one).  Where channels never forget an error
    # of a token stays, too: 700 tokens, each with sums of up to 144 products in 32 bits, sqrt(700 x 144) x 2^-24 x 5 = 1e-4, and twice that for
    # the largest of 10^5 elements
    assert (got.double() - want.double()).abs().max() < 2e-4
    assert (a.double() - b.double()).abs().max() < 2e-4
    assert torch.equal(b[:, H * vdim * dim:], start[:, H * vdim * dim:]) and torch.equal(b[0], start[0]) and torch.equal(b[S + 1], start[S + 1])
    if S == 1:  # walked one by one, the same recurrence in another order
        o.DELTA_WALK, c = N, start.clone()
        walked = o.delta_scan(q, k, v, ba, a_log, dt_bias, c, H, G, dim, vdim, slots, cu, decay=decay)
        assert (got - walked).abs().max() < 2e-4 and not torch.equal(got, walked)


@pytest.mark.parametrize("H,vdim,lens,chunks", [(130, 16, [350, 350, 1, 1, 1], False), (130, 16, [1] * 5 + [700], True), (2, 64, [1] * 70 + [700], True),
                                                (32, 64, [250] * 2 + [1] * 66 + [250], False), (32, 64, [250] + [1] * 66 + [450], True)])
def test_which_requests_go_in_chunks_is_seen_on_the_device(H, vdim, lens, chunks, monkeypatch):
    """The host launches both; the requests go in chunks where the long ones are few enough, wherever among over 64 requests they are, else they are
    walked, and never both."""
    from litellmengine_amd.csrc.ops import HipOps

    o, dim, N, S, rand = HipOps(), 64, sum(lens), len(lens), torch.Generator().manual_seed(H)
    f = lambda *shape: torch.randn(shape, generator=rand).cuda()
    unit = lambda t: torch.nn.functional.normalize(t, dim=-1)
    q, k, v, ba, a_log, dt_bias = unit(f(N, dim)), unit(f(N, dim)), f(N, H * vdim), f(N, 2 * H), f(H), f(H)
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    cu, slots = ints([sum(lens[:i]) for i in range(S + 1)]), ints(list(range(S)))
    start, names, run = 0.3 * f(S, H * vdim * dim), [], o._run
    monkeypatch.setattr(o, "_run", lambda lib, name, *a: (names.append(name), run(lib, name, *a))[1])
    a, b, c = start.clone(), start.clone(), start.clone()
    want = REF.delta_scan(q, k, v, ba, a_log, dt_bias, a, H, 1, dim, vdim, slots, cu)
    got = o.delta_scan(q, k, v, ba, a_log, dt_bias, b, H, 1, dim, vdim, slots, cu)
    assert names == ["lle_delta_chunks", "lle_delta_scan"]
    assert (got - want).abs().max() < 2e-4 and (a - b).abs().max() < 2e-4  # (as above)
    o.DELTA_WALK = N
    walked = o.delta_scan(q, k, v, ba, a_log, dt_bias, c, H, 1, dim, vdim, slots, cu)
    assert torch.equal(got, walked) != chunks and torch.equal(b, c) != chunks


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "decay", "state"])
@pytest.mark.parametrize("value", [math.inf, math.nan])
def test_what_is_not_finite_stays_behind_its_token(what, value, dim):
    """Token 24, inside a chunk, brings something that is not finite: rows before it are what they were, and in all others and in the states
    nothing else is finite or not than where the tokens are walked."""
    from litellmengine_amd.csrc.ops import HipOps

    o, H, vdim, N, token = HipOps(), 2, 64, 200, 24
    rand = torch.Generator().manual_seed(1)
    f = lambda *shape: torch.randn(shape, generator=rand).cuda()
    unit = lambda t: torch.nn.functional.normalize(t, dim=-1)
    q, k, v, beta, decay, state = unit(f(N, dim)), unit(f(N, dim)), f(N, H * vdim), f(N, H), torch.sigmoid(3.0 * f(N, H * dim)), 0.3 * f(1, H * vdim * dim)
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()

    def run(own):
        return o.delta_scan(q, k, v, beta, None, None, own, H, 1, dim, vdim, ints([0]), ints([0, N]), decay=decay)

    clean = run(state.clone())
    operand = {"q": q, "k": k, "v": v, "beta": beta, "decay": decay}.get(what, state)
    operand[0 if what == "state" else token, 1] = value
    chunks, walked = state.clone(), state.clone()
    got = run(chunks)
    o.DELTA_WALK = N
    want = run(walked)
    assert torch.equal(got.isfinite(), want.isfinite()) and torch.equal(chunks.isfinite(), walked.isfinite())
    fine = want.isfinite()
    assert (got - want)[fine].abs().max() < 2e-4 if fine.any() else what == "state"  # (as above)
    if what != "state":
        assert torch.equal(got[:token], clean[:token])


@pytest.mark.parametrize("tokens", [0, 3, 150, 161])
def test_a_single_request_of_fewer_tokens_than_rows(tokens):
    """Rows behind the request's last token belong to nobody; whether it is long is seen on the device, not by the rows."""
    from litellmengine_amd.csrc.ops import HipOps

    o, H, dim, N = HipOps(), 2, 64, 200
    rand = torch.Generator().manual_seed(1)
    f = lambda *shape: torch.randn(shape, generator=rand).cuda()
    unit = lambda t: torch.nn.functional.normalize(t, dim=-1)
    q, k, v, ba, a_log, dt_bias, state = unit(f(N, dim)), unit(f(N, dim)), f(N, H * dim), f(N, 2 * H), f(H), f(H), 0.3 * f(1, H * dim * dim)
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    a, b = state.clone(), state.clone()
    head = [t[:tokens] for t in (q, k, v, ba)]
    want = REF.delta_scan(*head, a_log, dt_bias, a, H, 1, dim, dim, ints([0]), ints([0, tokens])) if tokens else v[:0]
    got = o.delta_scan(q, k, v, ba, a_log, dt_bias, b, H, 1, dim, dim, ints([0]), ints([0, tokens]))
    assert torch.equal(got[:0], want) if tokens == 0 else (got[:tokens] - want).abs().max() < 2e-4  # (as above)
    assert (a - b).abs().max() < 2e-4


def test_more_requests_than_a_grid_holds():
    """65600 requests of one token: the ones at the edges of the launches that they are cut into."""
    from litellmengine_amd.csrc.ops import HipOps

    S, dim = 65600, 16
    gen = torch.Generator(device="cuda").manual_seed(1)
    f = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    q, k, v, ba, a_log, dt_bias, state = f(S, dim), f(S, dim), f(S, dim), f(S, 2), f(1), f(1), f(S, dim * dim)
    slots, cu = torch.arange(S, dtype=torch.int32, device="cuda"), torch.arange(S + 1, dtype=torch.int32, device="cuda")
    at = torch.tensor([0, 1, 65534, 65535, 65536, S - 1], device="cuda")
    want_state = state[at].clone()
    want = REF.delta_scan(q[at], k[at], v[at], ba[at], a_log, dt_bias, want_state, 1, 1, dim, dim, slots[:6], cu[:7])
    got = HipOps().delta_scan(q, k, v, ba, a_log, dt_bias, state, 1, 1, dim, dim, slots, cu)
    # (keys that are no unit vectors: values of |k| |q| |S|, some hundreds, with sums of 16 products in 32 bits)
    scale = float(want.abs().max())
    assert (got[at] - want).abs().max() < 32 * 2**-24 * max(1.0, scale) and (state[at] - want_state).abs().max() < 32 * 2**-24 * max(1.0, scale)
