"""The state-space recurrence's chunks, whose workgroups take several heads of a group one after the
other: every number of value tiles (odd ones hand the next head's entry rows over), widths of LDS rows,
states of one and of two register sets, sizes that 16-byte loads do not fit, and more heads a group than
a workgroup holds step sizes of."""

import pytest
import torch

from tests.test_kezasun_kernels_gpu import ops
from tests.test_rorevik_kernels_gpu import REF, close, ssd_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("together,H,G,vdim,n", [
    (3, 6, 2, 48, 132), (4, 4, 1, 80, 128), (2, 4, 2, 16, 20), (5, 5, 1, 20, 6), (4, 4, 1, 6, 33), (2, 2, 1, 144, 64), (2, 2, 1, 208, 100),
    (40, 40, 1, 16, 16), (34, 68, 2, 32, 24), (37, 37, 1, 12, 8)])
def test_heads_of_a_workgroup(together, H, G, vdim, n, monkeypatch):
    """The rows and states are those of a workgroup a head to the last bit, and the oracle's."""
    o = ops()
    q_lens = [130, 33, 1, 64]
    c, dt_in, dt_bias, a_log, D, wide, seq_slots, cu = ssd_case(H, G, vdim, n, q_lens)
    args = (c, dt_in, dt_bias, a_log, D)
    got = {}
    for k in (1, together):
        monkeypatch.setattr(o, "ssd_heads_a_group", lambda *a, k=k: k)
        state = wide.clone()
        got[k] = o.ssd_scan(*args, state, H, G, vdim, n, seq_slots, cu, 1, 130), state
    assert torch.equal(got[1][0], got[together][0]) and torch.equal(got[1][1], got[together][1])
    state = wide.clone()
    want = REF.ssd_scan(*args, state, H, G, vdim, n, seq_slots, cu)
    # sums of at most 64 tokens and n <= 132 channels, in 32 bits: under 64 roundings of the largest result
    close(got[together][0], want, 64 * 2**-24 * max(1.0, float(want.abs().max())))
    close(got[together][1], state, 64 * 2**-24 * max(1.0, float(state.abs().max())))


@pytest.mark.parametrize("H,G,vdim,q_lens", [(2, 1, 16, [33]), (3, 3, 48, [64]), (4, 2, 64, [65, 1, 127]), (4, 1, 80, [128, 32, 129, 7]), (6, 2, 32, [400]),
                                             (64, 2, 64, [1, 193])])
def test_chunks_one_after_the_other(H, G, vdim, q_lens, monkeypatch):
    """States of 128 channels kept in registers: the shortest request of one chunk, whole last chunks and ones of one token, beside
    requests that are walked; the oracle's rows and states, and those of the chunks side by side."""
    o = ops()
    c, dt_in, dt_bias, a_log, D, wide, seq_slots, cu = ssd_case(H, G, vdim, 128, q_lens)
    args, got = (c, dt_in, dt_bias, a_log, D), {}
    for streams in (True, False):
        monkeypatch.setattr(o, "ssd_streams", lambda *a, s=streams: s)
        state = wide.clone()
        got[streams] = o.ssd_scan(*args, state, H, G, vdim, 128, seq_slots, cu, min(q_lens), max(q_lens)), state
    state = wide.clone()
    want = REF.ssd_scan(*args, state, H, G, vdim, 128, seq_slots, cu)
    # sums of at most 64 tokens and 128 channels, in 32 bits: under 64 roundings of the largest result
    for rows, states in got.values():
        close(rows, want, 64 * 2**-24 * max(1.0, float(want.abs().max())))
        close(states, state, 64 * 2**-24 * max(1.0, float(state.abs().max())))
    behind = H * vdim * 128
    assert torch.equal(got[True][1][:, behind:], wide[:, behind:])  # what lies behind the matrices stays
    untouched = [i for i in range(wide.shape[0]) if i not in seq_slots.tolist()]
    assert torch.equal(got[True][1][untouched], wide[untouched])


def test_a_steep_drop_inside_a_chunk():
    """Decays that end a state at once, and none at all: later tokens' exponents never rise above zero, what is forgotten is gone."""
    o = ops()
    H, G, vdim, N = 2, 1, 16, 150
    c = torch.randn((N, H * vdim + 2 * 128), generator=torch.Generator().manual_seed(2)).cuda()
    dt_in = torch.zeros((N, H)).cuda()
    dt_in[70, 0] = 2000.0  # head 0: the decay of token 70 is exp(-2000)
    dt_in[:, 1] = -60.0  # head 1: no step at all
    zeros, D = torch.zeros(H).cuda(), torch.zeros(H).cuda()
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    state = torch.ones((2, H * vdim * 128)).cuda()
    got = o.ssd_scan(c, dt_in, zeros, zeros, D, state, H, G, vdim, 128, ints([1]), ints([0, N]), N, N)
    want_state = torch.ones((2, H * vdim * 128)).cuda()
    want = REF.ssd_scan(c, dt_in, zeros, zeros, D, want_state, H, G, vdim, 128, ints([1]), ints([0, N]))
    scale = float(want.abs().max())
    assert torch.isfinite(got).all() and (got - want).abs().max() < 128 * 2**-24 * scale
    assert (state - want_state).abs().max() < 64 * 2**-24 * float(want_state.abs().max())


def test_a_drop_further_than_its_exponent():
    """A decay of exp(-3e38), finite as it is: what was before is gone, what comes after is not touched."""
    o = ops()
    H, G, vdim, N = 2, 1, 16, 150
    c = torch.randn((N, H * vdim + 2 * 128), generator=torch.Generator().manual_seed(2)).cuda()
    dt_in = torch.full((N, H), -200.0).cuda()  # (exp(69) would end the state with any other step of head 0)
    dt_in[70, 0] = 3.0e8
    a_log = torch.tensor([69.0, 0.0]).cuda()  # exp(69) 3e8 = 2.8e38
    zeros, D = torch.zeros(H).cuda(), torch.zeros(H).cuda()
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    state, want_state = torch.ones((2, H * vdim * 128)).cuda(), torch.ones((2, H * vdim * 128)).cuda()
    got = o.ssd_scan(c, dt_in, zeros, a_log, D, state, H, G, vdim, 128, ints([1]), ints([0, N]), N, N)
    want = REF.ssd_scan(c, dt_in, zeros, a_log, D, want_state, H, G, vdim, 128, ints([1]), ints([0, N]))
    assert torch.isfinite(got).all()
    for part in (slice(0, 70), slice(70, N)):  # (from token 70 on rows of head 0 are of the order of 3e8)
        assert (got[part] - want[part]).abs().max() < 128 * 2**-24 * float(want[part].abs().max())
    assert (state - want_state).abs().max() < 64 * 2**-24 * float(want_state.abs().max())


@pytest.mark.parametrize("a_log", [-8.0, -4.0, -2.0, 0.0])
def test_decays_inside_a_chunk_to_two_ulps(a_log):
    """y of the token behind x = 1 is 32 exp(-exp(a_log) dt), dt from 32 to 95 and exact in 32 bits; arguments from -0.01 to -95."""
    o = ops()
    H, vdim, N = 64, 16, 40
    c = torch.zeros((N, H * vdim + 2 * 128))
    c[0, : H * vdim] = 1.0  # x of token 0 alone
    c[:, H * vdim], c[:, H * vdim + 128] = 1.0, 1.0  # B and C of channel 0
    dt_in = torch.full((N, H), -200.0)  # (steps of 1e-87: none)
    dt_in[0] = 32.0
    dt_in[1] = 32.0 + torch.arange(H)
    zeros, state = torch.zeros(H).cuda(), torch.zeros((1, H * vdim * 128)).cuda()
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    y = o.ssd_scan(c.cuda(), dt_in.cuda(), zeros, zeros + a_log, zeros, state, H, 1, vdim, 128, ints([0]), ints([0, N]), N, N)
    arg = -torch.exp(torch.tensor(a_log, dtype=torch.float64)) * dt_in[1].double()
    want = 32.0 * torch.exp(arg)
    got = y[1].view(H, vdim)[:, 0].cpu().double()
    # the argument is off by an ulp of exp(a_log) and half a one of its product: |arg| 1.5 ulps; the exponential and two products: four; results below
    # 2^-126 are gone
    assert ((got - want).abs() < (1.5 * arg.abs() + 4) * 2**-23 * want + 32 * 2**-126).all()
    assert torch.equal(y[2:].view(-1, H, vdim)[:, :, 0].cpu().double(), got.expand(N - 2, H))  # (nothing happens any more)


@pytest.mark.parametrize("what", ["x", "B", "C", "dt", "state"])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_what_is_not_finite(what, value, monkeypatch):
    """In the chunks one after the other nothing is lost that the chunks side by side keep: no row before the token's tile of sixteen, no other state (and
    no row before the token where its step size is what is not finite, which there is a factor of what an earlier row takes 0 times)."""
    o = ops()
    H, G, vdim, N, token = 4, 2, 32, 150, 88
    c, dt_in, dt_bias, a_log, D, wide, seq_slots, cu = ssd_case(H, G, vdim, 128, [N])
    inner, slot = H * vdim, int(seq_slots[0])
    if what == "state":
        wide[slot, 3 * vdim * 128 + 7] = value
    elif what == "dt":
        dt_in[token, 1] = value
    else:
        c[token, {"x": vdim + 3, "B": inner + 5, "C": inner + G * 128 + 5}[what]] = value
    got = {}
    for streams in (True, False):
        monkeypatch.setattr(o, "ssd_streams", lambda *a, s=streams: s)
        state = wide.clone()
        got[streams] = o.ssd_scan(c, dt_in, dt_bias, a_log, D, state, H, G, vdim, 128, seq_slots, cu, N, N), state
    assert torch.equal(got[True][1].isfinite(), got[False][1].isfinite())
    for a, b in zip(got[True], got[False]):
        fine = b.isfinite()  # (tolerance as above)
        assert a[fine].isfinite().all()
        assert (a - b)[fine].abs().max() < 2 * 64 * 2**-24 * max(1.0, float(b[fine].abs().max()))
    if what != "state":
        assert got[True][0][: token if what == "dt" else token // 16 * 16].isfinite().all() and not got[True][0][token].isfinite().all()


def test_a_long_request_of_wide_rows(monkeypatch):
    """32767 tokens of 512 heads: the rest of the request behind a chunk is over 4 GiB, so that a count of its bytes in 32 bits is too small for the first
    chunks.  Rows and states are those of the chunks side by side."""
    o = ops()
    H, G, vdim, n, N = 512, 1, 64, 128, 32767
    assert o.ssd_streams(N, H, vdim, n, N) and 4 * N * (H * vdim + 2 * G * n) > 1 << 32
    gen = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda")
    c = torch.zeros((N, H * vdim + 2 * G * n), device="cuda")
    c[:512], c[-100:] = rand(512, c.shape[1]), rand(100, c.shape[1])
    dt_in, dt_bias, a_log, D = rand(N, H), rand(H), rand(H) - 8.0, rand(H)  # (decays of a thousandth a token: the first chunks are still seen)
    ints = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    got = {}
    for streams in (True, False):
        monkeypatch.setattr(o, "ssd_streams", lambda *a, s=streams: s)
        state = torch.zeros((1, H * vdim * n), device="cuda")
        y = o.ssd_scan(c, dt_in, dt_bias, a_log, D, state, H, G, vdim, n, ints([0]), ints([0, N]), N, N)
        got[streams] = y[:1024].clone(), y[-200:].clone(), state
        del y
    for a, b in zip(got[True], got[False]):  # sums of at most 64 tokens and 128 channels, in 32 bits: under 64 roundings of the largest result
        close(a, b, 64 * 2**-24 * max(1.0, float(b.abs().max())))
