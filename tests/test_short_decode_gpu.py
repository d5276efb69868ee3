"""Decode steps of up to 256 keys a request: the launch with a wavefront for every 32 keys and one for the new token."""
import pytest
import torch

from tests.test_kernels_gpu import attention_case, ops, rnd

pytestmark = pytest.mark.gpu


# a request's first token, the edges of halves, steps and pages, the most keys that the launch takes; beyond them the general
# one.  In each list one token's place is not written (slot -1): it attends to what the page holds.
@pytest.mark.parametrize("lens", [[1, 2, 15, 16, 17], [31, 32, 33, 64, 97], [255, 256, 160, 1], [257, 40]])
@pytest.mark.parametrize("nq,nkv,d,P,window", [(16, 8, 128, 16, None), (8, 8, 64, 48, None), (13, 1, 128, 32, 40), (14, 1, 128, 16, None),
                                               (32, 2, 64, 16, 17), (4, 4, 128, 64, 1)])
@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32, None])
def test_short_decode_equals_its_two_halves(wdtype, nq, nkv, d, P, window, lens):
    requests = [(n - 1, 1) for n in lens]
    args, mq, mk = attention_case(torch.bfloat16, nq, nkv, d, P, window, requests,
                                  pages=sum(-(-n // P) for n in lens) + 3, max_pages=-(-max(lens) // P) + 1)
    _, kv, table, seq_slots, cu, kv_lens, token_seq, _, scale = args
    S = len(lens)
    qkv = rnd((S, (nq + 2 * nkv) * d), torch.bfloat16, 70, 1.5)
    slots = torch.tensor([int(table[int(seq_slots[s]), (n - 1) // P]) * P + (n - 1) % P for s, n in enumerate(lens)], dtype=torch.int32)
    slots[1] = -1
    slots = slots.cuda()
    inv = (1e6 ** (-(2.0 * torch.arange(d // 2, dtype=torch.float64)) / d)).float().cuda()
    o = ops()
    cs = o.rope_table((kv_lens - 1).int(), inv)
    qw = kw = None
    if wdtype is not None:
        qw, kw = ((1 + 0.2 * rnd((d,), torch.float32, seed)).to(wdtype) for seed in (71, 72))
    a, b = kv.clone(), kv.clone()
    q = o.qk_norm_rope_write(qkv, slots, qw, kw, cs, d, 1e-5, a, nq, nkv, d, True)
    want = o.paged_attention(q, a, table, seq_slots, cu, kv_lens, token_seq, window, scale, *mq, mk).double()
    run = lambda pool, write: o.qk_norm_rope_attention(qkv, slots, qw, kw, cs, 1e-5, pool, nq, nkv, d, write, table, seq_slots, cu, kv_lens,
                                                       None, window, scale, mk).double()
    got = run(b, True)
    # both round the same 32-bit results to bfloat16: a key may be one unit in the last place off where a product was fused differently
    assert not torch.equal(b, kv) and (a.float() - b.float()).abs().max() <= 2.0 ** -7 * a.float().abs().max()
    # weights in bfloat16 (2^-9 relative each) on values of size 4 at most, rounded once more
    assert (got - want).abs().max() < 2e-2
    c = a.clone()
    assert (run(c, False) - want).abs().max() < 2e-2 and torch.equal(c, a)


def test_a_request_without_a_token_is_left_alone():
    """Three requests, the second with no token in this step: the others' rows are theirs."""
    args, mq, mk = attention_case(torch.bfloat16, 4, 2, 64, 16, None, [(20, 1), (40, 1)])
    _, kv, table, seq_slots, _, kv_lens, _, _, scale = args
    o = ops()
    qkv = rnd((2, 8 * 64), torch.bfloat16, 5)
    cs = o.rope_table((kv_lens - 1).int(), torch.ones(32, device="cuda"))
    slots = torch.full((2,), -1, dtype=torch.int32, device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    run = lambda s, cu, lens, seq: o.qk_norm_rope_attention(qkv, slots, None, None, cs, 1e-5, kv, 4, 2, 64, True, table, s, cu, lens, seq, None, scale, mk)
    want = run(seq_slots, i32([0, 1, 2]), kv_lens, None)
    three = lambda x: torch.stack([x[0], x[0], x[1]])
    got = run(three(seq_slots), i32([0, 1, 1, 2]), three(kv_lens), i32([0, 2]))
    assert (got.double() - want.double()).abs().max() < 2e-2
    with pytest.raises(Exception, match="one token"):
        run(three(seq_slots), i32([0, 1, 1, 2]), three(kv_lens), None)


@pytest.mark.parametrize("lens", [[1, 2, 15, 16, 17], [31, 32, 33, 64, 97], [255, 256, 160, 1]])
@pytest.mark.parametrize("nq,nkv,d,P,window,rot,cap", [(16, 4, 128, 16, None, 64, 30.0), (8, 8, 64, 48, None, 64, None), (13, 1, 128, 32, 40, 8, None),
                                                       (4, 2, 64, 16, 17, 0, 5.0), (4, 4, 128, 64, 1, 128, None)])
def test_short_decode_with_pairs_equals_its_two_halves(lens, nq, nkv, d, P, window, rot, cap):
    """The rotation of neighbouring pairs, capped scores, columns beside q, k and v."""
    requests = [(n - 1, 1) for n in lens]
    args, mq, mk = attention_case(torch.bfloat16, nq, nkv, d, P, window, requests,
                                  pages=sum(-(-n // P) for n in lens) + 3, max_pages=-(-max(lens) // P) + 1)
    _, kv, table, seq_slots, cu, kv_lens, token_seq, _, scale = args
    S = len(lens)
    u = rnd((S, (nq + 2 * nkv) * d + 24), torch.bfloat16, 70, 1.5)
    slots = torch.tensor([int(table[int(seq_slots[s]), (n - 1) // P]) * P + (n - 1) % P for s, n in enumerate(lens)], dtype=torch.int32)
    slots[1] = -1
    slots = slots.cuda()
    o = ops()
    cs = o.rope_table((kv_lens - 1).int(), (1e4 ** (-torch.arange(rot // 2, dtype=torch.float64) / 32)).float().cuda()) if rot else None
    a, b = kv.clone(), kv.clone()
    q = o.pair_rope_write(u, None, slots, cs, None, a, nq, nkv, d, d, True)
    want = o.paged_attention(q, a, table, seq_slots, cu, kv_lens, token_seq, window, scale, *mq, mk, softcap=cap).double()
    assert o.can_fuse_pair_rope_attention(u, d, d, rot, kv, nq, 1, mk, S) and not o.can_fuse_pair_rope_attention(u, d, d, rot, kv, nq, 1, 257, S)
    run = lambda pool, write: o.pair_rope_attention(u, slots, cs, pool, nq, nkv, d, write, table, seq_slots, cu, kv_lens, window, scale, mk, cap).double()
    got = run(b, True)
    # the same 32-bit rotation, rounded once: a unit in the last place where a product was fused differently
    assert not torch.equal(b, kv) and (a.float() - b.float()).abs().max() <= 2.0 ** -7 * a.float().abs().max()
    assert (got - want).abs().max() < 2e-2  # (as above)
    c = a.clone()
    assert (run(c, False) - want).abs().max() < 2e-2 and torch.equal(c, a)


# float32: the edges of its steps of 16 keys, of a wavefront's second step (176), the most keys that the launch takes
@pytest.mark.parametrize("lens", [[1, 2, 15, 16, 17], [31, 32, 33, 64, 97], [175, 176, 177, 178], [255, 256, 240, 193]])
@pytest.mark.parametrize("nq,nkv,d,P,window", [(16, 8, 128, 16, None), (8, 8, 64, 48, None), (10, 1, 128, 32, 40), (32, 2, 64, 16, 17), (4, 4, 128, 64, 1)])
@pytest.mark.parametrize("wdtype", [torch.bfloat16, torch.float32, None])
def test_short_decode_in_float32_equals_its_two_halves(wdtype, nq, nkv, d, P, window, lens):
    requests = [(n - 1, 1) for n in lens]
    args, mq, mk = attention_case(torch.float32, nq, nkv, d, P, window, requests,
                                  pages=sum(-(-n // P) for n in lens) + 3, max_pages=-(-max(lens) // P) + 1)
    _, kv, table, seq_slots, cu, kv_lens, token_seq, _, scale = args
    S = len(lens)
    o = ops()
    fits = lambda keys, group=nq // nkv, rot=d, heads=96: o.can_fuse_rope_attention(torch.float32, d, rot, P, group, 1, keys, S, heads)
    assert fits(mk) and not fits(257) and not fits(mk, 17) and not fits(mk, rot=d // 2) and fits(176, heads=1) and not fits(177, heads=1)
    qkv = rnd((S, (nq + 2 * nkv) * d), torch.float32, 70, 1.5)
    slots = torch.tensor([int(table[int(seq_slots[s]), (n - 1) // P]) * P + (n - 1) % P for s, n in enumerate(lens)], dtype=torch.int32)
    slots[1] = -1
    for s, n in enumerate(lens):  # what lies behind a request's last key in its page is nobody's
        page, off = int(table[int(seq_slots[s]), (n - 1) // P]), (n - 1) % P
        kv[page, 0, :, off + 1:] = float("nan")
        kv[page, 1].view(nkv, d, P)[:, :, off + 1:] = float("nan")
    slots = slots.cuda()
    inv = (1e6 ** (-(2.0 * torch.arange(d // 2, dtype=torch.float64)) / d)).float().cuda()
    cs = o.rope_table((kv_lens - 1).int(), inv)
    qw = kw = None
    if wdtype is not None:
        qw, kw = ((1 + 0.2 * rnd((d,), torch.float32, seed)).to(wdtype) for seed in (71, 72))
    a, b = kv.clone(), kv.clone()
    q = o.qk_norm_rope_write(qkv, slots, qw, kw, cs, d, 1e-5, a, nq, nkv, d, True)
    a.nan_to_num_(0.0)
    want = o.paged_attention(q, a, table, seq_slots, cu, kv_lens, token_seq, window, scale, *mq, mk).double()
    run = lambda pool, write: o.qk_norm_rope_attention(qkv, slots, qw, kw, cs, 1e-5, pool, nq, nkv, d, write, table, seq_slots, cu, kv_lens,
                                                       None, window, scale, mk).double()
    got = run(b, True)
    # sums of 128 products in 32 bits, in another order: 128 x 2^-24 = 8e-6 of values of size 4 and of scores of size 10
    assert (got - want).abs().max() < 1e-4
    written = b.nan_to_num(0.0)
    assert not torch.equal(written, kv.nan_to_num(0.0)) and (a - written).abs().max() < 1e-5
    c = a.clone()
    assert (run(c, False) - want).abs().max() < 1e-4 and torch.equal(c, a)


# as many workgroups as the launch takes and one request more, which the general launches take
@pytest.mark.parametrize("dtype,nq,nkv,d,S", [(torch.bfloat16, 8, 8, 64, 64), (torch.bfloat16, 32, 2, 64, 128), (torch.float32, 4, 8, 64, 64),
                                              (torch.float32, 16, 8, 64, 96)])
@pytest.mark.parametrize("more", [0, 1])
def test_many_requests(dtype, nq, nkv, d, S, more):
    nq, P, n, S = max(nq, nkv), 16, 33, S + more
    o, i32 = ops(), lambda x: torch.as_tensor(x, dtype=torch.int32).cuda()
    kv, qkv = rnd((3 * S, 2, nkv, P, d), dtype, 1), rnd((S, (nq + 2 * nkv) * d), dtype, 2, 1.5)
    table = i32(torch.randperm(3 * S, generator=torch.Generator().manual_seed(3)).view(S, 3))
    slots, seqs, cu, lens = (table[:, 2] * P).int(), i32(range(S)), i32(range(S + 1)), i32([n] * S)
    cs = o.rope_table((lens - 1).int(), torch.ones(d // 2, device="cuda"))
    a, b = kv.clone(), kv.clone()
    q = o.qk_norm_rope_write(qkv, slots, None, None, cs, d, 1e-6, a, nq, nkv, d, True)
    want = o.paged_attention(q, a, table, seqs, cu, lens, seqs, None, d ** -0.5, 1, 1, n).double()
    fits = lambda S, kv_heads: o.can_fuse_rope_attention(dtype, d, d, P, nq // nkv, 1, n, S, kv_heads)
    if dtype == torch.float32:
        if o.compute_units() == 256:
            assert [S for S in (64, 65, 87, 88, 96, 97, 256) if fits(S, 8)] == [64, 88, 96] and fits(256, 2) and not fits(257, 2)
        if not fits(S, nkv):
            return
    got = o.qk_norm_rope_attention(qkv, slots, None, None, cs, 1e-6, b, nq, nkv, d, True, table, seqs, cu, lens, None, None, d ** -0.5, n).double()
    assert (got - want).abs().max() < (2e-2 if dtype == torch.bfloat16 else 1e-4)  # (as above)
    assert (a.float() - b.float()).abs().max() <= (2.0 ** -7 * 8 if dtype == torch.bfloat16 else 1e-5)


def test_which_float32_steps_of_a_runner_take_the_short_launch(monkeypatch):
    """A decode step runs as a graph whose bound on the keys is 256 at least: with 8 kv heads the short launch is for 12 requests and
    more, whatever their length.  Steps without graphs know how few keys there are."""
    from litellmengine_amd.cache import CacheManager
    from litellmengine_amd.config import Qwen3Config
    from litellmengine_amd.engine import ModelRunner, StepEntry
    from litellmengine_amd.models.build import random_model

    config = Qwen3Config.from_dict(dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=1, hidden_size=64,
                                        num_attention_heads=8, num_key_value_heads=8, head_dim=64, intermediate_size=64, vocab_size=128,
                                        rope_theta=1e4, rms_norm_eps=1e-6, tie_word_embeddings=True))
    model = random_model(config, 3, "float32")
    o, taken = model.ctx.ops, []
    launch = o.qk_norm_rope_attention
    monkeypatch.setattr(o, "qk_norm_rope_attention", lambda qkv, *a: taken.append(qkv.shape[0]) or launch(qkv, *a))
    if o.compute_units() != 256:
        pytest.skip("the rule counts workgroups for 256 CUs")
    for graphs, want in ((True, [(1, False), (8, False), (12, True), (64, True), (100, False)]), (False, [(1, True), (8, True), (64, True), (100, False)])):
        cache = CacheManager(model, page_size=16, num_pages=200, max_requests=128, dtype=torch.float32, device=model.ctx.device)
        runner = ModelRunner(model, cache, use_graphs=graphs)
        for n, short in want:
            slots = [runner.admit() for _ in range(n)]
            runner.step([StepEntry(s, [1, 2, 3], [2]) for s in slots])
            taken.clear()
            runner.step([StepEntry(s, [4], [0]) for s in slots])
            assert bool(taken) == short, (graphs, n)
            for s in slots:
                runner.release(s)
