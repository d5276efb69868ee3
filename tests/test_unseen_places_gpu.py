"""Attention over pages that hold anything where no request's key is: pages are handed on as they are, so a request that ended
with infinities must not be found in the next one's results."""
import pytest
import torch

from tests.test_kernels_gpu import attention_case, ops, rnd

pytestmark = pytest.mark.gpu
NAN = float("nan")


def spoil(args, P, window, requests, fresh=False, keep_first=0):
    """The pool with NaN in every place whose key no row sees (and, `fresh`, where a new token's will be)."""
    _, kv, table, slots = args[:4]
    seen = torch.zeros((kv.shape[0], P), dtype=torch.bool)
    for s, (past, n) in enumerate(requests):
        first = max(0, past - window + 1) if window else 0
        for j in [*range(min(keep_first, past + n)), *range(first, past + n - (n if fresh else 0))]:
            seen[int(table[int(slots[s]), j // P]), j % P] = True
    out, nobodys = kv.clone(), (~seen).to(kv.device)
    out[:, 0].masked_fill_(nobodys[:, None, :, None], NAN)
    shape = out[:, 1].shape  # values lie transposed
    values = out[:, 1].reshape(shape[0], shape[1], shape[3], P).masked_fill(nobodys[:, None, None, :], NAN)
    out[:, 1] = values.view(shape)
    assert out.isnan().any()
    return out


def case(dtype, nq, nkv, d, P, window, requests):
    need = [-(-(p + n) // P) for p, n in requests]
    return attention_case(dtype, nq, nkv, d, P, window, requests, pages=sum(need) + 3, max_pages=max(need) + 1)


REQUESTS = [[(0, 9), (17, 1), (30, 2), (5, 11)], [(1999, 1), (640, 1), (31, 1), (0, 1)], [(0, 150), (100, 70)], [(1500, 40), (1900, 1), (3, 30)]]


# one tile of rows and many, one row tile a wavefront and two, key splits; windows, kept first keys, capped scores
@pytest.mark.parametrize("requests", REQUESTS)
@pytest.mark.parametrize("nq,nkv,d,P,window,extra", [(8, 2, 128, 16, None, {}), (32, 8, 128, 16, 700, {}), (16, 2, 64, 32, 40, {}),
                                                     (3, 1, 160, 48, None, {}), (4, 2, 32, 16, 17, {}), (8, 2, 64, 16, 50, {"keep_first": 9}),
                                                     (8, 2, 128, 32, None, {"softcap": 20.0})])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_places_that_no_row_sees(dtype, nq, nkv, d, P, window, extra, requests):
    args, mq, mk = case(dtype, nq, nkv, d, P, window, requests)
    bad = [*args]
    bad[1] = spoil(args, P, window, requests, keep_first=extra.get("keep_first", 0))
    o = ops()
    for form in (1, 2, 3) if dtype == torch.bfloat16 else (0,):
        o.force_prefill_form = form
        try:
            want, got = (o.paged_attention(*a, *mq, mk, **extra) for a in (args, bad))
        finally:
            o.force_prefill_form = 0
        assert want.isfinite().all() and torch.equal(got, want), form


# the decode launches that write the new token themselves: short (one token a request) and general (token_seq given, more keys)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("write", [True, False])
@pytest.mark.parametrize("lens", [[1, 2, 15, 16, 17], [31, 32, 33, 64, 97], [176, 177, 255, 256], [257, 2000]])
@pytest.mark.parametrize("nq,nkv,d,P,window", [(16, 8, 128, 16, None), (8, 8, 64, 48, 20), (10, 1, 128, 32, 200)])
def test_the_new_tokens_place_and_those_behind_it(nq, nkv, d, P, window, lens, write, dtype):
    requests = [(n - 1, 1) for n in lens]
    args, _, mk = case(dtype, nq, nkv, d, P, window, requests)
    _, kv, table, seq_slots, cu, kv_lens, token_seq, _, scale = args
    S, o = len(lens), ops()
    qkv = rnd((S, (nq + 2 * nkv) * d), dtype, 70, 1.5)
    slots = torch.tensor([int(table[int(seq_slots[s]), (n - 1) // P]) * P + (n - 1) % P for s, n in enumerate(lens)], dtype=torch.int32).cuda()
    cs = o.rope_table((kv_lens - 1).int(), (1e6 ** (-(2.0 * torch.arange(d // 2, dtype=torch.float64)) / d)).float().cuda())
    qw, kw = (1 + 0.2 * rnd((d,), torch.float32, seed) for seed in (71, 72))
    bad = spoil(args, P, window, requests, fresh=write)
    short = mk <= 256
    seqs = [None] * short + [token_seq] * (dtype == torch.bfloat16)
    for seq in seqs:
        want, got = (o.qk_norm_rope_attention(qkv, slots, qw, kw, cs, 1e-5, pool.clone(), nq, nkv, d, write, table, seq_slots, cu, kv_lens,
                                              seq, window, scale, mk) for pool in (kv, bad))
        assert want.isfinite().all() and torch.equal(got, want)
    if dtype == torch.bfloat16 and short:
        pool, spoilt = kv.clone(), bad.clone()
        want, got = (o.pair_rope_attention(qkv, slots, cs, p, nq, nkv, d, write, table, seq_slots, cu, kv_lens, window, scale, mk, 30.0)
                     for p in (pool, spoilt))
        assert want.isfinite().all() and torch.equal(got, want)


@pytest.mark.parametrize("P,rank,rot,H,lens,pasts,window", [(16, 96, 8, 5, [7, 1, 1], [0, 40, 300], None), (32, 512, 64, 16, [40, 1, 1], [100, 1900, 333], None),
                                                            (16, 64, 32, 8, [1, 1, 1, 1], [0, 31, 32, 700], 50), (16, 128, 32, 4, [90, 1], [0, 70], 33)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_latents_that_no_row_sees(dtype, P, rank, rot, H, lens, pasts, window):
    from tests.test_birelix_kernels_gpu import latent_case

    c = latent_case(dtype, P, rank, rot, H, lens, pasts, 21, pages_total=160)
    q_lat, q_rot = rnd((H, c["N"], rank), dtype, 24, 0.3).transpose(0, 1), rnd((c["N"], H, rot), torch.float32, 23)
    pages = c["pages"].shape[0]
    seen = torch.zeros((pages, P), dtype=torch.bool)
    for s, (past, n) in enumerate(zip(pasts, lens)):
        for j in range(max(0, past - window + 1) if window else 0, past + n):
            seen[int(c["table"][int(c["seq_slots"][s]), j // P]), j % P] = True
    bad, nobodys = c["pages"].clone().view(pages, -1), (~seen).cuda()  # a page: latents by key, latents by element, rotated keys
    for part, by_key, width in ((0, True, rank), (P * rank, False, rank), (2 * P * rank, True, rot)):
        view = bad[:, part : part + P * width].view(pages, P, width) if by_key else bad[:, part : part + P * width].view(pages, width, P).transpose(1, 2)
        view.masked_fill_(nobodys[:, :, None], NAN)
    assert bad.isnan().any()
    run = lambda p: ops().latent_attention(q_lat, q_rot, p.view(c["pages"].shape), P, rank, rot, c["table"], c["seq_slots"], c["cu"], c["kv_lens"],
                                           c["token_seq"], None, window, 0.11, max(lens), max(c["kv_lens"].tolist()), dtype)
    want = run(c["pages"])
    assert want.isfinite().all() and torch.equal(run(bad), want)


@pytest.mark.parametrize("H,G,D,P", [(8, 4, 64, 16), (6, 2, 32, 16), (16, 2, 128, 16), (20, 5, 64, 48), (32, 8, 128, 16), (5, 1, 48, 8)])
@pytest.mark.parametrize("chunk", [None, 24, 100])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_places_that_no_row_sees_with_heads_mixed(dtype, H, G, D, P, chunk):
    from tests.test_telulorn_kernels_gpu import talking_case

    for lens, pasts in (([1, 37, 2, 1, 61, 1], [100, 0, 47, 99, 130, 0]), ([1, 1, 1, 1], [190, 23, 24, 1500])):
        args, most, slopes, talk = talking_case(dtype, lens, pasts, H, G, D, P)
        _, kv, table, slots = args[:4]
        seen = torch.zeros((kv.shape[0], P), dtype=torch.bool)
        for s, (past, n) in enumerate(zip(pasts, lens)):
            for j in range(past // chunk * chunk if chunk else 0, past + n):
                seen[int(table[int(slots[s]), j // P]), j % P] = True
        bad, nobodys = kv.clone(), (~seen).to(kv.device)
        bad[:, 0].masked_fill_(nobodys[:, None, :, None], NAN)
        bad[:, 1].view(kv.shape[0], G, D, P).masked_fill_(nobodys[:, None, None, :], NAN)
        assert bad.isnan().any()
        want, got = (ops().talking_attention(args[0], p, *args[2:], chunk, 0.2, slopes, talk, min(lens), max(lens), most) for p in (kv, bad))
        assert want.isfinite().all() and torch.equal(got, want)
