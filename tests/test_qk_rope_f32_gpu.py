"""Norm, rotation and cache write of float32 heads of 128 for many tokens: the same bits as for few, which a wavefront a head works on."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nq,nkv,page,first", [(94, 16, 8, 16, 0), (273, 5, 3, 24, 5), (1001, 1, 1, 8, 3), (300, 32, 8, 16, 16), (303, 6, 2, 256, 250)])
@pytest.mark.parametrize("weights", [None, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("write", [True, False])
def test_many_tokens_like_few(N, nq, nkv, page, first, weights, write):
    """A last group of heads that is not whole, tokens that fill no group of sixteen, runs of slots that start inside a page, go on in another
    one, and have gaps."""
    from litellmengine_amd.csrc.ops import default_ops

    o, d = default_ops(), 128
    g = torch.Generator(device="cuda").manual_seed(N + page)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    qkv, angle = rand(N, (nq + 2 * nkv) * d), rand(N, d // 2)
    cos_sin = torch.stack([angle.cos(), angle.sin()], dim=-1).contiguous()
    qw, kw = (None, None) if weights is None else (rand(d).to(weights), rand(d).to(weights))
    slots = torch.arange(first, first + N, dtype=torch.int32, device="cuda")
    slots[N // 2:] += 2 * page
    slots[7], slots[N - 3] = -1, -1
    pages = (first + N) // page + 4
    whole, parts = (torch.full((pages, 2, nkv, page, d), 7.0, device="cuda") for _ in range(2))
    call = lambda a, b, kv: o.qk_norm_rope_write(qkv[a:b].contiguous(), slots[a:b].contiguous(), qw, kw, cos_sin[a:b].contiguous(), d, 1e-6, kv, nq, nkv, d,
                                                 write_kv=write)
    q = call(0, N, whole)
    few = torch.cat([call(a, min(N, a + 40), parts) for a in range(0, N, 40)])
    assert torch.equal(q, few) and torch.equal(whole, parts)
    assert write != bool((whole == 7.0).all())
