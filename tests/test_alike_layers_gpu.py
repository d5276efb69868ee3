"""Layers that are alike launch what the first of them launched: the same bits as layer by layer, in every form that a layer's products
and its attention take, and not where a layer differs or a caller has put something in between."""
import pytest
import torch

from litellmengine_amd.cache import CacheManager
from litellmengine_amd.config import Qwen3Config, get_architecture
from litellmengine_amd.csrc.ops import HipOps
from litellmengine_amd.engine.batch import StepEntry
from litellmengine_amd.engine.runner import ModelRunner
from litellmengine_amd.models import make_context
from litellmengine_amd.models.decoder import DecoderLM
from litellmengine_amd.parts import PagedAttention
from litellmengine_amd.parts.norm import RMSNorm

pytestmark = pytest.mark.gpu
LAYERS = 8


def made(dtype, width=1024, ff=3072, heads=16, kv_heads=8, windows=None):
    config = Qwen3Config.from_dict({
        "architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "num_hidden_layers": LAYERS, "hidden_size": width,
        "num_attention_heads": heads, "num_key_value_heads": kv_heads, "head_dim": 64, "intermediate_size": ff, "vocab_size": 500,
        "rope_theta": 1e6, "rms_norm_eps": 1e-6, "tie_word_embeddings": True})
    model = get_architecture(config.architecture).build(config)
    ctx = make_context(dtype)
    rand = torch.Generator().manual_seed(5)
    weights = {}
    for name, spec in model.tensor_specs().items():
        w = torch.randn(spec.shape, generator=rand) * (0.02 if len(spec.shape) > 1 else 0.1) + (1.0 if len(spec.shape) == 1 else 0.0)
        weights[name] = w.to(ctx.dtype).cuda()
    model.bind(weights, ctx)
    cache = CacheManager(model, page_size=16, num_pages=400, max_requests=40, max_pages_per_request=80, dtype=ctx.dtype, device=ctx.device)
    return ModelRunner(model, cache, use_graphs=False)


def steps(runner, sizes):
    """A prompt of 50 tokens, then a step of requests of these sizes behind it, beside one token of the first request."""
    rand = torch.Generator().manual_seed(3)
    ids = lambda n: torch.randint(0, 500, (n,), generator=rand).tolist()
    first = runner.admit()
    out = [runner.step([StepEntry(first, ids(50), [49])])]
    slots = [runner.admit() for _ in sizes]
    entries = [StepEntry(first, ids(1), [0])] + [StepEntry(s, ids(n), list(range(0, n, 7))) for s, n in zip(slots, sizes)]
    out.append(runner.step(entries))
    kept = [g.data.clone() for g in runner.cache.groups]
    for s in reversed([first] + slots):
        runner.release(s)
    return out + kept


@pytest.fixture
def replays(monkeypatch):
    counted, run = [], HipOps.replay
    monkeypatch.setattr(HipOps, "replay", lambda self, *a: (counted.append(1), run(self, *a))[1])
    return counted


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("sizes", [[], [1, 1, 1], [15], [20], [40, 9], [100], [150], [250], [300, 200], [900], [1, 1, 700]])
def test_the_same_bits_as_layer_by_layer(monkeypatch, replays, dtype, sizes):
    got = steps(made(dtype), sizes)
    assert len(replays) == 2 * (LAYERS - 3)  # all but the first two layers and the last one, of two steps
    monkeypatch.setattr(DecoderLM, "ALIKE_LAYERS", 10 ** 6)
    want = steps(made(dtype), sizes)
    assert len(replays) == 2 * (LAYERS - 3)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("width,ff,heads,kv_heads", [(4096, 4096, 4, 2), (2048, 6144, 8, 1), (520, 1000, 3, 3)])
def test_other_widths(monkeypatch, replays, width, ff, heads, kv_heads):
    runner = made("bfloat16", width, ff, heads, kv_heads)
    got = [steps(runner, sizes) for sizes in ([5], [130], [500])]
    assert replays
    monkeypatch.setattr(DecoderLM, "ALIKE_LAYERS", 10 ** 6)
    runner = made("bfloat16", width, ff, heads, kv_heads)
    want = [steps(runner, sizes) for sizes in ([5], [130], [500])]
    for a, b in zip(sum(got, []), sum(want, [])):
        assert torch.equal(a, b)


def test_decode_graphs_hold_the_same_launches(monkeypatch):
    def run():
        runner = made("bfloat16")
        runner.use_graphs = True
        slots = [runner.admit() for _ in range(3)]
        out = [runner.step([StepEntry(s, list(range(5 + s, 30)), [0]) for s in slots])]
        for t in range(4):  # one capture, three replays
            out.append(runner.step([StepEntry(s, [t + s], [0]) for s in slots]))
        return out

    got = run()
    monkeypatch.setattr(DecoderLM, "ALIKE_LAYERS", 10 ** 6)
    for a, b in zip(got, run()):
        assert torch.equal(a, b)


def test_layers_that_differ_or_are_watched_run_by_themselves(replays):
    runner = made("bfloat16")
    model, ops = runner.model, runner.model.ctx.ops
    model.blocks[4].mixer.scale *= 0.5  # neither stretch is long enough
    want = steps(runner, [60])[:2]
    assert not replays
    model.blocks[4].mixer.scale *= 2.0
    calls, plain = [], model.blocks[4].forward
    model.blocks[4].forward = lambda *a, **kw: (calls.append(1), plain(*a, **kw))[1]
    got = steps(runner, [60])[:2]
    assert not replays and len(calls) == 2 and not torch.equal(got[1], want[1])
    del model.blocks[4].forward
    linear = ops.linear
    ops.linear = lambda *a, **kw: (calls.append(1), linear(*a, **kw))[1]
    try:
        watched = steps(runner, [60])[:2]
    finally:
        del ops.linear
    assert not replays and len(calls) > LAYERS
    again = steps(runner, [60])[:2]
    assert replays
    for a, b, c in zip(got, watched, again):
        assert torch.equal(a, b) and torch.equal(a, c)
    # a weight that begins elsewhere: another kernel may take it
    w = model.blocks[3].mixer.o.weight
    moved = torch.empty(w.numel() + 1, dtype=w.dtype, device=w.device)[1:].view(w.shape)
    moved.copy_(w)
    model.blocks[3].mixer.o.weight = moved
    del replays[:]
    steps(runner, [60])
    assert not replays


@pytest.mark.parametrize("cls,name,a_layer", [(HipOps, "linear", 3), (HipOps, "paged_attention", 1), (PagedAttention, "forward", 1), (RMSNorm, "forward", 2)])
def test_a_function_replaced_on_its_class_is_called_for_every_layer(monkeypatch, replays, cls, name, a_layer):
    runner = made("bfloat16")
    steps(runner, [60])
    assert replays
    del replays[:]
    calls, plain = [], getattr(cls, name)
    monkeypatch.setattr(cls, name, lambda *a, **kw: (calls.append(1), plain(*a, **kw))[1])
    steps(runner, [60])
    assert not replays and len(calls) >= 2 * LAYERS * a_layer


def test_weights_that_ask_for_gradients(monkeypatch, replays):
    """Products of the library's go into tensors that are there, which torch refuses where a gradient is asked for."""
    def run():
        runner = made("bfloat16")
        for block in runner.model.blocks:
            for linear in (block.mixer.qkv, block.mixer.o, block.feed_forward.gate_up, block.feed_forward.down):
                linear.weight.requires_grad_(True)
        return steps(runner, [300, 200])

    got = run()
    assert replays
    monkeypatch.setattr(DecoderLM, "ALIKE_LAYERS", 10 ** 6)
    for a, b in zip(got, run()):
        assert torch.equal(a, b)
