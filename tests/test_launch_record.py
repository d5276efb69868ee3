"""What may be launched again for another layer: launches whose operands are whole tensors, parts and operations that are as they were written."""
import ctypes

import pytest
import torch

from litellmengine_amd.config import Qwen3Config, get_architecture
from litellmengine_amd.csrc.record import LaunchRecord, Replay
from litellmengine_amd.parts import PagedAttention
from litellmengine_amd.parts.base import Norm, parts_as_written
from litellmengine_amd.parts.norm import RMSNorm


def replay_of(pointer):
    """(a Replay of one launch that takes `pointer(weight, given, left, made)`, the addresses that it launches with for another weight)"""
    weight, other, given, left, made = (torch.zeros(64) for _ in range(5))
    record, seen = LaunchRecord(0), []

    def launch(*args):
        seen.append(args)
        return 0

    launch.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    record.launch(launch, "lib", "name", (weight.data_ptr(), pointer(weight, given, left, made)), 0)
    replay = Replay(record, [weight], [given], [left])
    if replay.ok:
        assert replay.run([other], [other.data_ptr()]) is None
        assert seen[0][0] == other.data_ptr()
    return replay, seen, left


def test_a_launch_that_reads_what_was_taken_over():
    replay, seen, left = replay_of(lambda weight, given, left, made: given.data_ptr())
    assert replay.ok and seen[0][1] == left.data_ptr()
    replay, seen, _ = replay_of(lambda weight, given, left, made: made.data_ptr() + 16)
    assert replay.ok and len(seen) == 1


@pytest.mark.parametrize("pointer", [lambda weight, given, left, made: given.data_ptr() + 16, lambda weight, given, left, made: weight.data_ptr() + 16])
def test_a_launch_that_points_inside_a_tensor_is_not_launched_again(pointer):
    """Inside an operand, or inside what the layer before has left: the other layer's place is not known."""
    assert not replay_of(pointer)[0].ok


def blocks():
    config = Qwen3Config.from_dict({
        "architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "num_hidden_layers": 2, "hidden_size": 64, "num_attention_heads": 2,
        "num_key_value_heads": 1, "head_dim": 32, "intermediate_size": 96, "vocab_size": 100, "rope_theta": 1e6, "rms_norm_eps": 1e-6})
    return get_architecture(config.architecture).build(config).blocks


PARTS = [(lambda b: b, ["forward", "entry_norm", "chained_norm", "input_norm"]), (lambda b: b.norm_in, ["forward", "fold"]),
         (lambda b: b.norm_post, ["forward", "fold"]), (lambda b: b.mixer, ["forward"]), (lambda b: b.feed_forward, ["forward"]),
         (lambda b: b.mixer.qkv, ["forward"]), (lambda b: b.mixer.o, ["forward"]), (lambda b: b.feed_forward.down, ["forward"]),
         (lambda b: b.mixer.position, ["fused_rotary"])]


@pytest.mark.parametrize("part,names", PARTS)
def test_a_part_with_a_function_of_its_own(part, names):
    """Whichever function that a pass calls a caller has replaced on a part, its block says no launches until it is gone again."""
    block, other = blocks()
    assert block.launches() is not None
    p = part(block)
    for name in names:
        plain = getattr(p, name)
        setattr(p, name, lambda *a, **kw: plain(*a, **kw))
        assert block.launches() is None and other.launches() is not None
        delattr(p, name)
        assert block.launches() is not None


@pytest.mark.parametrize("cls,name", [(PagedAttention, "forward"), (RMSNorm, "forward"), (PagedAttention, "entry"), (Norm, "fold")])
def test_a_class_with_another_function(cls, name, monkeypatch):
    """Replaced, added over a base's, or replaced on a base."""
    assert parts_as_written()
    monkeypatch.setattr(cls, name, lambda self, *a: None, raising=False)
    assert not parts_as_written()
    monkeypatch.undo()
    assert parts_as_written()


def test_results_made_after_a_tracing_mode():
    """What a mode of fake tensors has made is not what later results are made like."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from litellmengine_amd.csrc import ops

    kind, cpu = torch.float64, torch.device("cpu")
    with FakeTensorMode():
        ops._made((2,), dtype=kind, device=cpu)
    try:
        assert type(ops._made((2,), dtype=kind, device=cpu)) is torch.Tensor
    finally:
        ops._of_kind.pop((kind, cpu), None)
