"""What may be launched again for another layer: launches whose operands are whole tensors."""
import ctypes

import pytest
import torch

from litellmengine_amd.csrc.record import LaunchRecord, Replay


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
