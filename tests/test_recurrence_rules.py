"""Which state-space steps take their chunks one after the other; what the delta rule keeps of its chunks."""
from types import SimpleNamespace

import pytest

from litellmengine_amd.csrc import build
from litellmengine_amd.csrc.ops import HipOps

CARD = SimpleNamespace(compute_units=lambda: 256)


@pytest.mark.parametrize("heads,vdim,lens,streams", [
    (32, 64, [512], True), (32, 64, [513], False), (64, 64, [2048], True), (32, 64, [1024, 1024], True),
    (4, 16, [256], True), (4, 16, [257], False), (32, 32, [300], False), (32, 32, [300] * 2, True), (8, 64, [448], True), (8, 64, [449], False),
    (64, 64, [32767], True), (64, 64, [32768], False), (64, 72, [64], False)])
def test_chunks_one_after_the_other(heads, vdim, lens, streams):
    """A chain of chunks is short, or there are workgroups enough to hide it; few workgroups of small heads are done sooner side by side."""
    assert HipOps.ssd_streams(CARD, sum(lens), heads, vdim, 128, max(lens)) == streams
    assert not HipOps.ssd_streams(CARD, sum(lens), heads, vdim, 64, max(lens))


def test_tokens_whose_chunks_a_step_keeps():
    """The delta rule's chunks of 30000 tokens of 32 heads of 64 x 64 fit what a step may keep, those of 31000 do not."""
    floats = build.load_library("delta").lle_delta_chunk_floats
    assert 0 < floats(30000, 1, 32, 64, 64) <= HipOps.DELTA_CHUNK_FLOATS < floats(31000, 1, 32, 64, 64)
    assert floats(70000, 65536, 1, 64, 64) == 0  # (more requests than a launch takes)
