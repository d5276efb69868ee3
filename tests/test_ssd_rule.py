"""Which state-space steps take their chunks one after the other."""
from types import SimpleNamespace

import pytest

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
