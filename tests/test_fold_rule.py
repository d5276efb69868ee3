"""Which attention layers let a norm's work go into the products around it."""
import pytest
import torch

from litellmengine_amd.parts import PagedAttention, RotaryHalfSplit
from litellmengine_amd.parts.base import BuildContext


@pytest.mark.parametrize("nq,d", [(3, 26), (1, 6), (5, 2), (2, 26), (3, 32)])
def test_float32_heads_whose_columns_are_no_fours(nq, d):
    """The output projection of 78, 6 or 10 columns takes the plain float32 product, which knows no folded norm."""
    hidden = 512
    mixer = PagedAttention("a.", hidden, nq, 1, d, RotaryHalfSplit(d, 1e4), qk_norm_eps=1e-6)
    weights = {name: torch.ones(spec.shape) for name, spec in mixer.tensor_specs().items()}
    mixer.bind(weights, BuildContext(dtype=torch.float32, device=torch.device("cpu"), ops=None))
    assert mixer.folds_norm == (nq * d % 4 == 0)
