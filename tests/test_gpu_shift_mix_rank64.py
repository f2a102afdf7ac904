"""Rank 64: a step of the token sums goes through the kernel's tiles in two parts of the rank's columns."""
import pytest
import torch

from test_gpu_shift_mix import test_layer_forward_and_backward_edges as _edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,C,wdt", [
    (1, 31, 64, torch.float32),          # less than one step, one workgroup
    (1, 33, 128, torch.bfloat16),        # one token into the second step
    (2, 2080, 64, torch.float32),        # a range boundary every 32 tokens
    (1, 4129, 2048, torch.float32),      # several steps a range (an odd and an even number of parts), the last range one token into a step
])
def test_parts_of_a_step(oracle, B, T, C, wdt):
    _edges(oracle, B, T, C, 64, wdt)
