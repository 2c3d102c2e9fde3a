"""How far weights are scaled up so that 64-bit fixed point holds them exactly."""
from fractions import Fraction

import pytest
import torch

from bmtk_amd.simulator import SUM_SHIFT_MAX, fixed_point_shift


class Table:
    def __init__(self, weights, targets=None):
        self.weights = torch.tensor(weights, dtype=torch.float32)
        self.indices = torch.tensor(targets if targets is not None else range(len(weights)), dtype=torch.int32)
        self.nnz = self.weights.numel()


@pytest.mark.parametrize("weights", [[0.25, -3.0, 0.0], [2.0 ** -9], [2.0 ** -9 * (1 + 2.0 ** -23)], [1.1, -0.0017, 3e-5], [2.0 ** -32, -1.0],
                                     [2.0 ** -33], [3 * 2.0 ** -70, 5 * 2.0 ** -60], [1e-30], []])
def test_smallest_shift_that_leaves_whole_multiples(weights):
    t = Table(weights)
    shift = fixed_point_shift([t], 10)
    exact = [Fraction(float(w)) * 2 ** 32 for w in t.weights]
    assert all((x * 2 ** shift).denominator == 1 for x in exact)
    assert shift == 0 or any((x * 2 ** (shift - 1)).denominator != 1 for x in exact)


def test_denormal_weights_need_more_than_there_is():
    assert fixed_point_shift([Table([1e-44])], 1) == 149 - 32 <= SUM_SHIFT_MAX
    assert fixed_point_shift([Table([1e-44, 1e-3])], 2) is None


def test_what_reaches_a_neuron_has_to_fit():
    assert fixed_point_shift([Table([2.0 ** 28] * 3, [0, 0, 0])], 1) == 0
    assert fixed_point_shift([Table([2.0 ** 28] * 4, [0, 0, 0, 0])], 1) is None
    assert fixed_point_shift([Table([2.0 ** 28] * 4, [0, 0, 1, 1])], 2) == 0
    assert fixed_point_shift([Table([2.0 ** 28] * 2, [0, 0]), Table([2.0 ** 28] * 2, [0, 0])], 1) is None   # several tables add up
    assert fixed_point_shift([Table([2.0 ** 10]), Table([2.0 ** -50])], 1) == 18
    assert fixed_point_shift([Table([2.0 ** 12]), Table([2.0 ** -50])], 1) is None
    for bad in (float("inf"), float("nan")):
        assert fixed_point_shift([Table([1.0, bad])], 2) is None
