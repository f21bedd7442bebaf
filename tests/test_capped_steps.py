"""The closed form of the patterns' block counts against the sum it stands for."""
from sparseattentioninfer_amd.patterns.base import capped_steps


def test_capped_steps_is_the_sum():
    for first in range(0, 9):
        for n in range(0, 9):
            for cap in range(0, 12):
                assert capped_steps(first, n, cap) == sum(min(first + i, cap) for i in range(n)), (first, n, cap)
