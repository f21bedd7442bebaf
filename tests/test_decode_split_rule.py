"""Split counts of a decode launch (no GPU): their limits, and the launches whose workgroups share lists."""
import pytest

from sparseattentioninfer_amd import ops


@pytest.mark.parametrize("Hq,rows", [(32, 8), (32, 4), (16, 8), (8, 8), (32, 32), (24, 8), (28, 4), (12, 4), (24, 4), (10, 2)])
def test_counts_stay_within_their_limits(Hq, rows):
    for B in (0, 1, 2, 3, 5, 8, 13, 16, 64, 500):
        for n in (0, 1, 2, 3, 7, 8, 24, 27, 64, 129, 5000):
            s = ops.decode_splits(B, Hq, rows, n)
            assert 1 <= s <= max(1, min(32, n // 2)), (B, n, s)


@pytest.mark.parametrize("B,Hq,rows,n,want", [
    (8, 32, 8, 27, 4), (16, 32, 8, 27, 2), (64, 32, 8, 27, 1), (1, 32, 8, 500, 32), (4, 32, 4, 64, 8),   # four heads: 256 workgroups
    (8, 24, 8, 64, 8), (12, 24, 8, 27, 8), (8, 24, 8, 14, 1), (4, 24, 8, 128, 16), (4, 24, 8, 40, 8),    # three to a list
    (16, 24, 4, 128, 8), (16, 24, 4, 27, 1), (8, 24, 4, 40, 2), (3, 24, 8, 128, 3),                      # six, two to a workgroup
    (4, 32, 32, 27, 4), (3, 32, 32, 27, 5), (8, 32, 32, 27, 1), (2, 32, 32, 27, 4)])                     # a list per head
def test_workgroups_that_share_a_list(B, Hq, rows, n, want):
    assert ops.decode_splits(B, Hq, rows, n) == want
