"""The timed tile choice of the modes that fold in FP32: candidates that measure the same give the same order of sums in
every process, and the mid tile's own K pieces only run where they are clearly faster (CPU, with given timings)."""
import pytest

from wgpkernels_amd import int8 as wq

# mode, whether the mid tile's split 1 is in K pieces of its own, timings in us, the choice
CASES = [
    ("block", False, {(10, 1): 1990, (10, 0): 2003}, (10, 0)),                                     # the same: whole K
    ("block", False, {(10, 1): 2003, (10, 0): 1990}, (10, 0)),
    ("block", False, {(10, 1): 133.0, (10, 0): 137.0}, (10, 1)),                                   # the split 3% faster
    ("block", True, {(10, 1): 62.2, (10, 0): 105.0, (18, 1): 58.7, (18, 0): 75.0}, (10, 1)),       # 6%: the long tile's pieces
    ("block", True, {(10, 1): 51.4, (10, 0): 104.0, (18, 1): 40.8, (18, 0): 53.4}, (18, 1)),       # 26%: its own
    ("block", True, {(10, 1): 62.2, (10, 0): 59.5, (18, 1): 58.7, (18, 0): 59.0}, (18, 0)),
    ("block", False, {(10, 1): 52.4, (10, 0): 53.7, (18, 1): 51.9, (18, 0): 52.0}, (18, 0)),       # mid, whole K either way
    ("block+g", True, {(12, 1): 77.4, (12, 0): 169.0, (19, 1): 76.7, (19, 0): 110.0}, (12, 1)),
    ("block+g", False, {(12, 1): 131.0, (12, 0): 180.0, (19, 1): 132.0, (19, 0): 132.0}, (12, 1)),  # another tile: the fastest
    ("exact+g", True, {(14, 1): 40.3, (14, 0): 80.0, (20, 1): 39.0, (20, 0): 60.0}, (20, 1)),      # another order in any case
    ("row", True, {(0, 1): 30.0, (0, 0): 30.2, (16, 1): 29.9, (16, 0): 31.0}, (16, 1)),            # INT32 sums: the fastest
    ("exact", True, {(1, 1): 30.0, (1, 0): 30.2}, (1, 1)),
]


@pytest.mark.parametrize("mode,own,timings,expected", CASES)
def test_choice_keeps_the_order_of_sums(monkeypatch, mode, own, timings, expected):
    class Library:
        def wq8_gemm_workspace(self, m, n, k, variant, cus, split, sizes):
            sizes[0], sizes[1] = 4096 if own else 0, 0

    monkeypatch.setattr(wq, "library", Library)
    assert wq._choose_tile(mode, timings, 512, 5120, 13824, 256) == expected
