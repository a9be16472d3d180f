"""The prefetch rule of test_prefetch_rule.py at even L that are no multiple
of 8 (half-rows that end inside a Philox block)."""
import pytest

from test_prefetch_rule import test_prefetched_sites_are_not_written_by_the_chunk_before as check


@pytest.mark.parametrize("L", [10, 18, 34, 50, 66, 98, 100, 126, 130, 138, 182, 254])
def test_even_sizes(L):
    check(L)
