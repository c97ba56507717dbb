"""The ensemble's layout without a GPU: the search that is off, and the assignment that replaces it."""

import pytest

from wrfdc.ensemble import assign_longest_first, autotune


def test_autotune_is_off_before_it_touches_a_domain():
    class Untouchable:
        def __getattr__(self, name):
            raise AssertionError(f"autotune read {name}")

    with pytest.raises(RuntimeError, match="is off"):
        autotune([Untouchable()])


def test_longest_first():
    assert assign_longest_first([5.0, 9.0, 3.0, 4.0], 2) == [1, 0, 0, 1]
    assert assign_longest_first([1.0], 16) == [0]
