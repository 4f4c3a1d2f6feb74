"""The rules that send a search to the screened entry points, at the lines
where they change (no GPU: sizes only)."""

import pytest


@pytest.mark.parametrize("rows", [2**31 - 64, 2**31, 2**32])
def test_searches_beyond_the_screens_limits_are_scanned(rows):
    """The ragged screen refuses 2**31 - 64 reference rows and more, which the
    ragged scan takes."""
    from mps_pointops import flat, ops

    for D in (3, 64):
        assert not flat._screened(rows, 1 << 20, 4, D, 16)
        assert not ops._screened(rows >> 14, 1 << 10, 1 << 14, D, 16)
        assert flat._screened(1 << 20, 1 << 20, 4, D, 16)
