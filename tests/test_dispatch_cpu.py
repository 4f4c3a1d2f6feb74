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


@pytest.mark.parametrize("B,M,N,route", [
    (32, 8192, 8192, "grid"), (8, 16384, 16384, "grid"), (1, 32768, 32768, "grid"),
    (4, 32768, 32768, "grid"), (1, 100_000, 100_000, "grid"), (8, 4096, 32768, "grid"),
    (8, 8192, 8192, "screen"), (16, 4096, 4096, "screen"), (1, 1000, 32768, "screen"),
    (32, 4096, 8192, "screen"), (32, 8192, 512, "scan"), (4, 300, 300, "scan"),
])
def test_nearest_search_takes_the_grid_where_close_clouds_need_it(monkeypatch, B, M, N, route):
    """Clouds that lie close to each other are searched fastest by the grid from
    about 2**30 pairs on; the screen's time does not depend on the data."""
    import torch

    from mps_pointops import chamfer

    taken = []
    for name in ("grid", "screen", "scan"):
        monkeypatch.setattr(chamfer, f"_nearest_{name}", lambda *a, name=name: taken.append(name))
    q, r = torch.empty(1, 1, 3).expand(B, M, 3), torch.empty(1, 1, 3).expand(B, N, 3)
    chamfer._nearest_device(q, r, None, None, 2, full=True)
    assert taken == [route]
