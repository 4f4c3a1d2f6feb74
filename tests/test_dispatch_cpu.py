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
    (4, 32768, 32768, "grid"), (1, 100_000, 100_000, "grid"), (8, 4096, 32768, "grid"), (1, 4096, 32768, "grid"),
    (1, 16384, 16384, "screen"),
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


@pytest.mark.parametrize("B,M,N,D,k,screened", [
    (4096, 16, 16, 8, 4, False), (65536, 16, 16, 8, 4, False), (16384, 8, 32, 8, 4, False),
    (1024, 32, 32, 8, 8, False), (1024, 64, 32, 16, 8, True), (1024, 64, 64, 8, 8, True),
    (1000, 1, 2000, 8, 8, False), (1024, 16, 1024, 8, 8, False), (1024, 24, 1024, 8, 8, True),
    (1024, 16, 1024, 64, 8, True), (2048, 1, 1024, 64, 8, False), (64, 1, 20000, 16, 8, True),
    (512, 64, 64, 64, 16, False), (512, 64, 96, 64, 16, True), (512, 64, 64, 64, 33, True),
    (8, 2048, 2048, 64, 20, True), (1, 2048, 500, 33, 10, False),
])
def test_feature_searches_are_screened_where_a_block_has_queries_enough(B, M, N, D, k, screened):
    from mps_pointops import ops

    assert ops._screened(B, M, N, D, k) is screened


@pytest.mark.parametrize("clouds,x,y,D,k,screened", [
    (16384, 64, 1, 3, 8, False), (1024, 256, 8, 3, 8, False), (1024, 256, 24, 3, 8, True),
    (1024, 1024, 4, 3, 16, False), (256, 1024, 16, 3, 16, True), (53, 20000, 1, 3, 16, True),
    (32, 1024, 32, 3, 1, False), (128, 1024, 32, 3, 1, True), (4096, 128, 8, 16, 8, False),
    (512, 256, 24, 16, 8, True), (8192, 128, 4, 64, 16, False), (2048, 128, 8, 64, 16, True),
    (3, 20000, 20000, 3, 16, True), (32, 1000, 1000, 3, 16, True), (5000, 16, 16, 3, 8, False),
])
def test_ragged_searches_are_screened_where_a_cloud_has_queries_enough(clouds, x, y, D, k, screened):
    from mps_pointops import flat

    assert flat._screened(clouds * x, clouds * y, clouds, D, k) is screened
