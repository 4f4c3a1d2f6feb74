"""Searches screened on the matrix cores over inputs that once made the screen
useless: results against the scanning entry points, and times against the same
search of ordinary input.  The times are minima of several calls and their limits
lie well above what is measured (an order of magnitude below what they caught)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# (B, M, N, D, k): config 2's search, a small one (no workspace), features
SHAPES = [(32, 1024, 4096, 3, 16), (16, 512, 1024, 3, 16), (8, 1024, 2048, 64, 20)]


def _best(call) -> float:
    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(3):
        call()
    times = []
    for _ in range(5):
        begin.record()
        for _ in range(10):
            call()
        end.record()
        end.synchronize()
        times.append(begin.elapsed_time(end))
    return min(times)


def _cloud(shape):
    B, M, N, D, k = shape
    g = torch.Generator().manual_seed(N + D)
    r = torch.rand(B, N, D, generator=g) if D == 3 else torch.randn(B, N, D, generator=g)
    return r.cuda(), torch.randperm(N, generator=g)[:M].cuda(), k


def _scan(q, r, k):
    """The same search by the entry points' scan: more than 64 neighbours."""
    from mps_pointops import _native

    B, M, D = q.shape
    wide = 65
    dist = torch.empty(B, M, wide, device="cuda")
    idx = torch.empty(B, M, wide, dtype=torch.long, device="cuda")
    args = (q.data_ptr(), r.data_ptr(), dist.data_ptr(), idx.data_ptr(), B, M, r.shape[1])
    if D == 3:
        _native.call("pointops_knn3", *args, wide, _native.stream(q.device))
    else:
        _native.call("pointops_knn_feat", *args, D, wide, _native.stream(q.device))
    return dist[..., :k], idx[..., :k]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("value", [20.0, 1e3, 1e6, 1e30, float("inf"), float("nan")])
@pytest.mark.parametrize("at", [7, 0])
def test_one_stray_reference_costs_itself(cuda_device, shape, value, at):
    import mps_pointops as mp

    r, pick, k = _cloud(shape)
    pick = torch.where(pick == at, at + 1, pick)  # (the stray asks nothing)
    q = r[:, pick].contiguous()
    plain = _best(lambda: mp.knn(q, r, k))
    r[:, at] = value
    got = mp.knn(q, r, k)
    want = _scan(q, r, k)
    assert torch.equal(got[1], want[1])
    assert torch.equal(got[0], want[0])
    assert _best(lambda: mp.knn(q, r, k)) < 1.5 * plain


@pytest.mark.parametrize("value", [50.0, float("nan")])
def test_strays_of_ragged_clouds_cost_themselves(cuda_device, value):
    from mps_pointops import flat

    sizes = [20000, 15000, 25000]
    x = torch.rand(sum(sizes), 3, generator=torch.Generator().manual_seed(1)).cuda()
    ptr = torch.tensor([0, *sizes]).cumsum(0).cuda()
    y = x.clone()
    plain = _best(lambda: flat.knn_indices(x, y, ptr, ptr, 16))
    x[::5000] = value
    assert _best(lambda: flat.knn_indices(x, y, ptr, ptr, 16)) < 1.5 * plain


def _copies(r, g):
    r[:, r.shape[1] // 2:] = 0.0
    return r


def _clusters(r, g):
    B, N, D = r.shape
    centre = torch.randn(B, 16, D, generator=g).cuda()
    which = torch.randint(0, 16, (B, N, 1), generator=g).cuda().expand(-1, -1, D)
    return centre.gather(1, which) + 0.05 * r


def _lattice(r, g):
    return (r * 4).round()


@pytest.mark.parametrize("shape", SHAPES + [(1, 700, 20000, 3, 64), (2, 70, 9000, 3, 1), (1, 100, 5000, 40, 33)])
@pytest.mark.parametrize("kind", [_copies, _clusters, _lattice])
@pytest.mark.parametrize("few", [False, True])
def test_queries_left_over(cuda_device, shape, kind, few):
    """More references within the limit than a list holds, for all or a few of
    a block's queries (which the waves then share), over one and several ranges
    of tiles."""
    from mps_pointops import ops

    r, pick, k = _cloud(shape)
    g = torch.Generator().manual_seed(7)
    r = kind(r, g).contiguous()
    q = r[:, pick].contiguous()
    if few:  # only every 50th query lies among them
        keep = torch.arange(q.shape[1], device="cuda") % 50 == 0
        q = torch.where(keep[:, None], q, q + 3.0 + torch.rand(q.shape, generator=g).cuda())
    from mps_pointops import _native

    want = _scan(q, r, k)
    dist, idx = torch.empty_like(want[0]).contiguous(), torch.empty_like(want[1]).contiguous()
    B, M, D = q.shape
    N = r.shape[1]
    ws = torch.empty(_native.size_query("pointops_knn_screen_workspace_bytes", B, N, D),
                     dtype=torch.uint8, device="cuda")
    _native.call("pointops_knn_screen", q.data_ptr(), r.data_ptr(), dist.data_ptr(), idx.data_ptr(),
                 ws.data_ptr(), B, M, N, D, k, _native.stream(q.device))
    assert torch.equal(idx, want[1])
    assert torch.equal(dist, want[0])
    got = ops.knn(q, r, k)  # whichever entry point serves it
    assert torch.equal(got[1], want[1])
    assert torch.equal(got[0], want[0])


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", [_copies, _clusters])
def test_queries_left_over_take_no_longer_than_a_scan(cuda_device, shape, kind):
    """Against the scan of the same pairs (more than 64 neighbours), which needs
    several times as long as the search of ordinary input."""
    import mps_pointops as mp

    r, pick, k = _cloud(shape)
    r = kind(r, torch.Generator().manual_seed(7)).contiguous()
    q = r[:, pick].contiguous()
    assert _best(lambda: mp.knn(q, r, k)) < _best(lambda: _scan(q, r, k))


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,M,N,k", [(128, 24, 1, 1), (128, 24, 33, 8), (64, 90, 95, 9), (3, 3000, 127, 16),
                                     (130, 64, 64, 17), (128, 63, 32, 32), (200, 12, 31, 8)])
@pytest.mark.parametrize("kind", ["normal", "copies", "bad"])
def test_small_feature_clouds_match_oracle(cuda_device, D, B, M, N, k, kind):
    """The lane kernel's range: the edges of its rule, one to its largest number
    of references, ties and rows that are not finite."""
    import numpy as np

    import mps_pointops as mp
    from oracle import oracle as O

    g = torch.Generator().manual_seed(N + k)
    r, q = torch.randn(B, N, D, generator=g), torch.randn(B, M, D, generator=g)
    if kind == "copies":
        r[:, ::2] = q[:, :1]
    elif kind == "bad":
        r[:, 0] = float("nan")
        q[:, 1, 3] = float("inf")
    dist, idx = mp.knn(q.cuda(), r.cuda(), k)
    want_d, want_i = O.knn_feat(q, r, k)
    np.testing.assert_array_equal(idx.cpu().numpy(), want_i)
    np.testing.assert_array_equal(dist.cpu().numpy().view(np.int32), np.asarray(want_d).view(np.int32))


@pytest.mark.parametrize("kind", [_copies, _clusters, _lattice])
@pytest.mark.parametrize("D,k", [(3, 1), (3, 64), (20, 16)])
@pytest.mark.parametrize("sizes_x,sizes_y", [([9000, 31, 0, 4064], [70, 3, 5, 130]), ([12097], [700])])
def test_ragged_queries_left_over(cuda_device, kind, D, k, sizes_x, sizes_y):
    """The same over ragged clouds, of one and several ranges of tiles."""
    from mps_pointops import _native

    g = torch.Generator().manual_seed(k + D)
    x = kind(torch.rand(1, sum(sizes_x), D, generator=g).cuda(), g)[0].contiguous()
    y = x[torch.randint(0, len(x), (sum(sizes_y),), generator=g).cuda()].contiguous()
    px, py = (torch.tensor([0, *s]).cumsum(0).cuda() for s in (sizes_x, sizes_y))
    want, got = (torch.full((len(y), k), f, dtype=torch.long, device="cuda") for f in (-7, -8))
    st = _native.stream(x.device)
    args = (y.data_ptr(), x.data_ptr(), py.data_ptr(), px.data_ptr())
    _native.call("pointops_knn_flat", *args, want.data_ptr(), len(y), len(sizes_x), D, k, st)
    ws = torch.empty(_native.size_query("pointops_knn_flat_screen_workspace_bytes", len(x), len(sizes_x), D),
                     dtype=torch.uint8, device="cuda")
    _native.call("pointops_knn_flat_screen", *args, got.data_ptr(), ws.data_ptr(), len(y), len(x),
                 len(sizes_x), D, k, st)
    assert torch.equal(got, want)


@pytest.mark.parametrize("B,M,N", [(2, 4096, 9000), (1, 5000, 32768), (1, 4100, 33000)])
@pytest.mark.parametrize("kind", ["stray", "shift", "far", "copies", "lattice"])
def test_nearest_by_the_grid_and_the_screen(cuda_device, B, M, N, kind):
    """Queries that the grid leaves to the screen (none, some, all of them, and
    those of crowded cells), on both sides of its limits' line, against the scan."""
    from mps_pointops import chamfer

    g = torch.Generator().manual_seed(N)
    r = torch.randn(B, N, 3, generator=g)
    r = r / r.norm(dim=-1, keepdim=True)
    q = r[:, torch.randint(0, N, (M,), generator=g)] + 0.01 * torch.randn(B, M, 3, generator=g)
    if kind == "stray":
        r[:, 7] = 50.0
    elif kind == "shift":
        q = q + 0.4
    elif kind == "far":
        q[:, ::10] = 2 * torch.rand(B, len(range(0, M, 10)), 3, generator=g) - 1
    elif kind == "copies":
        r[:, N // 2:], q[:, M // 2:] = 0.0, 0.0
    elif kind == "lattice":
        r, q = (r * 10).round(), (q * 10).round() + 0.5
    q, r = q.cuda().contiguous(), r.cuda().contiguous()
    lengths = [torch.full((B,), n, dtype=torch.int64, device=q.device) for n in (M, N)]
    d, i = chamfer._nearest_grid(q, r)
    want_d, want_i = chamfer._nearest_scan(q, r, *lengths, 2)
    assert torch.equal(i, want_i)
    assert torch.equal(d.view(torch.int32), want_d.view(torch.int32))
