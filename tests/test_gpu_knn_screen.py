"""The screened kNN (pointops_knn_screen, pointops_knn_flat_screen) against the
scanning entry points, bit for bit, over the forms it accepts: edges of its
tiles, blocks and feature steps, the smallest and largest K, inputs that make
the screen loose (far from the origin, spread over octaves), that list too
many references (copies of one point), and that it must not serve (coordinates
that are not finite or too large)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(kind: str, g: torch.Generator, *shape: int) -> torch.Tensor:
    x = torch.randn(*shape, generator=g)
    if kind == "far":
        return x + 3000.0
    if kind == "octaves":
        return x * torch.exp2(torch.rand(*shape[:-1], 1, generator=g) * 40 - 20)
    if kind == "lattice":
        return (x * 3).round()
    if kind == "copies":  # most rows are one point
        same = torch.rand(*shape[:-1], 1, generator=g) < 0.7
        return torch.where(same, torch.ones(()), x)
    if kind == "outlier":  # one row far from all others
        x.view(-1, shape[-1])[0] = 1e6
        return x
    if kind == "tiny":
        return x * 1e-25
    if kind == "huge":
        return x * 1e17
    if kind == "overflow":  # squared distances beyond float32
        return x * 1e20
    if kind == "bad":  # a few rows that are not finite
        at = torch.rand(*shape[:-1], 1, generator=g)
        x = torch.where(at < 0.004, torch.tensor(float("inf")), x)
        return torch.where(at > 0.996, torch.tensor(float("nan")), x)
    return x


def _dense(q, r, k, screen):
    from mps_pointops import _native

    B, M, D = q.shape
    N = r.shape[1]
    dist = torch.full((B, M, k), -7.0, device="cuda")
    idx = torch.full((B, M, k), -7, dtype=torch.long, device="cuda")
    args = (q.data_ptr(), r.data_ptr(), dist.data_ptr(), idx.data_ptr())
    st = _native.stream(q.device)
    if screen:
        ws = torch.empty(_native.size_query("pointops_knn_screen_workspace_bytes", B, N, D),
                         dtype=torch.uint8, device="cuda")
        _native.call("pointops_knn_screen", *args, ws.data_ptr(), B, M, N, D, k, st)
    elif D == 3:
        # More than 64 neighbours (or fewer than 256 references): scanned.
        wide = k if N < 256 else min(N, 65)
        dist, idx = dist.new_empty(B, M, wide), idx.new_empty(B, M, wide)
        _native.call("pointops_knn3", q.data_ptr(), r.data_ptr(), dist.data_ptr(), idx.data_ptr(),
                     B, M, N, wide, st)
        return dist[..., :k], idx[..., :k]
    else:
        _native.call("pointops_knn_feat", *args, B, M, N, D, k, st)
    return dist, idx


@pytest.mark.parametrize("kind", ["normal", "far", "octaves", "lattice", "copies", "tiny", "huge",
                                  "overflow", "outlier", "bad"])
@pytest.mark.parametrize("D", [1, 3, 16, 33, 64, 100, 128])
@pytest.mark.parametrize("B,M,N,k", [(2, 65, 31, 1), (3, 130, 1000, 20), (1, 64, 33, 33), (2, 100, 256, 9),
                                     (1, 70, 511, 8),
                                     (2, 63, 2049, 64)])
def test_screen_matches_scan(cuda_device, kind, D, B, M, N, k):
    from mps_pointops import _native

    g = torch.Generator().manual_seed(D * 7 + N)
    r = _rows(kind, g, B, N, D)
    q = r[:, torch.randperm(N, generator=g)[:M]] if M < N else _rows(kind, g, B, M, D)
    print(f"screen {kind} D={D} B={B} M={M} N={N} k={k}", flush=True)
    q, r = q.cuda().contiguous(), r.cuda().contiguous()
    want = _dense(q, r, k, False)
    got = _dense(q, r, k, True)
    assert torch.equal(got[1], want[1])
    assert torch.equal(got[0], want[0])
    if D == 3:  # screened without a workspace from 256 or 512 references
        dist, idx = torch.empty_like(got[0]), torch.empty_like(got[1])
        _native.call("pointops_knn3", q.data_ptr(), r.data_ptr(), dist.data_ptr(), idx.data_ptr(),
                     B, M, N, k, _native.stream(q.device))
        assert torch.equal(idx, want[1])
        assert torch.equal(dist, want[0])


@pytest.mark.parametrize("kind", ["normal", "far", "copies", "bad"])
@pytest.mark.parametrize("D", [3, 40])
@pytest.mark.parametrize("sizes_x,sizes_y,k", [
    ([5, 0, 300, 64, 33, 1], [70, 3, 0, 64, 129, 1], 16),
    ([31, 32, 33, 2000], [65, 64, 63, 500], 64),
    ([1], [200], 3),
])
def test_flat_screen_matches_scan(cuda_device, kind, D, sizes_x, sizes_y, k):
    from mps_pointops import _native

    g = torch.Generator().manual_seed(D + k)
    x, y = _rows(kind, g, sum(sizes_x), D).cuda(), _rows(kind, g, sum(sizes_y), D).cuda()
    px = torch.tensor([0, *sizes_x]).cumsum(0).cuda()
    py = torch.tensor([0, *sizes_y]).cumsum(0).cuda()
    st = _native.stream(x.device)
    want = torch.full((len(y), k), -7, dtype=torch.long, device="cuda")
    _native.call("pointops_knn_flat", y.data_ptr(), x.data_ptr(), py.data_ptr(), px.data_ptr(),
                 want.data_ptr(), len(y), len(sizes_x), D, k, st)
    ws = torch.empty(_native.size_query("pointops_knn_flat_screen_workspace_bytes", len(x),
                                        len(sizes_x), D), dtype=torch.uint8, device="cuda")
    got = torch.full_like(want, -8)
    _native.call("pointops_knn_flat_screen", y.data_ptr(), x.data_ptr(), py.data_ptr(),
                 px.data_ptr(), got.data_ptr(), ws.data_ptr(), len(y), len(x), len(sizes_x), D, k,
                 st)
    assert torch.equal(got, want)


@pytest.mark.parametrize("kind", ["uniform", "lattice", "copies", "far", "overflow"])
@pytest.mark.parametrize("B,M,N", [(3, 1, 512), (2, 63, 513), (1, 65, 1023), (2, 300, 4097), (1, 1000, 32768)])
def test_nearest_screen_matches_scan(cuda_device, kind, B, M, N):
    """The Chamfer loss's nearest reference and squared distance, bit for bit:
    ties, more copies of one point than a list holds, clouds far from the
    origin, distances that overflow."""
    from mps_pointops import chamfer

    g = torch.Generator().manual_seed(B * M + N)
    q, r = torch.rand(B, M, 3, generator=g), torch.rand(B, N, 3, generator=g)
    if kind == "lattice":
        q, r = (q * 6).round(), (r * 6).round()
    elif kind == "copies":
        r[:, : N // 2] = q[:, :1]
    elif kind == "far":
        q, r = q + 1e4, r + 1e4
    elif kind == "overflow":
        q[:, ::2] *= 3e19
        r[:, 1::3] *= -3e19
    q, r = q.cuda(), r.cuda()
    assert chamfer._screen_eligible(q, r, 2, True)
    lengths = [torch.full((B,), n, dtype=torch.int64, device=q.device) for n in (M, N)]
    d, i = chamfer._nearest_device(q, r, *lengths, 2, full=True)
    want_d, want_i = chamfer._nearest_scan(q, r, *lengths, 2)
    assert torch.equal(i, want_i)
    assert torch.equal(d.view(torch.int32), want_d.view(torch.int32))
