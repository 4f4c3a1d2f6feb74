"""The device checks and edge lists (checks.hip) against tensor operations:
values at the limits in every position a block or a wave can hold them, ids
with gaps, and rows without edges."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 256, 257, 1024 * 256 + 1]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n", SIZES)
def test_range_check(cuda_device, dtype, n):
    from mps_pointops import _native

    v = torch.randint(0, 10, (n,), dtype=dtype, device="cuda")
    low, high = v.clone(), v.clone()
    low[0], high[-1] = -1, 10
    assert _native.outside([(v, 0, 9), (low, 0, 9), (high, 0, 9), (low, -1, 9)]) == [
        False, True, True, False]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_finite_check_looks_below_the_lengths(cuda_device, dtype):
    from mps_pointops import _native

    x = torch.randn(3, 70, 5, dtype=dtype, device="cuda")
    lengths = torch.tensor([70, 0, 69], device="cuda")
    x[1] = float("nan")
    x[2, 69] = float("inf")
    bad = x.clone()
    bad[2, 68, 4] = -float("inf")
    assert _native.nonfinite([(x, lengths), (bad, lengths), (x, None), (x[:1], None)]) == [
        False, True, True, False]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("n", SIZES)
def test_batch_vectors(cuda_device, dtype, n):
    from mps_pointops import flat

    g = torch.Generator().manual_seed(n)
    ids = torch.randint(0, 40, (n,), generator=g).sort().values * 3  # gaps
    dev = ids.to(dtype).cuda()
    assert flat._clouds_in([(dev, n, dev.device, "batch")]) == [int(ids[-1]) + 1]
    clouds = int(ids[-1]) + 4
    want = torch.searchsorted(ids, torch.arange(clouds + 1))
    assert torch.equal(flat._offsets(dev, n, dev.device, clouds).cpu(), want)
    for at in {0, n // 2, n - 1}:
        wrong = dev.clone()
        wrong[at] = -1 if at == 0 else wrong[at - 1] - 1
        with pytest.raises(ValueError, match="sorted"):
            flat._clouds_in([(wrong, n, dev.device, "batch")])


@pytest.mark.parametrize("Q,K", [(1, 1), (5, 64), (300, 65), (70, 130)])
def test_edge_lists(cuda_device, Q, K):
    from mps_pointops import flat

    g = torch.Generator().manual_seed(Q)
    table = torch.randint(-Q, Q, (Q, K), generator=g).clamp_min(-1).cuda()
    table[Q // 2] = -1
    q, k = torch.nonzero(table >= 0, as_tuple=True)
    edges = torch.stack((q, table[q, k]))
    assert torch.equal(flat._edge_index(table), edges)
    open_edges = edges[:, edges[0] != edges[1]]
    assert torch.equal(flat._edge_index(table, True), open_edges)
    assert torch.equal(flat._edge_index(table, True, True), open_edges.flip(0))
