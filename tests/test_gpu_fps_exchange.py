"""Farthest point sampling where the exchanges' candidate cut is hard: many
points at exactly the same running distance (lattices, repeated points, one
point repeated), distances spread over many octaves, points that are never
sampled, and clouds at the edges of the kernels' sizes; every index against
the oracle."""

import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _cloud(kind: str, n: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(n)
    if kind == "lattice":  # integer coordinates: most distances tie
        return torch.randint(0, 12, (2, n, 3), generator=g).float()
    if kind == "repeated":  # every point about 16 times
        base = torch.randn(2, max(n // 16, 1), 3, generator=g)
        pick = torch.randint(0, base.shape[1], (2, n), generator=g)
        return base.gather(1, pick[..., None].expand(-1, -1, 3)).contiguous()
    if kind == "one":
        return torch.ones(2, n, 3)
    x = torch.randn(2, n, 3, generator=g)
    if kind == "octaves":  # distances from 2^-60 to 2^60
        return x * torch.exp2(torch.rand(2, n, 1, generator=g) * 60 - 30)
    x[0, ::3] *= 1e-3  # "never": points at the origin, all but 5 of one cloud
    x[1, 5:] *= 1e-3
    return x


@pytest.mark.parametrize("kind", ["lattice", "repeated", "one", "octaves", "never"])
@pytest.mark.parametrize("n", [9, 511, 1024, 1025, 4096, 8193, 24576])
def test_fps_with_hard_cuts_matches_oracle(cuda_device, kind, n):
    import mps_pointops as mp

    xyz = _cloud(kind, n)
    npoint = min(n, 600)
    skip = kind == "never"
    got = mp.furthest_point_sample(xyz.cuda(), npoint, 3, skip, strategy="single")
    np.testing.assert_array_equal(got.cpu().numpy(), O.fps(xyz, npoint, 3, skip))


@pytest.mark.parametrize("sizes", [[8193, 1, 64, 700, 0, 4097], [24576, 24575, 513, 2], [9000, 512, 16384]])
def test_ragged_fps_with_a_large_cloud_matches_oracle(cuda_device, sizes):
    """Clouds of every size in one launch of the kernel the largest needs."""
    from mps_pointops import flat

    g = torch.Generator().manual_seed(len(sizes))
    x = torch.randn(sum(sizes), 3, generator=g)
    ptr = [0] + torch.tensor(sizes).cumsum(0).tolist()
    got = flat.fps(x.cuda(), ratio=0.02, random_start=False, ptr=ptr).cpu().numpy()
    want = []
    for a, b in zip(ptr, ptr[1:]):
        count = int(np.ceil(np.float32(b - a) * np.float32(0.02)))
        if count:
            want.append(a + O.fps(x[None, a:b], count, 0)[0])
    np.testing.assert_array_equal(got, np.concatenate(want))


@pytest.mark.parametrize("kind", ["lattice", "repeated", "one", "octaves", "never", "infinite"])
@pytest.mark.parametrize("n", [65, 24577, 140_000])
def test_one_cloud_over_the_chip_with_hard_cuts_matches_oracle(cuda_device, kind, n):
    """The exchanging kernels of one cloud over many workgroups, whose runs of up
    to 64 live candidates and longer ones take different code."""
    import mps_pointops as mp

    xyz = _cloud("octaves" if kind == "infinite" else kind, n)[:1].contiguous()
    if kind == "infinite":
        xyz[0, 7] = float("inf")
        xyz[0, 40, 1] = float("-inf")
    npoint = min(n, 700)
    skip = kind == "never"
    got = mp.furthest_point_sample(xyz.cuda(), npoint, 3, skip, strategy="multigroup")
    np.testing.assert_array_equal(got.cpu().numpy(), O.fps(xyz, npoint, 3, skip))


@pytest.mark.parametrize("n,side", [(8193, 4), (9000, 10), (16384, 13), (24576, 29)])
def test_lattices_beyond_8192_points(cuda_device, n, side):
    """Runs that go on through points at one distance: the indices, and a time
    below that of the kernel that takes one step at a time whatever the data (it
    was up to twice that when each such step cost an exchange)."""
    import mps_pointops as mp
    from mps_pointops import _native

    g = torch.Generator().manual_seed(n)
    xyz = torch.randint(0, side, (2, n, 3), generator=g).float()
    x, npoint = xyz.cuda(), 1000
    got = mp.furthest_point_sample(x, npoint, 3)
    np.testing.assert_array_equal(got.cpu().numpy(), O.fps(xyz, npoint, 3))
    ptr, out_ptr = (torch.tensor([0, m, 2 * m], device="cuda") for m in (n, npoint))
    starts = torch.full((2,), 3, device="cuda")
    out = torch.empty(2 * npoint, dtype=torch.long, device="cuda")
    scratch = torch.empty(2 * n, device="cuda")

    def stepwise():
        _native.call("pointops_fps_flat", x.data_ptr(), ptr.data_ptr(), out_ptr.data_ptr(),
                     starts.data_ptr(), out.data_ptr(), scratch.data_ptr(), 2, 2 * n, n,
                     _native.stream(x.device))

    times = []
    for call in (stepwise, lambda: mp.furthest_point_sample(x, npoint, 3)):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        call()
        each = []
        for _ in range(5):
            begin.record()
            call()
            end.record()
            end.synchronize()
            each.append(begin.elapsed_time(end))
        times.append(min(each))
    assert torch.equal(out.view(2, -1) - torch.tensor([[0], [n]], device="cuda"), got)
    assert times[1] < times[0]


def test_threads_sampling_clouds_of_different_sizes(cuda_device):
    """The kernel's dynamic LDS differs per call, its limit belongs to the
    process: calls of several threads leave each other's alone."""
    from concurrent.futures import ThreadPoolExecutor

    import mps_pointops as mp

    clouds = [torch.rand(1, n, 3, generator=torch.Generator().manual_seed(n)).cuda()
              for n in (8193, 24576, 12000, 20000)]
    want = [mp.furthest_point_sample(x, 64) for x in clouds]

    def sample(i):
        return i % 4, mp.furthest_point_sample(clouds[i % 4], 64)

    with ThreadPoolExecutor(4) as pool:
        for i, got in pool.map(sample, range(80)):
            assert torch.equal(got, want[i])


def test_unaligned_scratch_is_served(cuda_device):
    """Scratch at any 4-byte boundary, as the running distances need: the
    kernel that reads 16 bytes at a time is left out."""
    from mps_pointops import _native

    n = 9000
    xyz = torch.rand(1, n, 3, generator=torch.Generator().manual_seed(1))
    x, out = xyz.cuda(), torch.empty(1, 100, dtype=torch.long, device="cuda")
    size = _native.size_query("pointops_fps_dense_scratch_bytes", 1, n)
    scratch = torch.empty(size + 16, dtype=torch.uint8, device="cuda")
    for offset in (0, 4):
        _native.call("pointops_fps_dense", x.data_ptr(), out.data_ptr(), scratch.data_ptr() + offset,
                     1, n, 100, 0, 0, _native.stream(x.device))
        np.testing.assert_array_equal(out.cpu().numpy(), O.fps(xyz, 100, 0))
