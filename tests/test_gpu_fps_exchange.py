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
