"""The row kernels of the point-transformer layers (pointops_group_rows, its
backward, pointops_knn_finish) against the tensor operations they replace:
outputs bit for bit, gradients within the rounding of a float32 sum in another
order, second derivatives, missing neighbours, both index widths."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# A point's gradient sums at most 200 terms of magnitude below about 5 here;
# two orders of such a sum differ by at most 2 * 200 * 2**-24 of their total.
TOL = 200 * 5 * 200 * 2.0**-23


def _grouped(pointcept, native, monkeypatch, *args):
    with monkeypatch.context() as m:
        if not native:
            m.setattr(pointcept, "_native_rows", lambda *t: False)
        return pointcept.grouping(*args)


@pytest.mark.parametrize("M,K,C,N", [(1, 1, 1, 1), (21, 3, 32, 50), (64, 1, 5, 64), (65, 16, 100, 300),
                                     (7, 9, 33, 20), (3, 2, 9000, 5)])
@pytest.mark.parametrize("with_xyz", [False, True])
@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_grouping_matches_tensor_operations(cuda_device, monkeypatch, M, K, C, N, with_xyz, own, dtype):
    from mps_pointops import pointcept

    g = torch.Generator().manual_seed(M * K + C)
    if own:
        M = N
    idx = torch.randint(-1, N, (M, K), generator=g).to(dtype).cuda()
    feat = torch.randn(N, C, generator=g).cuda().requires_grad_()
    xyz = torch.randn(N, 3, generator=g).cuda().requires_grad_()
    new = None if own else torch.randn(M, 3, generator=g).cuda().requires_grad_()
    inputs = [feat] + ([xyz] + ([] if own else [new]) if with_xyz else [])
    results = []
    for native in (True, False):
        out = _grouped(pointcept, native, monkeypatch, idx, feat, xyz, new, with_xyz)
        weight = torch.linspace(-1, 1, out.numel(), device="cuda").view_as(out).requires_grad_()
        first = torch.autograd.grad((out * weight).sum(), inputs, create_graph=True)
        second = torch.autograd.grad(sum((t * t).sum() for t in first), weight)
        results.append((out.detach(), first, second))
    (out, first, second), (want, want_first, want_second) = results
    assert torch.equal(out, want)
    for a, b in zip(first, want_first):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=TOL * 1e-2)
    torch.testing.assert_close(second[0], want_second[0], rtol=1e-4, atol=TOL)


def test_forward_mode_and_vmap_take_the_tensor_operations(cuda_device):
    from mps_pointops import pointcept

    idx = torch.tensor([[0, -1], [1, 1]], device="cuda")
    xyz = torch.randn(3, 3, device="cuda")
    feat, tangent = torch.randn(3, 4, device="cuda"), torch.randn(3, 4, device="cuda")
    new = torch.randn(2, 3, device="cuda")
    _, jvp = torch.func.jvp(lambda f: pointcept.grouping(idx, f, xyz, new, True), (feat,), (tangent,))
    assert torch.equal(jvp[..., 3:], pointcept.grouping(idx, tangent, xyz))
    many = torch.randn(5, 2, 2, 7, device="cuda")
    f = feat.clone().requires_grad_()
    out = pointcept.grouping(idx, f, xyz, new, True)
    each = torch.stack([torch.autograd.grad(out, f, g, retain_graph=True)[0] for g in many])
    batched = torch.autograd.grad(out, f, many, is_grads_batched=True)[0]
    torch.testing.assert_close(batched, each, rtol=1e-5, atol=1e-5)  # sums of at most 4 terms


def test_batched_second_gradients_match_one_at_a_time(cuda_device):
    from mps_pointops import pointcept

    idx = torch.tensor([[0, -1], [1, 1], [2, 0]], device="cuda")
    inputs = [torch.randn(3, c, device="cuda").requires_grad_() for c in (4, 3)]
    out = pointcept.grouping(idx, *inputs, None, True)
    weight = torch.randn_like(out).requires_grad_()
    first = torch.autograd.grad((out * weight).sum(), inputs, create_graph=True)
    many = [torch.randn(5, *t.shape, device="cuda") for t in first]
    batched = torch.autograd.grad(first, weight, many, retain_graph=True, is_grads_batched=True)[0]
    for i in range(5):
        one = torch.autograd.grad(first, weight, [m[i] for m in many], retain_graph=True)[0]
        torch.testing.assert_close(batched[i], one, rtol=1e-6, atol=1e-6)


def test_a_trace_and_a_subclass_keep_the_tensor_operations(cuda_device):
    from mps_pointops import pointcept

    class Marked(torch.Tensor):
        pass

    idx = torch.tensor([[0, -1], [1, 1], [2, 0]], device="cuda")
    feat, other = torch.randn(3, 4, device="cuda"), torch.randn(3, 4, device="cuda")
    xyz = torch.randn(3, 3, device="cuda")
    traced = torch.jit.trace(lambda f, x: pointcept.grouping(idx, f, x, None, True), (feat, xyz))
    assert torch.equal(traced(other, xyz), pointcept.grouping(idx, other, xyz, None, True))
    assert isinstance(pointcept.grouping(idx, feat.as_subclass(Marked), xyz), Marked)


@pytest.mark.parametrize("with_xyz", [False, True])
@pytest.mark.parametrize("own_idx", [False, True])
def test_indices_may_be_written_to_after_the_call(cuda_device, with_xyz, own_idx):
    """The gradient belongs to the indices of the call, whether the caller
    passed them or got them back."""
    from mps_pointops import pointcept

    g = torch.Generator().manual_seed(5)
    xyz = torch.randn(40, 3, generator=g).cuda()
    offset = torch.tensor([3, 40], dtype=torch.int32, device="cuda")  # 3 < K: -1 among them
    idx, _ = pointcept.knn_query(5, xyz, offset)
    weight = torch.randn(40, 5, 9 if with_xyz else 6, generator=g).cuda()
    grads = []
    for write in (False, True):
        feat = torch.ones(40, 6, device="cuda").requires_grad_()
        out, at = pointcept.knn_query_and_group(feat, xyz, offset, nsample=5, with_xyz=with_xyz,
                                                idx=idx.clone() if own_idx else None)
        assert torch.equal(at, idx)
        if write:
            at[at < 0] = 0
        grads.append(torch.autograd.grad(out, feat, weight)[0])
    torch.testing.assert_close(grads[1], grads[0], rtol=1e-5, atol=1e-5)  # sums of at most 40 terms


@pytest.mark.parametrize("with_xyz", [False, True])
def test_deterministic_algorithms_repeat_the_gradient(cuda_device, with_xyz):
    """Bit for bit, with thousands of terms on each of a few rows."""
    from mps_pointops import pointcept

    g = torch.Generator().manual_seed(6)
    idx = torch.randint(-1, 4, (2000, 32), generator=g).cuda()
    feat, xyz = torch.randn(4, 16, generator=g).cuda(), torch.randn(4, 3, generator=g).cuda()
    new = torch.randn(2000, 3, generator=g).cuda().requires_grad_() if with_xyz else None
    inputs = [feat.requires_grad_()] + ([xyz.requires_grad_(), new] if with_xyz else [])
    weight = torch.randn(2000, 32, 19 if with_xyz else 16, generator=g).cuda()
    out = pointcept.grouping(idx, feat, xyz, new, with_xyz)
    torch.use_deterministic_algorithms(True)
    try:
        first, *others = (torch.autograd.grad(out, inputs, weight, retain_graph=True) for _ in range(8))
    finally:
        torch.use_deterministic_algorithms(False)
    for other in others:
        for a, b in zip(first, other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("M,K", [(1, 1), (85, 3), (256, 16)])
def test_knn_finish_matches_tensor_operations(cuda_device, M, K):
    from mps_pointops import _native

    g = torch.Generator().manual_seed(M)
    x, y = torch.randn(40, 3, generator=g).cuda(), torch.randn(M, 3, generator=g).cuda()
    x[::7] *= 1e6  # beyond the ceiling
    x[3] = float("nan")
    idx = torch.randint(-1, 40, (M, K), generator=g).cuda()
    out = torch.empty(M, K, dtype=torch.int32, device="cuda")
    dist = torch.empty(M, K, device="cuda")
    _native.call("pointops_knn_finish", y.data_ptr(), x.data_ptr(), idx.data_ptr(), out.data_ptr(),
                 dist.data_ptr(), M, K, 1e10, 1e5, _native.stream(x.device))
    d = y[:, None] - x[idx.clamp_min(0)]
    sq = d[..., 0] * d[..., 0]
    sq = sq + d[..., 1] * d[..., 1]
    sq = sq + d[..., 2] * d[..., 2]
    valid = (idx >= 0) & (sq < 1e10)
    assert torch.equal(out, torch.where(valid, idx, -1).int())
    assert torch.equal(dist, torch.where(valid, sq.sqrt(), 1e5))
