"""ctypes binding of libpointops_hip.so (the C ABI in include/pointops_hip.h).

This is the only way the package reaches the GPU: there is no CPU or PyTorch
fallback.  Loading fails loudly when the library is missing or was built for
another architecture; every call checks the returned hipError_t.

The reference compiles Metal shaders on first use and checks the SIMD width
(_ball_query_mps.py:34-63); the equivalent gate here is that the library is
present and the device is gfx950 (checked once per device).
"""

from __future__ import annotations

import ctypes
import functools
import os
from pathlib import Path

import torch

LIB_NAME = "libpointops_hip.so"
LIB_PATH = Path(__file__).resolve().with_name(LIB_NAME)

_vp = ctypes.c_void_p
_i64 = ctypes.c_int64
_i32 = ctypes.c_int32
_f32 = ctypes.c_float
_size = ctypes.c_size_t

# name -> argument types (pointers as void*), restype int (hipError_t)
_SIGNATURES: dict[str, list] = {
    "pointops_fps_dense": [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "pointops_fps_large": [_vp, _vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "pointops_fps_large_noalloc": [_vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "pointops_fps_flat": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_fps_flat_sorted": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_knn3": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_knn3_grid": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_knn3_windowed": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_knn_feat": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _vp],
    "pointops_knn_screen": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _vp],
    "pointops_nearest3_screen": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_knn_flat_screen": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i64, _vp],
    "pointops_knn_flat": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_ball_query_f32": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _f32, _vp],
    "pointops_ball_query_multi_f32": [_vp, _vp, _i64, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_ball_query_f16": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _f32, _vp],
    "pointops_radius_flat_f32": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _f32, _i32, _vp],
    "pointops_radius_flat_f16": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _f32, _i32, _vp],
    "pointops_ball_query_backward_f32": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64,
                                         _i64, _vp],
    "pointops_ball_query_backward_f16": [_vp, _vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64,
                                         _i64, _vp],
    "pointops_three_nn": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_three_interpolate": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_three_interpolate_backward": [_vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_three_interpolate_backward_csr": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64,
                                                _vp],
    "pointops_three_interpolate_csr_build": [_vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_three_interpolate_backward_from_csr": [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_ball_query_pn2_f32": [_vp, _vp, _vp, _i64, _i64, _i64, _i64, _f32, _vp],
    "pointops_ball_query_grid_f32": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _f32, _vp],
    "pointops_ball_query_auto_f32": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _f32, _vp],
    "pointops_nearest3_grid": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _vp],
    "pointops_group_points": [_vp, _vp, _i32, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_group_points_backward": [_vp, _i64, _vp, _i32, _vp, _vp, _i64, _i64, _i64, _i64, _vp],
    "pointops_group_points_rel": [_vp, _vp, _vp, _vp, _i32, _vp, _i64, _i64, _i64, _i64, _i64, _vp],
    "pointops_check_range": [_vp, _i32, _i64, _i64, _i64, _vp, _vp],
    "pointops_check_finite": [_vp, _i32, _vp, _i64, _i64, _i64, _vp, _vp],
    "pointops_segment_check": [_vp, _i32, _i64, _vp, _vp],
    "pointops_segment_offsets": [_vp, _i32, _i64, _i64, _vp, _vp],
    "pointops_edge_count": [_vp, _i64, _i64, _i32, _vp, _vp],
    "pointops_edge_write": [_vp, _vp, _i64, _i64, _i32, _vp, _vp, _vp],
    "pointops_knn_finish": [_vp, _vp, _vp, _vp, _vp, _i64, _i64, _f32, _f32, _vp],
    "pointops_group_rows": [_vp, _vp, _vp, _vp, _i32, _vp, _i64, _i64, _i64, _vp],
    "pointops_group_rows_backward": [_vp, _vp, _i32, _vp, _vp, _vp, _i64, _i64, _i64, _i32, _vp],
    "pointops_chamfer_nearest_f32": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "pointops_chamfer_nearest_f64": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "pointops_chamfer_backward_f32": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "pointops_chamfer_backward_f64": [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i64, _i64, _i64, _i32, _vp],
    "pointops_fps_query_pipeline_f32": [_vp, _vp, _vp, _i64, _vp, _vp, _vp, _vp, _i64, _vp, _vp,
                                        _vp, _vp, _i64, _i64, _i64, _i64, _i32, _i64, _vp, _vp],
}
_SIZE_QUERIES: dict[str, list] = {
    "pointops_fps_dense_scratch_bytes": [_i64, _i64],
    "pointops_fps_query_pipeline_workspace_bytes": [_i64, _i64, _i64, _i64],
    "pointops_fps_large_workspace_bytes": [_i64, _i64],
    "pointops_fps_flat_scratch_bytes": [_i64, _i64],
    "pointops_fps_flat_sorted_scratch_bytes": [_i64, _i64],
    "pointops_knn3_grid_workspace_bytes": [_i64, _i64, _i64],
    "pointops_knn3_windowed_workspace_bytes": [_i64, _i64, _i64],
    "pointops_knn_screen_workspace_bytes": [_i64, _i64, _i64],
    "pointops_knn_flat_screen_workspace_bytes": [_i64, _i64, _i64],
    "pointops_three_interpolate_backward_workspace_bytes": [_i64, _i64, _i64],
    "pointops_ball_query_grid_workspace_bytes": [_i64, _i64, _i64],
    "pointops_ball_query_backward_workspace_bytes": [_i64, _i64],
    "pointops_ball_query_auto_workspace_bytes": [_i64, _i64, _i64],
    "pointops_group_points_backward_workspace_bytes": [_i64, _i64, _i64, _i64],
}


@functools.lru_cache(maxsize=1)
def library() -> ctypes.CDLL:
    """Load the native library (once).  Raises if it has not been built."""
    path = Path(os.environ.get("POINTOPS_HIP_LIB", LIB_PATH))
    if not path.exists():
        raise RuntimeError(
            f"mps_pointops native library not found at {path}; build it with "
            "`python mps-pointops_amd/build.py` (hipcc, gfx950)"
        )
    lib = ctypes.CDLL(str(path))
    for name, args in _SIGNATURES.items():
        fn = getattr(lib, name)
        fn.argtypes = args
        fn.restype = ctypes.c_int
    for name, args in _SIZE_QUERIES.items():
        fn = getattr(lib, name)
        fn.argtypes = args
        fn.restype = _size
    lib.pointops_abi_version.restype = ctypes.c_int
    lib.pointops_device_supported.argtypes = [ctypes.c_int]
    lib.pointops_device_supported.restype = ctypes.c_int
    if lib.pointops_abi_version() != 1:
        raise RuntimeError(f"{path.name} has an unexpected ABI version")
    return lib


@functools.lru_cache(maxsize=None)
def _check_device(index: int) -> None:
    if not library().pointops_device_supported(index):
        name = torch.cuda.get_device_properties(index).gcnArchName
        raise RuntimeError(
            f"mps_pointops kernels are built for gfx950 (MI355X); cuda:{index} is {name}"
        )


@functools.lru_cache(maxsize=1)
def _hip_error_string():
    try:
        hip = ctypes.CDLL("libamdhip64.so")
        hip.hipGetErrorString.argtypes = [ctypes.c_int]
        hip.hipGetErrorString.restype = ctypes.c_char_p
        return hip.hipGetErrorString
    except OSError:
        return None


def require_device(device: torch.device) -> int:
    """Index of a usable ROCm device, after the one-time capability check."""
    if device.type != "cuda":
        raise ValueError(
            f"mps_pointops runs on ROCm GPU tensors (device='cuda'); got {device.type}"
        )
    index = device.index if device.index is not None else torch.cuda.current_device()
    _check_device(index)
    return index


def ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def stream(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream


def call(name: str, *args) -> None:
    """Enqueue an entry point that computes an operator's results; RuntimeError
    on a non-zero status.  (The argument checks below go to _enqueue directly,
    so that replacing ``call`` shows which kernels a result came from.)"""
    _enqueue(name, *args)


def _enqueue(name: str, *args) -> None:
    status = getattr(library(), name)(*args)
    if status != 0:
        getter = _hip_error_string()
        text = getter(status).decode() if getter is not None else f"hipError {status}"
        raise RuntimeError(f"{name} failed: {text}")


def size_query(name: str, *args) -> int:
    return int(getattr(library(), name)(*args))


def plain(*tensors: torch.Tensor) -> bool:
    """Whether kernels on raw pointers may stand in for tensor operations on
    these: no subclasses and no batched gradients (which may hold no memory of
    their own; a backward's thread does not see the transform), and outside
    function transforms, forward-mode differentiation, tracing, compilation and
    dispatch modes, all of which see tensor operations only."""
    return (all(type(t) in (torch.Tensor, torch.nn.Parameter) and torch._C._has_storage(t)
                for t in tensors)
            and torch._C._functorch.peek_interpreter_stack() is None
            and torch.autograd.forward_ad._current_level < 0
            and torch._C._len_torch_dispatch_stack() == 0
            and not torch.jit.is_tracing()
            and not torch.compiler.is_compiling())


def outside(checks: list[tuple[torch.Tensor, int, int]]) -> list[bool]:
    """For each (int32/int64 tensor, lo, hi), whether any value lies outside
    [lo, hi]; all on one ROCm device, read with one synchronisation."""
    device = checks[0][0].device
    if not plain(*(values for values, _, _ in checks)):
        return [bool(((v < lo) | (v > hi)).any().item()) for v, lo, hi in checks]
    flags = torch.zeros(len(checks), dtype=torch.int32, device=device)
    for i, (values, lo, hi) in enumerate(checks):
        values = values.contiguous()
        _enqueue("pointops_check_range", values.data_ptr(), 8 * values.element_size(), values.numel(),
                 lo, hi, flags.data_ptr() + 4 * i, stream(device))
    return [flag != 0 for flag in flags.tolist()]


def nonfinite(clouds: list[tuple[torch.Tensor, torch.Tensor | None]]) -> list[bool]:
    """For each (float32/float64 (B, P, D) points, lengths or None), whether a
    row below its cloud's length has a coordinate that is not finite; all on
    one ROCm device, read with one synchronisation."""
    device = clouds[0][0].device
    flags = torch.zeros(len(clouds), dtype=torch.int32, device=device)
    for i, (points, lengths) in enumerate(clouds):
        points = points.detach().contiguous()
        lengths = None if lengths is None else lengths.contiguous()
        _enqueue("pointops_check_finite", points.data_ptr(), 8 * points.element_size(), ptr(lengths),
                 *points.shape, flags.data_ptr() + 4 * i, stream(device))
    return [flag != 0 for flag in flags.tolist()]
