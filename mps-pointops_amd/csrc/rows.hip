// Row-major neighbourhood grouping for gfx950 (the point-transformer layers of
// pointcept.py): (N, C) rows gathered at (M, K) indices into (M, K, 3 + C),
// the neighbours' positions relative to their query first, its gradients, and
// the finish of the kNN that finds the indices.  -1 marks a missing neighbour:
// zeros forward, no gradient.
//
// All three are bound by memory traffic; as separate tensor operations
// (gather, where, subtract, where, concatenate, and a scatter per input
// backward) the rows crossed memory about ten times.  Each kernel here reads
// and writes them once.  At 60000 queries, K = 16, C = 32 (134 MB of rows):
// grouping 52 us, its backward 214 us (34 M float atomics, the bound), the
// finish 8.5 us, in place of about 1000 us of tensor operations; the whole
// layer with its kNN 1279 -> 624 us.
#include "pointops_common.hpp"
#include "pointops_hip.h"

namespace pointops {
namespace {

constexpr int kRowsThreads = 256;
constexpr int kRowsPerBlock = 64;

template <typename I>
__device__ __forceinline__ int64_t row_index(const I* __restrict__ idx, int64_t r) {
    return static_cast<int64_t>(idx[r]);
}

// A block's 64 output rows are one contiguous run of 64 W floats: consecutive
// threads write consecutive floats, each from its row's feature (consecutive
// reads within a row) or from the row's offsets in LDS.
template <typename I>
__global__ __launch_bounds__(kRowsThreads) void group_rows_kernel(
    const float* __restrict__ feat, const float* __restrict__ xyz, const float* __restrict__ centres,
    const I* __restrict__ idx, float* __restrict__ out, int64_t rows, int K, int C, int off,
    uint32_t magic) {
    __shared__ int64_t at[kRowsPerBlock];
    __shared__ float rel[kRowsPerBlock][3];
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock;
    const int count = static_cast<int>(min<int64_t>(kRowsPerBlock, rows - row0));
    const int tid = threadIdx.x;
    if (tid < count) {
        const int64_t j = row_index(idx, row0 + tid);
        at[tid] = j;
        if (off != 0) {
            const float* c = centres + 3 * ((row0 + tid) / K);
#pragma unroll
            for (int a = 0; a < 3; ++a) rel[tid][a] = j < 0 ? 0.f : xyz[3 * j + a] - c[a];
        }
    }
    __syncthreads();
    const uint32_t W = static_cast<uint32_t>(C + off);
    const uint32_t total = static_cast<uint32_t>(count) * W;
    float* o = out + row0 * W;
#pragma unroll 4
    for (uint32_t e = tid; e < total; e += kRowsThreads) {
        const uint32_t r = magic != 0 ? __umulhi(e, magic) : e / W;
        const uint32_t c = e - r * W;
        const int64_t j = at[r];
        float v;
        if (static_cast<int>(c) < off) v = rel[r][c];
        else v = j < 0 ? 0.f : feat[j * C + (c - off)];
        store_once(o + e, v);
    }
}

// One wave per query: its K W gradients are contiguous, each added to its
// neighbour's feature or position by a hardware float atomic, the order of
// whose additions is not fixed (where the caller has asked for deterministic
// algorithms it uses tensor operations instead); the query's own position
// takes the negated sum of its relative offsets' gradients.
template <typename I>
__global__ __launch_bounds__(kRowsThreads) void group_rows_grad_kernel(
    const float* __restrict__ g, const I* __restrict__ idx, float* __restrict__ gfeat,
    float* __restrict__ gxyz, float* __restrict__ gcentres, int64_t M, int K, int C, int off,
    uint32_t magic) {
    const int64_t m = static_cast<int64_t>(blockIdx.x) * (kRowsThreads / kWave) + uniform(threadIdx.x / kWave);
    const int lane = lane_id();
    if (m >= M) return;
    const uint32_t W = static_cast<uint32_t>(C + off);
    const uint32_t total = static_cast<uint32_t>(K) * W;
    const float* row = g + m * total;
    const I* at = idx + m * K;
    if (gfeat != nullptr || gxyz != nullptr) {
#pragma unroll 4
        for (uint32_t e = lane; e < total; e += kWave) {
            const uint32_t r = magic != 0 ? __umulhi(e, magic) : e / W;
            const int c = static_cast<int>(e - r * W) - off;
            const int64_t j = row_index(at, r);
            if (j < 0) continue;
            const float v = row[e];
            if (c < 0) {
                if (gxyz != nullptr) unsafeAtomicAdd(gxyz + 3 * j + (c + off), v);
            } else if (gfeat != nullptr) {
                unsafeAtomicAdd(gfeat + j * C + c, v);
            }
        }
    }
    if (gcentres != nullptr && lane < 3) {
        float s[4] = {0.f, 0.f, 0.f, 0.f};  // shorter sums round less
        for (int r0 = 0; r0 < K; r0 += 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = r0 + i;
                if (r < K && row_index(at, r) >= 0) s[i] = s[i] + row[static_cast<uint32_t>(r) * W + lane];
            }
        }
        gcentres[3 * m + lane] = -((s[0] + s[1]) + (s[2] + s[3]));
    }
}

// kNN's (M, K) rows: the Euclidean distance recomputed from the coordinates in
// the searches' order of operations, and int32 indices; a neighbour at or
// beyond `ceiling` (squared) is missing: index -1, distance `pad`.
__global__ __launch_bounds__(kRowsThreads) void knn_finish_kernel(
    const float* __restrict__ y, const float* __restrict__ x, const int64_t* __restrict__ idx,
    int32_t* __restrict__ out, float* __restrict__ dist, int64_t rows, int K, float ceiling, float pad) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kRowsThreads + threadIdx.x;
    if (i >= rows) return;
    const int64_t j = idx[i];
    float d = INFINITY;
    if (j >= 0) {
        const float* q = y + 3 * (i / K);
        const float* r = x + 3 * j;
        d = sqdist3(q[0], q[1], q[2], r[0], r[1], r[2]);
    }
    const bool valid = d < ceiling;
    out[i] = valid ? static_cast<int32_t>(j) : -1;
    dist[i] = valid ? sqrtf(d) : pad;
}

// floor(e / W) = umulhi(e, magic) for e < limit where limit W < 2^32; 0 (divide)
// otherwise.
uint32_t division_magic(int64_t W, int64_t limit) {
    if (W < 2 || limit * W >= (int64_t(1) << 32)) return 0;
    return static_cast<uint32_t>(((uint64_t(1) << 32) + W - 1) / W);
}

}  // namespace
}  // namespace pointops

using namespace pointops;

extern "C" {

hipError_t pointops_group_rows(const float* feat, const float* xyz, const float* centres,
                               const void* idx, int32_t idx_bits, float* out, int64_t M, int64_t K,
                               int64_t C, hipStream_t stream) {
    const int64_t off = xyz != nullptr ? 3 : 0;
    if (M < 0 || K < 0 || C < 0 || (idx_bits != 32 && idx_bits != 64)) return hipErrorInvalidValue;
    const int64_t rows = M * K, W = C + off;
    if (rows == 0 || W == 0) return hipSuccess;
    const int64_t blocks = (rows + kRowsPerBlock - 1) / kRowsPerBlock;
    if ((C > 0 && feat == nullptr) || (off != 0 && centres == nullptr) || K > INT32_MAX ||
        W > INT32_MAX / kRowsPerBlock || blocks > INT32_MAX)
        return hipErrorInvalidValue;
    const uint32_t magic = division_magic(W, kRowsPerBlock * W);
    const dim3 grid(static_cast<uint32_t>(blocks));
    if (idx_bits == 32)
        hipLaunchKernelGGL((group_rows_kernel<int32_t>), grid, dim3(kRowsThreads), 0, stream, feat, xyz, centres,
                           static_cast<const int32_t*>(idx), out, rows, static_cast<int>(K),
                           static_cast<int>(C), static_cast<int>(off), magic);
    else
        hipLaunchKernelGGL((group_rows_kernel<int64_t>), grid, dim3(kRowsThreads), 0, stream, feat, xyz, centres,
                           static_cast<const int64_t*>(idx), out, rows, static_cast<int>(K),
                           static_cast<int>(C), static_cast<int>(off), magic);
    return hipGetLastError();
}

hipError_t pointops_group_rows_backward(const float* g, const void* idx, int32_t idx_bits,
                                        float* grad_feat, float* grad_xyz, float* grad_centres,
                                        int64_t M, int64_t K, int64_t C, int32_t with_xyz,
                                        hipStream_t stream) {
    const int64_t off = with_xyz ? 3 : 0;
    if (M < 0 || K < 0 || C < 0 || (idx_bits != 32 && idx_bits != 64) ||
        (off == 0 && (grad_xyz != nullptr || grad_centres != nullptr)))
        return hipErrorInvalidValue;
    const int64_t W = C + off;
    if (M == 0) return hipSuccess;
    constexpr int64_t kPer = kRowsThreads / kWave;
    const int64_t blocks = (M + kPer - 1) / kPer;
    if (K > INT32_MAX || K * W > INT32_MAX || blocks > INT32_MAX) return hipErrorInvalidValue;
    const uint32_t magic = division_magic(W, K * W);
    const dim3 grid(static_cast<uint32_t>(blocks));
    if (idx_bits == 32)
        hipLaunchKernelGGL((group_rows_grad_kernel<int32_t>), grid, dim3(kRowsThreads), 0, stream, g,
                           static_cast<const int32_t*>(idx), grad_feat, grad_xyz, grad_centres, M,
                           static_cast<int>(K), static_cast<int>(C), static_cast<int>(off), magic);
    else
        hipLaunchKernelGGL((group_rows_grad_kernel<int64_t>), grid, dim3(kRowsThreads), 0, stream, g,
                           static_cast<const int64_t*>(idx), grad_feat, grad_xyz, grad_centres, M,
                           static_cast<int>(K), static_cast<int>(C), static_cast<int>(off), magic);
    return hipGetLastError();
}

hipError_t pointops_knn_finish(const float* y, const float* x, const int64_t* idx, int32_t* out,
                               float* dist, int64_t M, int64_t K, float ceiling, float pad,
                               hipStream_t stream) {
    if (M < 0 || K < 0) return hipErrorInvalidValue;
    const int64_t rows = M * K, blocks = (rows + kRowsThreads - 1) / kRowsThreads;
    if (rows == 0) return hipSuccess;
    if (K > INT32_MAX || blocks > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(knn_finish_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kRowsThreads), 0,
                       stream, y, x, idx, out, dist, rows, static_cast<int>(K), ceiling, pad);
    return hipGetLastError();
}

}  // extern "C"
