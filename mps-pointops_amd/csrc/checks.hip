// Argument checks and list bookkeeping on the device for gfx950: what the
// Python layer has to know before or after a search, each in one launch in
// place of four to eight tensor operations.  All are bound by launch latency
// (a few microseconds); flags and results are read back by the caller, several
// checks with one synchronisation.
#include "pointops_common.hpp"
#include "pointops_hip.h"

namespace pointops {
namespace {

constexpr int kCheckThreads = 256;
constexpr int64_t kCheckMaxBlocks = 1024;  // grid-stride beyond 256 K values

dim3 check_grid(int64_t n) {
    const int64_t blocks = (n + kCheckThreads - 1) / kCheckThreads;
    return dim3(static_cast<uint32_t>(blocks < kCheckMaxBlocks ? blocks : kCheckMaxBlocks));
}

// A wave's verdict, stored by one lane (every writer stores 1: no atomic).
__device__ __forceinline__ void raise(bool bad, int32_t* flag) {
    if (ballot(bad) != 0 && lane_id() == 0) __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename I>
__global__ __launch_bounds__(kCheckThreads) void check_range_kernel(const I* __restrict__ v, int64_t n,
                                                                    int64_t lo, int64_t hi,
                                                                    int32_t* __restrict__ flag) {
    bool bad = false;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kCheckThreads + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCheckThreads)
        bad |= v[i] < lo || v[i] > hi;
    raise(bad, flag);
}

template <typename T>
__global__ __launch_bounds__(kCheckThreads) void check_finite_kernel(const T* __restrict__ p,
                                                                     const int64_t* __restrict__ lengths,
                                                                     int64_t n, int64_t row, int64_t D,
                                                                     int32_t* __restrict__ flag) {
    bool bad = false;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kCheckThreads + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCheckThreads) {
        if (isfinite(p[i])) continue;
        const int64_t b = i / row;
        bad |= lengths == nullptr || (i - b * row) / D < lengths[b];
    }
    raise(bad, flag);
}

// out[0] = the first id, out[1] = 1 if any is below its predecessor (0 on
// entry), out[2] = the last id.
template <typename I>
__global__ __launch_bounds__(kCheckThreads) void segment_check_kernel(const I* __restrict__ ids, int64_t n,
                                                                      int64_t* __restrict__ out) {
    bool bad = false;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kCheckThreads + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCheckThreads) {
        if (i == 0) out[0] = ids[0];
        else bad |= ids[i] < ids[i - 1];
        if (i == n - 1) out[2] = ids[i];
    }
    if (ballot(bad) != 0 && lane_id() == 0)
        __hip_atomic_store(out + 1, int64_t(1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// offsets[c] = first row whose id is at least c, for sorted ids: a binary
// search per cloud, whatever gaps the ids have.
template <typename I>
__global__ __launch_bounds__(kCheckThreads) void segment_offsets_kernel(const I* __restrict__ ids, int64_t n,
                                                                        int64_t clouds,
                                                                        int64_t* __restrict__ offsets) {
    for (int64_t c = static_cast<int64_t>(blockIdx.x) * kCheckThreads + threadIdx.x; c <= clouds;
         c += static_cast<int64_t>(gridDim.x) * kCheckThreads) {
        int64_t lo = 0, hi = n;
        while (lo < hi) {
            const int64_t mid = lo + (hi - lo) / 2;
            if (ids[mid] < c) lo = mid + 1;
            else hi = mid;
        }
        offsets[c] = lo;
    }
}

__device__ __forceinline__ bool is_edge(int64_t j, int64_t q, bool skip_self) {
    return j >= 0 && !(skip_self && j == q);
}

// One wave per query row of the (Q, K) table.
__global__ __launch_bounds__(kCheckThreads) void edge_count_kernel(const int64_t* __restrict__ table, int64_t Q,
                                                                   int64_t K, bool skip_self,
                                                                   int64_t* __restrict__ counts) {
    const int64_t q = static_cast<int64_t>(blockIdx.x) * (kCheckThreads / kWave) + uniform(threadIdx.x / kWave);
    if (q >= Q) return;
    const int lane = lane_id();
    int64_t count = 0;
    for (int64_t k0 = 0; k0 < K; k0 += kWave)
        count += __popcll(ballot(k0 + lane < K && is_edge(table[q * K + k0 + lane], q, skip_self)));
    if (lane == 0) counts[q] = count;
}

// edges[a E + e] the query and edges[(1 - a) E + e] the reference of edge e,
// row-major over the table; ends[q] is the number of edges of rows 0 .. q.
__global__ __launch_bounds__(kCheckThreads) void edge_write_kernel(const int64_t* __restrict__ table,
                                                                   const int64_t* __restrict__ ends, int64_t Q,
                                                                   int64_t K, bool skip_self, int64_t* __restrict__ first,
                                                                   int64_t* __restrict__ second) {
    const int64_t q = static_cast<int64_t>(blockIdx.x) * (kCheckThreads / kWave) + uniform(threadIdx.x / kWave);
    if (q >= Q) return;
    const int lane = lane_id();
    int64_t at = q == 0 ? 0 : ends[q - 1];
    for (int64_t k0 = 0; k0 < K; k0 += kWave) {
        const int64_t j = k0 + lane < K ? table[q * K + k0 + lane] : -1;
        const uint64_t edges = ballot(is_edge(j, q, skip_self));
        if ((edges >> lane) & 1u) {
            const int64_t e = at + lanes_below(edges);
            first[e] = q;
            second[e] = j;
        }
        at += __popcll(edges);
    }
}

}  // namespace
}  // namespace pointops

using namespace pointops;

extern "C" {

hipError_t pointops_check_range(const void* values, int32_t bits, int64_t n, int64_t lo, int64_t hi,
                                int32_t* flag, hipStream_t stream) {
    if (n < 0 || (bits != 32 && bits != 64) || flag == nullptr) return hipErrorInvalidValue;
    if (n == 0) return hipSuccess;
    if (bits == 32)
        hipLaunchKernelGGL((check_range_kernel<int32_t>), check_grid(n), dim3(kCheckThreads), 0, stream,
                           static_cast<const int32_t*>(values), n, lo, hi, flag);
    else
        hipLaunchKernelGGL((check_range_kernel<int64_t>), check_grid(n), dim3(kCheckThreads), 0, stream,
                           static_cast<const int64_t*>(values), n, lo, hi, flag);
    return hipGetLastError();
}

hipError_t pointops_check_finite(const void* points, int32_t bits, const int64_t* lengths, int64_t B,
                                 int64_t P, int64_t D, int32_t* flag, hipStream_t stream) {
    if (B < 0 || P < 0 || D < 1 || (bits != 32 && bits != 64) || flag == nullptr) return hipErrorInvalidValue;
    const int64_t n = B * P * D;
    if (n == 0) return hipSuccess;
    if (bits == 32)
        hipLaunchKernelGGL((check_finite_kernel<float>), check_grid(n), dim3(kCheckThreads), 0, stream,
                           static_cast<const float*>(points), lengths, n, P * D, D, flag);
    else
        hipLaunchKernelGGL((check_finite_kernel<double>), check_grid(n), dim3(kCheckThreads), 0, stream,
                           static_cast<const double*>(points), lengths, n, P * D, D, flag);
    return hipGetLastError();
}

hipError_t pointops_segment_check(const void* ids, int32_t bits, int64_t n, int64_t* out, hipStream_t stream) {
    if (n < 1 || (bits != 32 && bits != 64) || out == nullptr) return hipErrorInvalidValue;
    if (bits == 32)
        hipLaunchKernelGGL((segment_check_kernel<int32_t>), check_grid(n), dim3(kCheckThreads), 0, stream,
                           static_cast<const int32_t*>(ids), n, out);
    else
        hipLaunchKernelGGL((segment_check_kernel<int64_t>), check_grid(n), dim3(kCheckThreads), 0, stream,
                           static_cast<const int64_t*>(ids), n, out);
    return hipGetLastError();
}

hipError_t pointops_segment_offsets(const void* ids, int32_t bits, int64_t n, int64_t clouds,
                                    int64_t* offsets, hipStream_t stream) {
    if (n < 0 || clouds < 0 || (bits != 32 && bits != 64) || offsets == nullptr) return hipErrorInvalidValue;
    if (bits == 32)
        hipLaunchKernelGGL((segment_offsets_kernel<int32_t>), check_grid(clouds + 1), dim3(kCheckThreads), 0, stream,
                           static_cast<const int32_t*>(ids), n, clouds, offsets);
    else
        hipLaunchKernelGGL((segment_offsets_kernel<int64_t>), check_grid(clouds + 1), dim3(kCheckThreads), 0, stream,
                           static_cast<const int64_t*>(ids), n, clouds, offsets);
    return hipGetLastError();
}

hipError_t pointops_edge_count(const int64_t* table, int64_t Q, int64_t K, int32_t skip_self,
                               int64_t* counts, hipStream_t stream) {
    constexpr int64_t kPer = kCheckThreads / kWave;
    if (Q < 0 || K < 0 || (Q + kPer - 1) / kPer > INT32_MAX) return hipErrorInvalidValue;
    if (Q == 0) return hipSuccess;
    hipLaunchKernelGGL(edge_count_kernel, dim3(static_cast<uint32_t>((Q + kPer - 1) / kPer)), dim3(kCheckThreads),
                       0, stream, table, Q, K, skip_self != 0, counts);
    return hipGetLastError();
}

hipError_t pointops_edge_write(const int64_t* table, const int64_t* ends, int64_t Q, int64_t K,
                               int32_t skip_self, int64_t* queries, int64_t* references,
                               hipStream_t stream) {
    constexpr int64_t kPer = kCheckThreads / kWave;
    if (Q < 0 || K < 0 || (Q + kPer - 1) / kPer > INT32_MAX) return hipErrorInvalidValue;
    if (Q == 0) return hipSuccess;
    hipLaunchKernelGGL(edge_write_kernel, dim3(static_cast<uint32_t>((Q + kPer - 1) / kPer)), dim3(kCheckThreads),
                       0, stream, table, ends, Q, K, skip_self != 0, queries, references);
    return hipGetLastError();
}

}  // extern "C"
