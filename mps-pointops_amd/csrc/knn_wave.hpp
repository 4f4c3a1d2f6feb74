// One wave per kNN query: the sorted list spread over the wave and the scan of
// the references that fills it (described in knn.hip), shared by the
// wave-per-query kernels and by the queries the screened search leaves over.
#pragma once

#include "pointops_common.hpp"

namespace pointops {
namespace {

// Sequential squared L2 in D dimensions: s = d0^2; s = s + dt^2 (dt = r - q).
__device__ __forceinline__ float sqdist_nd(const float* __restrict__ r, const float* __restrict__ q,
                                           int D) {
    const float first = r[0] - q[0];
    float s = first * first;
    for (int t = 1; t < D; ++t) {
        const float delta = r[t] - q[t];
        const float term = delta * delta;
        s = s + term;
    }
    return s;
}

// The same chain with rows read 16 bytes at a time (D % 4 == 0 and both rows
// 16-byte aligned): a lane's row is then D / 4 requests.
__device__ __forceinline__ float sqdist_rows(const float* __restrict__ r, const float* __restrict__ q,
                                             int D) {
    float s = 0.f;  // 0 + d0^2 = d0^2
#pragma unroll 8
    for (int t = 0; t < D; t += 4) {
        const float4 x = *reinterpret_cast<const float4*>(r + t);
        const float4 y = *reinterpret_cast<const float4*>(q + t);
        const float d0 = x.x - y.x, d1 = x.y - y.y, d2 = x.z - y.z, d3 = x.w - y.w;
        s = s + d0 * d0;
        s = s + d1 * d1;
        s = s + d2 * d2;
        s = s + d3 * d3;
    }
    return s;
}

__device__ __forceinline__ int64_t segment_of(const int64_t* __restrict__ ptr, int64_t batch,
                                              int64_t q) {
    int64_t lo = 0, hi = batch;
    while (lo < hi) {
        const int64_t mid = lo + (hi - lo) / 2;
        if (ptr[mid + 1] <= q) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ uint32_t gcd_u32(uint32_t a, uint32_t b) {
    while (b != 0) {
        const uint32_t t = a % b;
        a = b;
        b = t;
    }
    return a;
}

// Chunk stride ~ golden ratio * chunks, bumped until coprime to chunks.
__device__ __forceinline__ uint32_t visit_stride(uint32_t chunks) {
    if (chunks <= 2) return 1;
    uint32_t s = static_cast<uint32_t>(static_cast<double>(chunks) * 0.6180339887498949 + 0.5) % chunks;
    if (s == 0) s = 1;
    while (gcd_u32(s, chunks) != 1) {
        s = (s + 1) % chunks;
        if (s == 0) s = 1;
    }
    return s;
}

// Insert candidate (cd, ci) into the wave-distributed sorted list.
template <int SLOTS>
__device__ __forceinline__ void list_insert(float (&ld)[SLOTS], int (&li)[SLOTS], int K, int lane,
                                            float cd, int ci) {
    int pos = 0;
#pragma unroll
    for (int r = 0; r < SLOTS; ++r) {
        const int s = r * kWave + lane;
        pos += __popcll(ballot(s < K && before(ld[r], li[r], cd, ci)));
    }
    int carry_d = 0, carry_i = 0;
#pragma unroll
    for (int r = 0; r < SLOTS; ++r) {
        const int s = r * kWave + lane;
        // Lane 63 of the previous register moves to lane 0 of this one.
        const int next_carry_d = readlane(f2i(ld[r]), kWave - 1);
        const int next_carry_i = readlane(li[r], kWave - 1);
        const float shifted_d = i2f(wave_shr1(f2i(ld[r]), carry_d));
        const int shifted_i = wave_shr1(li[r], carry_i);
        if (s > pos) {
            ld[r] = shifted_d;
            li[r] = shifted_i;
        } else if (s == pos) {
            ld[r] = cd;
            li[r] = ci;
        }
        carry_d = next_carry_d;
        carry_i = next_carry_i;
    }
}

template <int SLOTS>
__device__ __forceinline__ void list_tail(const float (&ld)[SLOTS], const int (&li)[SLOTS], int K,
                                          float& td, int& ti) {
    const int r_last = (K - 1) / kWave;
    const int l_last = (K - 1) % kWave;
    int d = 0, i = 0;
#pragma unroll
    for (int r = 0; r < SLOTS; ++r) {
        if (r == r_last) {
            d = readlane(f2i(ld[r]), l_last);
            i = readlane(li[r], l_last);
        }
    }
    td = i2f(d);
    ti = i;
}

// One wave: scan n references and keep the K best keys (VEC: rows as
// sqdist_rows reads them).
template <int SLOTS, bool DIM3, bool FINITE_ONLY, bool VEC>
__device__ __forceinline__ void scan_refs_by(const float* __restrict__ qp, const float* __restrict__ rp,
                                          int n, int D, int K, int lane, float (&ld)[SLOTS],
                                          int (&li)[SLOTS]) {
    float td = INFINITY;
    int ti = -1;  // 0xFFFFFFFF: every real index is before it
    const uint32_t chunks = (static_cast<uint32_t>(n) + kWave - 1) / kWave;
    if (chunks == 0) return;
    float qx = 0.f, qy = 0.f, qz = 0.f;
    if (DIM3) {
        qx = qp[0];
        qy = qp[1];
        qz = qp[2];
    }
    const uint32_t stride = visit_stride(chunks);
    uint32_t chunk = 0;
    for (uint32_t c = 0; c < chunks; ++c) {
        const int j = static_cast<int>(chunk * kWave) + lane;
        chunk += stride;
        if (chunk >= chunks) chunk -= chunks;
        float d = INFINITY;
        bool valid = j < n;
        if (valid) {
            if (DIM3) {
                const float* r = rp + 3 * static_cast<int64_t>(j);
                d = sqdist3(r[0], r[1], r[2], qx, qy, qz);
            } else {
                const float* r = rp + static_cast<int64_t>(j) * D;
                d = VEC ? sqdist_rows(r, qp, D) : sqdist_nd(r, qp, D);
            }
            if (FINITE_ONLY) valid = isfinite(d);
        }
        uint64_t pending = ballot(valid && before(d, j, td, ti));
        while (pending != 0) {
            const int src = __builtin_ctzll(pending);
            pending &= pending - 1;
            const float cd = i2f(readlane(f2i(d), src));
            const int ci = readlane(j, src);
            if (!before(cd, ci, td, ti)) continue;  // an earlier insert raised the bar
            list_insert<SLOTS>(ld, li, K, lane, cd, ci);
            list_tail<SLOTS>(ld, li, K, td, ti);
        }
    }
}

template <int SLOTS, bool DIM3, bool FINITE_ONLY>
__device__ __forceinline__ void scan_refs(const float* __restrict__ qp, const float* __restrict__ rp,
                                          int n, int D, int K, int lane, float (&ld)[SLOTS],
                                          int (&li)[SLOTS]) {
    if (!DIM3 && D % 4 == 0 && (reinterpret_cast<uintptr_t>(rp) | reinterpret_cast<uintptr_t>(qp)) % 16 == 0)
        scan_refs_by<SLOTS, DIM3, FINITE_ONLY, true>(qp, rp, n, D, K, lane, ld, li);
    else
        scan_refs_by<SLOTS, DIM3, FINITE_ONLY, false>(qp, rp, n, D, K, lane, ld, li);
}

}  // namespace
}  // namespace pointops
