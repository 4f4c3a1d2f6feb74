// Exact kNN for gfx950, screened on the matrix cores.
//
// The searches define every rounding of a distance (knn.hip), which a matrix
// product cannot reproduce, but it can tell which references cannot be among
// the K nearest.  Each block serves 64 queries of one cloud; its eight waves
// split the cloud's tiles of 32 references and twice compute, for all pairs,
//
//     s = |r|^2 - 2 q.r     (the squared distance less |q|^2)
//
// on the matrix cores.  For D = 3 the operands are split into two bf16 parts
// and all the products and a three-part norm are the 16 slots of one
// v_mfma_f32_32x32x16_bf16; other widths take the coordinates, relative to a
// centre and scaled, in f16.  With d the exact kernels' rounded squared
// distance, |s + |q|^2 - d| <= 2 E |q|^2 + 2 E |r|^2 (see screen_error).  Each
// reference carries its own part of that, so that one far from the others
// loosens nothing but its own bound: s +- 2 E |r|^2 is the norm taken 1 +- 2 E
// times, which is a slot of the product for D = 3.
//
// Pass 1 keeps, per query, the minima of s + 2 E |r|^2 over 128 groups of
// references: one v_min3 for two pairs.  K groups hold K distinct references,
// so the K-th smallest minimum T bounds the K-th smallest d by T + |q|^2 + 2 E
// |q|^2, and every neighbour has s - 2 E |r|^2 <= T + 4 E |q|^2.  Pass 2 repeats
// the products and lists the references at or below that (about K + K^2 / 256
// of them, plus those within the error).  The listed references' distances are then computed as the searches
// define them, and ranked by (distance, index): the results are the other
// kernels' bit for bit.  Consecutive references fall into different groups,
// so an order that puts neighbours next to each other does not spoil T.
//
// References that are not finite or too far for the operands' ranges are left
// out: they lie beyond every reach that a served query may have.  (One such
// reference, or one point at 20 beside 32 unit cubes of 4096, left nearly every
// query of its cloud over when the bound took the cloud's largest norm: 390 to
// 430 us at config 2's shape, now 41 to 57.)
//
// A query with more than kScreenCap references listed (copies of one point,
// clusters tighter than E) or that the screen cannot serve (not finite or beyond
// 2^48 itself) is left over: pass 2's hits once more, as bits, ranked by exact
// distance 64 at a time in index order, inside the same launch.  One wave each
// over every reference, eight queries in turn, took five times as long: half of
// both clouds copies of one point 478 -> 80 us at config 2's shape, D = 64 features
// in 16 clusters of 0.05 1019 -> 205 us (the scans that came before the screen: 77 and 355
// us); half of them zeros, which tie as everyone's nearest, 1245 -> 394 (297).
//
// What bounds it: not the products (134 M pairs at config 2 are 5500 cycles a
// block) but the phases around them, in cycles of a block at 32 x 1024 queries
// x 4096 references, k = 16: prologue 4200, pass 1 5300, limits 7000, pass 2
// 21000 (the hits' masks and appends), exact distances and ranks 10500; at 8 x
// 2048 x 2048, D = 64, k = 20: 11200, 14000, 14000, 16500, 33000 (each listed
// row is 256 bytes from L2).  Measured: config 2 98 -> 43 us, 16 x 512 x 1024
// 41 -> 18 us, D = 64 359 -> 53 us, D = 128 590 -> 75 us (one lane per query,
// every pair's distance as defined), 3 ragged clouds of 20000, k = 16 1000 ->
// 190 us (one wave per query); k = 1, squared distances (the Chamfer loss's), both
// directions of 32 x 8192 x 8192 735 -> 450 us (cell grid).  Eight waves a block, since four left every
// phase waiting on its own latency (65 against 43 us at config 2); bfloat16 in
// three products instead of f16 in one took 61 us for D = 64.
#include <type_traits>

#include "knn_wave.hpp"
#include "pointops_common.hpp"
#include "pointops_hip.h"

namespace pointops {
namespace {

constexpr int kScreenThreads = 512;
constexpr int kScreenWaves = kScreenThreads / kWave;
constexpr int kPrepThreads = 256;
constexpr int kScreenQueries = 64;  // per block
constexpr int kTileRefs = 32;       // references per tile: the rows of one product
constexpr int kScreenGroups = 128;  // minima per query
constexpr int kScreenCap = 128;     // listed references per query
constexpr int kScreenMaxK = 64;
constexpr int kGroupStride = 72;    // floats between groups: 8 groups x 8 queries hit 64 banks
constexpr float kScreenMaxSq = 1.2676506e30f;      // 2^100: squares of sums stay finite
constexpr float kScreenMaxQuerySq = 7.9228163e28f;  // 2^96, and
constexpr float kScreenMaxReach = 3.1691265e29f;    // 2^98: see kernel
constexpr float kScreenMaxRow = 65000.f;            // scaled: f16, and
constexpr float kScreenMaxQuery = 32000.f;          // twice that for -2 q
constexpr float kScreenMaxReachF16 = 1e9f;          // below (65000 - 32000)^2

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct ScreenLayout {
    uint4* frag;    // per tile and k-step: 64 lanes x 8 bf16 or f16
    float* norm;    // D != 3: |r|^2 per tile row (+inf behind the last reference)
    float* far_sq;  // per tile: largest |r|^2, with the sign set where a row is left out
};

// Tiles are numbered by segment: segment b's begin at lo / 32 + b, where lo is
// its first row, which leaves room for a partial tile per segment.
__host__ __device__ inline int64_t screen_tiles(int64_t rows, int64_t batch) {
    return rows / kTileRefs + batch;
}

// k-steps of 16 dimensions.
__host__ __device__ inline int screen_steps(int64_t D) { return D == 3 ? 1 : static_cast<int>((D + 15) / 16); }

size_t screen_layout(int64_t rows, int64_t batch, int64_t D, ScreenLayout* L, char* base) {
    const int64_t tiles = screen_tiles(rows, batch);
    const size_t frag = static_cast<size_t>(tiles) * screen_steps(D) * kWave * sizeof(uint4);
    const size_t norm = D == 3 ? 0 : static_cast<size_t>(tiles) * kTileRefs * sizeof(float);
    if (L != nullptr) {
        L->frag = reinterpret_cast<uint4*>(base);
        L->norm = reinterpret_cast<float*>(base + frag);
        L->far_sq = reinterpret_cast<float*>(base + frag + norm);
    }
    return frag + norm + static_cast<size_t>(tiles) * sizeof(float);
}

// The relative error E of the screen: |s + |q|^2 - d| <= E (|q| + |r|)^2, which
// is at least |q - r|^2 and four times |q| |r|, and at most 2 |q|^2 + 2 |r|^2.
// D = 3: a two-part operand is within 2^-16 of the float (relative), so the
// doubled products of a pair are within 4 x 2^-16 |q| |r|, a quarter of which
// counts: 2^-16; 16 terms summed in float32, 2^-23 each (allowing for
// truncation), the norms and the exact kernels' own rounding add 2^-18.
// Others: an f16 operand is within 2^-11, so the doubled products are within
// 4 x 2^-11 |q| |r|: 2^-11; D terms at 2^-23 and 2 (D + 6) 2^-24 for the norms
// and the exact chain.  (Coordinates below f16's normal range lose at most
// 2^-25 of the scaled unit each, at most `lost` (|q| + |r|) in all; for a row,
// lost |r| <= 1e-5 |r|^2 + lost^2 / 4e-5, whose first part is counted here.)
__host__ __device__ inline float screen_error(int D) {
    return D == 3 ? 2.3e-5f : 4.8828125e-4f * 1.02f + static_cast<float>(D + 6) * 3.6e-7f + 5e-6f;
}
// bf16 bits of 2 E for D = 3, 0.5 % up (of which rounding |r|^2 takes 0.2 %).
constexpr uint32_t kScreenError3 = 0x3842u;
// Absolute slack, in the scale of s: operands and products below the normal
// ranges (far: the largest |r|), and exact distances (of unscaled coordinates)
// below float32's, each of whose roundings may be off by 2^-149.
__host__ __device__ inline float screen_slack(int D, float q, float far, float scale) {
    if (D == 3) return 1e-30f;
    const float tiny = scale * 5.3e-23f;  // 2^-74
    const float lost = static_cast<float>(D) * 1.2e-7f;
    return 1e-30f + lost * q + fminf(lost * far, lost * lost * 2.5e4f) +
           static_cast<float>(2 * D) * (tiny * tiny);
}

// bf16 parts of a float, rounded to nearest: v = hi + lo to 2^-18.
__device__ __forceinline__ uint32_t bf16_bits(float v) {
    const uint32_t u = static_cast<uint32_t>(f2i(v));
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_value(uint32_t bits) { return i2f(static_cast<int>(bits << 16)); }
__device__ __forceinline__ void bf16_split(float v, uint32_t& hi, uint32_t& lo) {
    hi = bf16_bits(v);
    lo = bf16_bits(v - bf16_value(hi));
}

__device__ __forceinline__ uint4 pack8(const uint32_t (&v)[8]) {
    return make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
}

__device__ __forceinline__ bf16x8 as_bf16(uint4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ f16x8 as_f16(uint4 v) { return __builtin_bit_cast(f16x8, v); }

// Eight floats rounded to f16 (to nearest; infinite beyond its range).
__device__ __forceinline__ uint4 f16_frag(const float (&f)[8]) {
    f16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = static_cast<_Float16>(f[i]);
    return __builtin_bit_cast(uint4, v);
}

// The value of the lane whose number differs in the bits X, within a group of 8.
template <int X>
__device__ __forceinline__ int xor8(int v) {
    constexpr int kQuadXor3 = 0x1B;
    if constexpr (X == 1) return dpp<kDppQuadXor1>(v);
    else if constexpr (X == 2) return dpp<kDppQuadXor2>(v);
    else if constexpr (X == 3) return dpp<kQuadXor3>(v);
    else if constexpr (X == 7) return dpp<kDppRowHalfMirror>(v);
    else return xor8<7 - X>(dpp<kDppRowHalfMirror>(v));
}
template <int X>
__device__ __forceinline__ int after8(uint32_t key, int i) {
    const uint32_t other = static_cast<uint32_t>(xor8<X>(static_cast<int>(key)));
    return other < key || (other == key && (i ^ X) < i) ? 1 : 0;
}
// Rank of a lane's key among its group of 8 lanes, equal keys by lane.
__device__ __forceinline__ int rank8(uint32_t key, int i) {
    return after8<1>(key, i) + after8<2>(key, i) + after8<3>(key, i) + after8<4>(key, i) +
           after8<5>(key, i) + after8<6>(key, i) + after8<7>(key, i);
}

// Row i of the eight that a segment of n rows is looked at by: spread over it,
// in no common step (clouds may carry something every so many rows).
__device__ __forceinline__ int64_t sample8(int64_t n, int i) {
    constexpr uint64_t lo = 27329ull << 48 | 18553ull << 32 | 9719ull << 16 | 2039ull;   // of 65536
    constexpr uint64_t hi = 60757ull << 48 | 51971ull << 32 | 43973ull << 16 | 35323ull;
    return (n * static_cast<int64_t>(((i < 4 ? lo : hi) >> (16 * (i & 3))) & 0xFFFFu)) >> 16;
}

// Of the two middle values of eight the one nearer to 0 (0 if neither is
// finite): with up to half of the eight somewhere else -- padding, strays --
// it lies among the others unless those are nearer to the origin.
__device__ __forceinline__ float nearer(float lower, float upper) {
    const float c = fabsf(upper) < fabsf(lower) ? upper : lower;
    return isfinite(c) ? c : 0.f;
}

// Centre of a 3-D segment for the screen (its coordinates are taken relative
// to it, which keeps E small for clouds far from the origin): per axis a middle
// one of 8 points spread over it.  Any point serves.  One wave, a lane per
// value; every wave of a launch computes the same for a segment.
__device__ __forceinline__ void screen_centre(const float* __restrict__ ref, int64_t n, int lane, float (&c)[3]) {
    const int i = lane & 7;
    const float v = ref[3 * sample8(n, i) + min(lane >> 3, 2)];
    const uint32_t bits = static_cast<uint32_t>(f2i(v));
    const uint32_t key = v != v ? 0xFFFFFFFFu : bits ^ ((bits >> 31) != 0 ? 0xFFFFFFFFu : 0x80000000u);
    const int rank = rank8(key, i);
    const uint64_t lower = ballot(rank == 3), upper = ballot(rank == 4);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const uint64_t group = uint64_t(0xFF) << (8 * a);
        c[a] = nearer(i2f(readlane(f2i(v), static_cast<int>(__builtin_ctzll(lower & group)))),
                      i2f(readlane(f2i(v), static_cast<int>(__builtin_ctzll(upper & group)))));
    }
}

// Eight dimensions from d0 of a row (0 behind the last).
__device__ __forceinline__ void load8(const float* __restrict__ r, int d0, int D, bool vec, float (&f)[8]) {
    if (vec) {
        // Unconditional loads (of dimension 0 behind the last), so that a
        // row's are all in flight together.
        const bool in_a = d0 < D, in_b = d0 + 4 < D;
        const float4 a = *reinterpret_cast<const float4*>(r + (in_a ? d0 : 0));
        const float4 b = *reinterpret_cast<const float4*>(r + (in_b ? d0 + 4 : 0));
        f[0] = in_a ? a.x : 0.f; f[1] = in_a ? a.y : 0.f; f[2] = in_a ? a.z : 0.f; f[3] = in_a ? a.w : 0.f;
        f[4] = in_b ? b.x : 0.f; f[5] = in_b ? b.y : 0.f; f[6] = in_b ? b.z : 0.f; f[7] = in_b ? b.w : 0.f;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = d0 + i < D ? r[d0 + i] : 0.f;
    }
}

// The middle one nearer to 0 of eight values (NaN counts as +inf).
__device__ __forceinline__ float middle_of(const float (&v)[8]) {
    float w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = v[i] == v[i] ? v[i] : INFINITY;
    auto order = [&](int i, int j) {
        const float a = w[i], b = w[j];
        w[i] = fminf(a, b);
        w[j] = fmaxf(a, b);
    };
    // Batcher's odd-even merge sort.
    order(0, 1); order(2, 3); order(4, 5); order(6, 7);
    order(0, 2); order(1, 3); order(4, 6); order(5, 7);
    order(1, 2); order(5, 6);
    order(0, 4); order(1, 5); order(2, 6); order(3, 7);
    order(2, 4); order(3, 5);
    order(1, 2); order(3, 4); order(5, 6);
    return nearer(w[3], w[4]);
}

// Centre and scale of a feature segment, from 8 rows spread over it: per
// dimension a middle value to centre[] (any serves), 0 behind D, and the power
// of two that takes the middle one of the rows' largest differences from it
// (of those that are not 0: repeated rows and padding) to [4, 8).  f16 reaches
// 8000 times further, and a row beyond that is not screened.  One wave, lane l
// for dimensions l and l + 64; every wave of a launch computes the same values
// for a segment.
constexpr int kScreenMaxD = 128;
__device__ __forceinline__ float screen_frame(const float* __restrict__ ref, int64_t n, int D, int lane,
                                              float* centre) {
    float most[8] = {};
    for (int t = lane; t < D; t += kWave) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = ref[sample8(n, i) * D + t];
        const float c = middle_of(v);
        centre[t] = c;
#pragma unroll
        for (int i = 0; i < 8; ++i) most[i] = fmaxf(most[i], fabsf(v[i] - c));  // (ignores NaN)
    }
    for (int t = D + lane; t < kScreenMaxD; t += kWave) centre[t] = 0.f;
    float mine = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float m = wave_max(most[i]);
        mine = (lane & 7) == i ? m : mine;
    }
    const bool some = mine > 1e-25f && mine < 1e25f;
    const int rank = rank8(some ? static_cast<uint32_t>(f2i(mine)) : 0xFFFFFFFFu, lane & 7);
    const int count = __popcll(ballot(some) & 0xFF);
    if (count == 0) return 1.f;
    const uint64_t at = ballot(rank == (count - 1) / 2) & 0xFF;
    const int bits = readlane(f2i(mine), static_cast<int>(__builtin_ctzll(at)));
    const int e = ((bits >> 23) & 0xFF) - 127;  // in [2^e, 2^(e+1))
    return i2f((2 - e + 127) << 23);
}

// Segment of the references (rows) or queries of tile / block t.
struct ScreenSegment {
    int64_t b;    // cloud
    int64_t lo;   // its first row
    int64_t n;    // its rows
    int64_t at;   // first row of this tile / block within it
};

// Tile or block `t` of `per` rows in the numbering of screen_tiles.
__device__ __forceinline__ ScreenSegment screen_segment(const int64_t* __restrict__ ptr, int64_t batch,
                                                        int64_t t, int per) {
    int64_t lo = 0, hi = batch - 1;
    while (lo < hi) {  // the last segment that begins at or before t
        const int64_t mid = lo + (hi - lo + 1) / 2;
        if (ptr[mid] / per + mid <= t) lo = mid;
        else hi = mid - 1;
    }
    ScreenSegment s;
    s.b = lo;
    s.lo = ptr[lo];
    s.n = ptr[lo + 1] - s.lo;
    s.at = (t - (s.lo / per + lo)) * per;
    return s;
}

// Half (lane / 32) of a 3-D reference's slots, its coordinates relative to the
// centre: h, h, l, l of the coordinates, the norm, and the norm once more for
// its part of the error bound; a row that is not `screened` is 0 with an
// infinite norm.  `sq`: its squared norm.
__device__ __forceinline__ uint4 ref_frag3(float x, float y, float z, float sq, bool screened, int half) {
    uint32_t h[3], l[3], nh, nm, nl;
    bf16_split(x, h[0], l[0]);
    bf16_split(y, h[1], l[1]);
    bf16_split(z, h[2], l[2]);
    nh = bf16_bits(sq);
    bf16_split(sq - bf16_value(nh), nm, nl);
    uint32_t v[8] = {h[0], h[1], h[2], h[0], h[1], h[2], l[0], l[1]};
    const uint32_t w[8] = {l[2], l[0], l[1], l[2], nh, nm, nl, nh};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = half ? w[i] : v[i];
        v[i] = screened ? v[i] : (half && i == 4 ? 0x7F80u : 0u);
    }
    return pack8(v);
}

// Whether a row or query is screened: finite, and close enough for the squares
// of sums to stay finite (NaN compares false).
__device__ __forceinline__ bool near_enough(float sq) { return sq < kScreenMaxSq; }

// One wave per tile: the references' fragments, norms and largest norm.
// Lane l holds row l % 32 and dimensions 8 (l / 32) .. + 7 of each k-step.
template <bool D3, bool FLAT>
__global__ __launch_bounds__(kPrepThreads) void screen_prep_kernel(
    const float* __restrict__ ref, const int64_t* __restrict__ ptr, const int* __restrict__ wanted,
    ScreenLayout L, int64_t batch, int64_t N, int64_t tiles, int D, int steps) {
    const int lane = lane_id();
    const int64_t t = static_cast<int64_t>(blockIdx.x) * (kPrepThreads / kWave) + uniform(threadIdx.x / kWave);
    if (t >= tiles) return;
    ScreenSegment s;
    if constexpr (FLAT) {
        s = screen_segment(ptr, batch, t, kTileRefs);
    } else {  // every cloud has the same number of tiles here
        const int64_t per = (N + kTileRefs - 1) / kTileRefs;
        s.b = t / per;
        if (wanted != nullptr && wanted[s.b] == 0) return;  // no query of the cloud is searched
        s.lo = s.b * N;
        s.n = N;
        s.at = (t - s.b * per) * kTileRefs;
    }
    if (s.at >= s.n) return;  // a number no segment uses
    const int row = lane & 31, half = lane >> 5;
    const bool valid = s.at + row < s.n;
    const float* r = ref + (s.lo + (valid ? s.at + row : 0)) * D;
    float sq = 0.f;
    bool screened;
    if constexpr (D3) {
        float c[3];
        screen_centre(ref + 3 * s.lo, s.n, lane, c);
        const float x = r[0] - c[0], y = r[1] - c[1], z = r[2] - c[2];
        sq = x * x + y * y + z * z;
        screened = valid && near_enough(sq);
        L.frag[t * kWave + lane] = ref_frag3(x, y, z, sq, screened, half);
    } else {
        // Coordinates relative to the segment's centre, scaled.
        const bool vec = D % 4 == 0 && reinterpret_cast<uintptr_t>(ref) % 16 == 0;
        __shared__ __align__(16) float centres[kPrepThreads / kWave][kScreenMaxD];
        float* const centre = centres[uniform(threadIdx.x / kWave)];
        const float scale = screen_frame(ref + s.lo * D, s.n, D, lane, centre);
        __builtin_amdgcn_wave_barrier();
        for (int k = 0; k < steps; ++k) {
            const int d0 = 16 * k + 8 * half;
            float f[8], o[8];
            load8(r, d0, D, vec, f);
            load8(centre, d0, kScreenMaxD, true, o);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                f[i] = valid ? (f[i] - o[i]) * scale : 0.f;  // (0 behind D)
                sq = sq + f[i] * f[i];
                if (!(fabsf(f[i]) < kScreenMaxRow)) sq = INFINITY;  // beyond f16, or NaN
            }
            L.frag[(t * steps + k) * kWave + lane] = f16_frag(f);
        }
        sq = sq + __shfl_xor(sq, 32, kWave);
        screened = valid && near_enough(sq);
        if (!screened)  // no products with what f16 made of it
            for (int k = 0; k < steps; ++k) L.frag[(t * steps + k) * kWave + lane] = make_uint4(0, 0, 0, 0);
        if (half == 0) L.norm[t * kTileRefs + row] = screened ? sq : INFINITY;
    }
    const float most = wave_max(screened ? sq : 0.f);
    const bool all = ballot(valid && !screened) == 0;
    if (lane == 0) L.far_sq[t] = all ? most : -most;
}

struct ScreenArgs {
    const float* query;
    const float* ref;
    const int64_t* ptr_y;  // FLAT: segment offsets of the queries and references
    const int64_t* ptr_x;
    float* dist;           // dense outputs
    int64_t* idx;          // dense or flat indices
    ScreenLayout L;
    int64_t batch, M, N;
    const int* list;        // LIST: per cloud, rows of its queries to search (M apart)
    const int* list_count;
    int D, K;
    bool squared;  // dense: distances squared, not their roots
};

// ---- the queries the screen leaves over
// Their references at or below the limit are found again as bits, kMaskTiles
// tiles at a time in index order, and ranked 64 at a time (LeftList).
constexpr int kMaskTiles = 126;
constexpr int kMaskStride = kMaskTiles + 1;  // words per query: odd, no bank conflicts
static_assert(kScreenQueries * kMaskStride <= kScreenQueries * kScreenCap, "masks fit the lists");
constexpr int kLeftMany = 8;    // more candidates at once are sorted and merged
constexpr int kLeftShares = 8;  // up to eight queries are searched by all waves, each a share

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int from) {
    const uint32_t lo = __shfl(static_cast<int>(v), from, kWave), hi = __shfl(static_cast<int>(v >> 32), from, kWave);
    return static_cast<uint64_t>(hi) << 32 | lo;
}
// One stage of a bitonic network on a word per lane: the lanes that differ in
// bit j exchange, ascending where `up`.
__device__ __forceinline__ uint64_t bitonic(uint64_t v, int j, bool up, int lane) {
    const uint64_t other = shfl64(v, lane ^ j);
    const bool least = ((lane & j) == 0) == up;
    return (other < v) == least ? other : v;
}

// The nearest references of one query, (distance bits, index) words in order
// over the lanes.  References are offered in index order, and only a distance
// below `below` is ranked: at first the bound that pass 1 gave, then, with
// K in the list, the K-th nearest so far (a later reference at that distance
// is behind it).  A list of zeros ends its query, which is how copies of one
// point are served.
struct LeftList {
    float d[1];
    int i[1];
    uint32_t below;

    __device__ __forceinline__ void settle(int K) {
        float last;
        int at;
        list_tail<1>(d, i, K, last, at);
        if (at != -1) below = min(below, static_cast<uint32_t>(f2i(last)));
    }
    // Takes the nearest 64 of the list and of another, in order.
    __device__ __forceinline__ void merge(uint64_t other, int lane) {
        const uint64_t mine = static_cast<uint64_t>(static_cast<uint32_t>(f2i(d[0]))) << 32 | static_cast<uint32_t>(i[0]);
        other = shfl64(other, kWave - 1 - lane);
        uint64_t word = other < mine ? other : mine;
#pragma unroll
        for (int j = kWave / 2; j > 0; j >>= 1) word = bitonic(word, j, true, lane);
        d[0] = i2f(static_cast<int>(word >> 32));
        i[0] = static_cast<int>(word);
    }
    // This lane's reference, if `in`: its index and distance.
    __device__ __forceinline__ void offer(bool in, int index, float dist, int K, int lane) {
        const int key = f2i(dist);  // (NaN is above every bound)
        uint64_t pending = ballot(in && static_cast<uint32_t>(key) < below);
        if (pending == 0) return;
        if (__popcll(pending) > kLeftMany) {
            uint64_t word = static_cast<uint64_t>(static_cast<uint32_t>(key)) << 32 | static_cast<uint32_t>(index);
            word = ((pending >> lane) & 1u) ? word : ~uint64_t(0);
#pragma unroll
            for (int k = 2; k <= kWave; k <<= 1)
#pragma unroll
                for (int j = k >> 1; j > 0; j >>= 1) word = bitonic(word, j, (lane & k) == 0, lane);
            merge(word, lane);
            settle(K);
            return;
        }
        do {
            const int src = __builtin_ctzll(pending);
            pending &= pending - 1;
            const int k = readlane(key, src);
            if (static_cast<uint32_t>(k) >= below) continue;  // an earlier one lowered it
            list_insert<1>(d, i, K, lane, i2f(k), readlane(index, src));
            settle(K);
        } while (pending != 0);
    }
};

// KS k-steps (D <= 16 KS); D3: one fragment holds everything.  Eight waves,
// each with an eighth of the tiles against all 64 queries (two columns of 32).
// PREP: the fragments come from screen_prep_kernel; otherwise (D3 only) each
// wave makes them from the coordinates as it goes, twice, which for small
// clouds costs less than a launch.  LIST: only the listed queries of each cloud.
template <int KS, bool D3, bool FLAT, bool PREP, bool LIST>
__global__ __launch_bounds__(kScreenThreads, D3 ? 4 : 2) void knn_screen_kernel(const ScreenArgs a) {
    constexpr int kBatch = D3 ? 4 : KS <= 4 ? 2 : 1;  // tiles in flight
    constexpr int kU = 2;               // columns of 32 queries
    constexpr int kFold = kScreenWaves * kTileRefs / kScreenGroups;  // rows of a lane per group
    // Pass 1's minima (and the rows of the exact phase).
    __shared__ __align__(16) float groups[kScreenGroups * kGroupStride + 1024];
    __shared__ __align__(16) uint32_t listed[kScreenQueries * kScreenCap];
    __shared__ __align__(16) uint32_t own_keys[D3 ? 4 : kScreenQueries * kScreenCap];
    __shared__ int count[kScreenQueries];
    __shared__ float limit[kScreenQueries];
    __shared__ float within[kScreenQueries];  // no less than the K-th smallest distance
    __shared__ float norm_q[kScreenQueries];
    __shared__ float far_red[kScreenWaves];
    __shared__ int left_q[kScreenQueries];
    __shared__ __align__(16) float centres[kScreenWaves][D3 ? 4 : kScreenMaxD];  // a copy per wave: no barrier
    // The exact phase: the listed references' keys (where the minima were, for
    // D3), and each wave's rows of 16 dimensions (where the minima were).
    uint32_t* const keys = D3 ? reinterpret_cast<uint32_t*>(groups) : own_keys;
    static_assert(kScreenGroups * kGroupStride >= kScreenQueries * kScreenCap, "keys fit");

    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = uniform(tid / kWave);
    const int col = lane & 31, half = lane >> 5;
    const int D = a.D;
    // This block's queries and their cloud's references.
    int64_t row0, ref0, n, tile0, b;
    int nq;
    if constexpr (FLAT) {
        const ScreenSegment s = screen_segment(a.ptr_y, a.batch, blockIdx.x, kScreenQueries);
        if (s.at >= s.n) return;  // a number no segment uses (uniform)
        b = s.b;
        row0 = s.lo + s.at;
        nq = static_cast<int>(min<int64_t>(kScreenQueries, s.n - s.at));
        ref0 = a.ptr_x[b];
        n = a.ptr_x[b + 1] - ref0;
        tile0 = ref0 / kTileRefs + b;
    } else {
        const CloudBlock cb = cloud_block(static_cast<uint32_t>((a.M + kScreenQueries - 1) / kScreenQueries));
        b = cb.b;
        const int64_t m0 = static_cast<int64_t>(cb.x) * kScreenQueries;
        row0 = b * a.M + m0;
        const int64_t rows = LIST ? a.list_count[b] : a.M;
        if (LIST && m0 >= rows) return;  // (uniform)
        nq = static_cast<int>(min<int64_t>(kScreenQueries, rows - m0));
        ref0 = b * a.N;
        n = a.N;
        tile0 = b * ((n + kTileRefs - 1) / kTileRefs);
    }
    // Row of query qi, of the queries and of the outputs.
    auto row_of = [&](int qi) -> int64_t { return LIST ? b * a.M + a.list[row0 + qi] : row0 + qi; };
    const int tiles = static_cast<int>((n + kTileRefs - 1) / kTileRefs);
    const int K = static_cast<int>(min<int64_t>(a.K, n));

    // ---- the queries' fragments, of -2 q (exact), and norms
    uint4 bq[kU][KS];
    float c[3] = {0.f, 0.f, 0.f};
    if constexpr (D3) {
        if (n > 0) screen_centre(a.ref + 3 * ref0, n, lane, c);
    }
    const bool vec = D % 4 == 0 && reinterpret_cast<uintptr_t>(a.query) % 16 == 0;
    const bool vec_rows = vec && reinterpret_cast<uintptr_t>(a.ref) % 16 == 0;
    float scale = 1.f;
    if constexpr (!D3) {
        if (n > 0) scale = screen_frame(a.ref + ref0 * D, n, D, lane, centres[wave]);
        else for (int t = lane; t < kScreenMaxD; t += kWave) centres[wave][t] = 0.f;
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
        const int qi = 32 * u + col;
        const float* q = a.query + row_of(qi < nq ? qi : 0) * D;
        float sq = 0.f;
        if constexpr (D3) {
            const float x = q[0] - c[0], y = q[1] - c[1], z = q[2] - c[2];
            sq = x * x + y * y + z * z;
            uint32_t h[3], l[3];
            bf16_split(-2.f * x, h[0], l[0]);
            bf16_split(-2.f * y, h[1], l[1]);
            bf16_split(-2.f * z, h[2], l[2]);
            // Slots: h, l, h, l against the references' h, h, l, l; 1 against
            // the norm's parts, and 2 E against the norm once more.
            uint32_t v[8] = {h[0], h[1], h[2], l[0], l[1], l[2], h[0], h[1]};
            const uint32_t w[8] = {h[2], l[0], l[1], l[2], 0x3F80u, 0x3F80u, 0x3F80u, kScreenError3};
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = half ? w[i] : v[i];
            bq[u][0] = pack8(v);
        } else {
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const int d0 = 16 * k + 8 * half;
                float f[8], o[8];
                load8(q, d0, D, vec, f);
                load8(centres[wave], d0, kScreenMaxD, true, o);
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    f[i] = (f[i] - o[i]) * scale;  // (0 behind D)
                    sq = sq + f[i] * f[i];
                    if (!(fabsf(f[i]) < kScreenMaxQuery)) sq = INFINITY;  // -2 f beyond f16, or NaN
                    f[i] = -2.f * f[i];
                }
                bq[u][k] = f16_frag(f);
            }
            sq = sq + __shfl_xor(sq, 32, kWave);
        }
        if (wave == 0 && half == 0) norm_q[qi] = sq;
    }
    if (tid < kScreenQueries) count[tid] = 0;
    // The wave's part of the largest |r|^2 (not needed for D3) and of whether
    // a row is left out (the sign).
    bool left_out = false;
    if constexpr (PREP) {
        float far_sq = 0.f;
        for (int i = tid; i < tiles; i += kScreenThreads) {
            const float v = a.L.far_sq[tile0 + i];
            far_sq = fmaxf(far_sq, fabsf(v));
            left_out = left_out || f2i(v) < 0;
        }
        far_sq = wave_max(far_sq);
        if (ballot(left_out) != 0) far_sq = -far_sq;
        if (lane == 0) far_red[wave] = far_sq;
    }

    // The screen of one tile against the wave's queries: acc[u][i] is s, with
    // the reference's part of the bound added (pass 1) or taken off (pass 2), of
    // reference 8 (i / 4) + 4 half + i % 4 and query 32 (u0 + u) + col.
    float norm_part = 1.f + 2.f * screen_error(D);  // (D3: a slot of the query's fragment)
    auto load = [&](int t, uint4 (&f)[KS], float4 (&nr)[D3 ? 1 : 4]) {
        if constexpr (!PREP) {  // the coordinates, for as_fragment
            const float* r = a.ref + 3 * (ref0 + min<int64_t>(t * kTileRefs + col, n - 1));
            f[0] = make_uint4(f2i(r[0]), f2i(r[1]), f2i(r[2]), 0);
            return;
        }
        const uint4* src = a.L.frag + (tile0 + t) * KS * kWave + lane;
#pragma unroll
        for (int k = 0; k < KS; ++k) f[k] = src[k * kWave];
        if constexpr (!D3) {
            const float* nrm = a.L.norm + (tile0 + t) * kTileRefs + 4 * half;
#pragma unroll
            for (int g = 0; g < 4; ++g) nr[g] = *reinterpret_cast<const float4*>(nrm + 8 * g);
        }
    };
    auto as_fragment = [&](int t, uint4& f) {
        if constexpr (!PREP) {
            const bool valid = t * kTileRefs + col < n;
            const float x = i2f(f.x) - c[0], y = i2f(f.y) - c[1], z = i2f(f.z) - c[2];
            const float sq = x * x + y * y + z * z;
            const bool screened = valid && near_enough(sq);
            left_out = left_out || (valid && !screened);
            f = ref_frag3(x, y, z, sq, screened, half);
        }
    };
    auto screen = [&](const uint4 (&f)[KS], const float4 (&nr)[D3 ? 1 : 4], f32x16 (&acc)[kU]) {
        if constexpr (D3) {
            const f32x16 zero = {};
#pragma unroll
            for (int u = 0; u < kU; ++u)
                acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16(f[0]), as_bf16(bq[u][0]), zero, 0, 0, 0);
        } else {
#pragma unroll
            for (int u = 0; u < kU; ++u)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    acc[u][4 * g] = nr[g].x * norm_part;
                    acc[u][4 * g + 1] = nr[g].y * norm_part;
                    acc[u][4 * g + 2] = nr[g].z * norm_part;
                    acc[u][4 * g + 3] = nr[g].w * norm_part;
                }
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int u = 0; u < kU; ++u)
                    acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16(f[k]), as_f16(bq[u][k]), acc[u], 0, 0, 0);
        }
    };
    // The wave's tiles of begin .. end - 1, kBatch at a time (the next ones
    // requested before the current ones are used): use(j, t, acc) for t = t0 +
    // kScreenWaves j, then flush(t0), for every batch.  Tiles behind the last
    // are replaced by the wave's first; use() sees t.
    auto walk = [&](int begin, int end, auto use, auto flush) {
        const int t_first = begin + wave;
        if (t_first >= end) return;
        uint4 f[kBatch][KS];
        float4 nr[kBatch][D3 ? 1 : 4];
        auto fetch = [&](int t0) {
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int t = t0 + j * kScreenWaves;
                load(t < end ? t : t_first, f[j], nr[j]);
            }
        };
        fetch(t_first);
        for (int t0 = t_first; t0 < end; t0 += kBatch * kScreenWaves) {
            uint4 cf[kBatch][KS];
            float4 cn[kBatch][D3 ? 1 : 4];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
#pragma unroll
                for (int k = 0; k < KS; ++k) cf[j][k] = f[j][k];
#pragma unroll
                for (int g = 0; g < (D3 ? 1 : 4); ++g) cn[j][g] = nr[j][g];
            }
            fetch(t0 + kBatch * kScreenWaves);
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                f32x16 acc[kU];
                const int t = t0 + j * kScreenWaves;
                as_fragment(t < end ? t : t_first, cf[j][0]);
                screen(cf[j], cn[j], acc);
                use(j, t, acc);
            }
            flush(t0);
        }
    };

    // Bit i from the sign of limit - s (set: beyond it): a comparison and a
    // select per bit wait for vcc each time (front end 367 -> 360 us, 3 ragged
    // clouds of 20000 with K = 16 and their grouping 631 -> 613 us).
    auto hits_of = [](float lim, const f32x16& acc) {
        uint32_t h = 0;
#pragma unroll
        for (int i = 15; i >= 0; --i)
            h = __builtin_amdgcn_alignbit(h, static_cast<uint32_t>(f2i(lim - acc[i])), 31);
        return ~h & 0xFFFFu;
    };

    // ---- pass 1: group minima
    {
        float m[kU][16];
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int i = 0; i < 16; ++i) m[u][i] = INFINITY;
        walk(0, tiles, [&](int, int, const f32x16 (&acc)[kU]) {  // (a tile again changes no minimum)
#pragma unroll
            for (int u = 0; u < kU; ++u)
#pragma unroll
                for (int i = 0; i < 16; ++i) m[u][i] = fminf(m[u][i], acc[u][i]);
        }, [](int) {});
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int i = 0; i < 16 / kFold; ++i) {
                float v = m[u][i];
                if constexpr (kFold == 2) v = fminf(v, m[u][i + 8]);  // 16 references on
                groups[((2 * wave + half) * (16 / kFold) + i) * kGroupStride + 32 * u + col] = v;
            }
    }
    if constexpr (!PREP) {
        const bool any = ballot(left_out) != 0;
        if (lane == 0) far_red[wave] = any ? -0.f : 0.f;
    }
    __syncthreads();  // minima, norms, largest norms, cleared counts
    float far_sq = 0.f;
    left_out = false;
#pragma unroll
    for (int w = 0; w < kScreenWaves; ++w) {
        far_sq = fmaxf(far_sq, fabsf(far_red[w]));
        left_out = left_out || f2i(far_red[w]) < 0;
    }

    // ---- the limit of each query: eight lanes per query, 16 groups each,
    // searched for the K-th smallest minimum.  Any threshold that K groups
    // reach serves; the search ends at one that few more reach.
    {
        const int qi = wave * 8 + (lane >> 3), part = lane & 7;
        const float nq_sq = norm_q[qi];
        float v[kScreenGroups / 8];
        float lo = INFINITY, hi = 0.f, sum = 0.f, some = 0.f;
#pragma unroll
        for (int k = 0; k < kScreenGroups / 8; ++k) {
            // fmaxf maps NaN to 0: such a query is not served by the screen.
            v[k] = fmaxf(groups[(8 * k + part) * kGroupStride + qi] + nq_sq, 0.f);
            const bool real = v[k] < INFINITY;  // the group holds a reference
            lo = fminf(lo, v[k]);
            hi = fmaxf(hi, real ? v[k] : 0.f);
            sum = sum + (real ? v[k] : 0.f);
            some = some + (real ? 1.f : 0.f);
        }
        auto dpp_f = [](float x, auto ctrl) { return i2f(dpp<decltype(ctrl)::value>(f2i(x))); };
        auto eight = [&](float x, auto op) {  // over the query's eight lanes
            x = op(x, dpp_f(x, std::integral_constant<int, kDppQuadXor1>{}));
            x = op(x, dpp_f(x, std::integral_constant<int, kDppQuadXor2>{}));
            return op(x, dpp_f(x, std::integral_constant<int, kDppRowHalfMirror>{}));
        };
        const float least = eight(lo, [](float x, float y) { return fminf(x, y); });
        hi = eight(hi, [](float x, float y) { return fmaxf(x, y); });  // every such group is within hi
        sum = eight(sum, [](float x, float y) { return x + y; });
        some = eight(some, [](float x, float y) { return x + y; });
        lo = least;
        // The first guess takes the minima as exponentially distributed above
        // the least; then the count says on which side, interpolating.
        float guess = least + (sum / some - least) * -__logf(1.f - fminf(static_cast<float>(K) / some, 0.99f));
        float reach_lo = 0.f, reach_hi = some;
        const int most = K + 2 + K / 8;
        bool done = some <= static_cast<float>(most);
        if (some < static_cast<float>(K)) {
            hi = 3e38f;  // everything finite is listed
        } else if (K == 1) {
            hi = least;  // one group reaches the least minimum
            done = true;
        }
        for (int it = 0; it < 12 && ballot(!done) != 0; ++it) {
            if (!(guess > lo && guess < hi) || it > 6) guess = 0.5f * (lo + hi);
            float reach = 0.f;
#pragma unroll
            for (int k = 0; k < kScreenGroups / 8; ++k) reach += v[k] <= guess ? 1.f : 0.f;
            reach = eight(reach, [](float x, float y) { return x + y; });
            if (!done) {
                if (reach >= K) {
                    hi = guess;
                    reach_hi = reach;
                } else {
                    lo = guess;
                    reach_lo = reach;
                }
                done = reach >= K && reach <= most;
                guess = lo + (hi - lo) * ((K + 1 - reach_lo) / (reach_hi - reach_lo));
            }
        }
        if (part == 0) {
            const float e = 2.f * screen_error(D) * nq_sq + screen_slack(D, sqrtf(nq_sq), sqrtf(far_sq), scale);
            const float reach = hi + e;  // K references are within it
            // Rows left out lie beyond every reach that is allowed here: (2^50 -
            // 2^48)^2 from such a query, or (65000 - 32000)^2 in one dimension.
            // (Norms in the coordinates' own scale, so that no distance overflows.)
            const float back = 1.f / scale;
            const bool served = qi < nq && nq_sq * back * back < kScreenMaxQuerySq &&
                                (D3 || far_sq * back * back < kScreenMaxSq) &&
                                (!left_out || (some >= static_cast<float>(K) &&
                                               reach < (D3 ? kScreenMaxReach : kScreenMaxReachF16)));
            // (Finite, so that the rows behind the last, at +inf, are not listed.)
            limit[qi] = served ? fminf(reach + e - nq_sq, 3e38f) : -INFINITY;
            within[qi] = served && some >= static_cast<float>(K) ? reach * 1.000001f * back * back : INFINITY;
            if (qi < nq && !served) count[qi] = kScreenCap + 1;
        }
    }
    __syncthreads();  // limits
    norm_part = 1.f - 2.f * screen_error(D);
    if constexpr (D3) {
#pragma unroll
        for (int u = 0; u < kU; ++u) bq[u][0].w ^= half ? 0x80000000u : 0u;  // - 2 E
    }

    // ---- pass 2: the references within each query's limit
    {
        float lim[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) lim[u] = limit[32 * u + col];
        // A batch's hits, 16 bits a tile, appended together: one atomic per
        // lane and column with hits.
        constexpr int kWords = (kBatch + 1) / 2;
        uint32_t hit[kU][kWords] = {};
        walk(0, tiles, [&](int j, int t, const f32x16 (&acc)[kU]) {
            const bool real = t < tiles;
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                float least = acc[u][0];
#pragma unroll
                for (int i = 1; i < 16; ++i) least = fminf(least, acc[u][i]);
                uint32_t h = 0;
                if (ballot(least <= lim[u]) != 0 && real) h = hits_of(lim[u], acc[u]);
                hit[u][j / 2] |= h << (16 * (j & 1));
            }
        }, [&](int t0) {
            int at[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                int n_hit = 0;
#pragma unroll
                for (int w = 0; w < kWords; ++w) n_hit += __popc(hit[u][w]);
                at[u] = 0;
                if (n_hit != 0) at[u] = atomicAdd(&count[32 * u + col], n_hit);
                if (at[u] + n_hit > kScreenCap) {  // left over: no more of its hits
                    lim[u] = -INFINITY;
#pragma unroll
                    for (int w = 0; w < kWords; ++w) hit[u][w] = 0;
                }
            }
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                uint32_t* list = listed + (32 * u + col) * kScreenCap;
#pragma unroll
                for (int w = 0; w < kWords; ++w)
                    while (hit[u][w] != 0) {
                        const int i = __builtin_ctz(hit[u][w]);
                        hit[u][w] &= hit[u][w] - 1;
                        // (Rows behind the last are at +inf, above every limit.)
                        const int t = t0 + (2 * w + (i >> 4)) * kScreenWaves;
                        list[at[u]] = t * kTileRefs + 8 * ((i >> 2) & 3) + 4 * half + (i & 3);
                        ++at[u];
                    }
            }
        });
    }
    __syncthreads();  // lists

    // This lane's reference row r against its query row q, as the searches
    // define it (all lanes take part).
    auto distance = [&](int64_t r, const float* q) -> float {
        if constexpr (D3) {
            const float* rr = a.ref + 3 * r;
            return sqdist3(rr[0], rr[1], rr[2], q[0], q[1], q[2]);
        } else if (vec_rows) {
            // The 64 rows, 16 dimensions at a time, through LDS: four lanes
            // read a row's 64 bytes together (a lane reading its own row
            // would fetch each of its cache lines once per 16 bytes).
            constexpr int kRow = 20;  // floats between rows: no bank conflicts
            float4* const rows = reinterpret_cast<float4*>(groups + wave * kWave * kRow);
            static_assert(kScreenWaves * kWave * kRow <= kScreenGroups * kGroupStride + 1024, "rows fit");
            float d = 0.f;  // 0 + d0^2 = d0^2
            const int part = lane & 3;
            float4 next[4], qn[4];
            const float* src[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                qn[k] = 4 * k < D ? *reinterpret_cast<const float4*>(q + 4 * k) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int64_t other = __shfl(r, 16 * k + (lane >> 2), kWave);
                src[k] = a.ref + other * D + 4 * part;
                next[k] = 4 * part < D ? *reinterpret_cast<const float4*>(src[k]) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            for (int d0 = 0; d0 < D; d0 += 16) {
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int k = 0; k < 4; ++k) rows[(16 * k + (lane >> 2)) * (kRow / 4) + part] = next[k];
                __builtin_amdgcn_wave_barrier();
                float4 x4[4], qc[4];  // (behind D: not used)
#pragma unroll
                for (int k = 0; k < 4; ++k) x4[k] = rows[lane * (kRow / 4) + k];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    qc[k] = qn[k];
                    if (d0 + 16 + 4 * part < D) next[k] = *reinterpret_cast<const float4*>(src[k] + d0 + 16);
                    if (d0 + 16 + 4 * k < D) qn[k] = *reinterpret_cast<const float4*>(q + d0 + 16 + 4 * k);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (d0 + 4 * k >= D) break;
                    const float4 x = x4[k], y = qc[k];
                    const float x0 = x.x - y.x, x1 = x.y - y.y, x2 = x.z - y.z, x3 = x.w - y.w;
                    d = d + x0 * x0;
                    d = d + x1 * x1;
                    d = d + x2 * x2;
                    d = d + x3 * x3;
                }
            }
            return d;
        } else {
            return sqdist_nd(a.ref + r * D, q, D);
        }
    };

    // ---- exact distances: the wave's eight queries' lists end to end, a lane
    // per listed reference
    constexpr int kMine = kScreenQueries / kScreenWaves;
    const int q0 = wave * kMine;
    int first[kMine + 1];  // where each query's list begins
    first[0] = 0;
#pragma unroll
    for (int i = 0; i < kMine; ++i) {
        const int m = q0 + i < nq ? uniform(count[q0 + i]) : 0;
        first[i + 1] = first[i] + (m > kScreenCap ? 0 : m);  // (longer: left over)
    }
    for (int e0 = 0; e0 < first[kMine]; e0 += kWave) {
        const int e = e0 + lane;
        const bool valid = e < first[kMine];
        int i = 0, base = 0;
#pragma unroll
        for (int o = 1; o < kMine; ++o) {
            const bool in = valid && e >= first[o];
            i = in ? o : i;
            base = in ? first[o] : base;
        }
        const int slot = (q0 + i) * kScreenCap + (valid ? e - base : 0);
        const int64_t r = ref0 + (valid ? listed[slot] : 0);
        const float* q = a.query + row_of(q0 + i) * D;
        const float d = distance(r, q);
        if (valid) keys[slot] = static_cast<uint32_t>(f2i(d));
    }
    __builtin_amdgcn_wave_barrier();

    // ---- ranks: half a wave per query
    for (int i = half; i < kMine; i += 2) {
        const int qi = q0 + i;
        if (qi >= nq || count[qi] > kScreenCap) continue;
        const int m = count[qi];
        const uint4* list4 = reinterpret_cast<const uint4*>(listed + qi * kScreenCap);
        const uint4* key4 = reinterpret_cast<const uint4*>(keys + qi * kScreenCap);
        for (int e = col; e < m; e += 32) {
            const uint32_t key = keys[qi * kScreenCap + e], at = listed[qi * kScreenCap + e];
            const uint64_t mine = static_cast<uint64_t>(key) << 32 | at;
            int rank = 0;
            auto before_mine = [&](uint32_t k, uint32_t r, int o) {
                const uint64_t other = static_cast<uint64_t>(o < m ? k : 0xFFFFFFFFu) << 32 | r;
                return other < mine ? 1 : 0;
            };
#pragma unroll 2
            for (int o = 0; o < m; o += 4) {  // (entries behind the list are read, not counted)
                const uint4 k = key4[o >> 2], l = list4[o >> 2];
                rank += before_mine(k.x, l.x, o) + before_mine(k.y, l.y, o + 1) +
                        before_mine(k.z, l.z, o + 2) + before_mine(k.w, l.w, o + 3);
            }
            if (rank < K) {
                const int64_t slot = row_of(qi) * a.K + rank;
                if constexpr (FLAT) {
                    a.idx[slot] = ref0 + at;
                } else {
                    const float d = i2f(static_cast<int>(key));
                    a.dist[slot] = a.squared ? d : sqrtf(d);
                    a.idx[slot] = at;
                }
            }
        }
        if constexpr (FLAT)  // a segment of fewer than K references
            for (int s = K + col; s < a.K; s += 32) a.idx[row_of(qi) * a.K + s] = -1;
    }

    // ---- the queries left over
    const bool mine_left = lane < nq && count[lane] > kScreenCap;
    const uint64_t left = ballot(mine_left);  // the same in every wave
    if (left == 0) return;
    const int lefts = __popcll(left);
    const int shares = lefts <= kScreenQueries / kLeftShares ? kLeftShares : 1;
    if (wave == 0 && mine_left) left_q[lanes_below(left)] = lane;
    __syncthreads();  // left_q; every wave has ranked: the lists and keys are free
    // List `item` (a query and share; item % 8 is its wave): 64 keys, 64 indices.
    auto keys_of = [&](int item) { return keys + item * kScreenCap + lane; };
    for (int item = wave; item < lefts * shares; item += kScreenWaves) {
        keys_of(item)[0] = 0x7F800000u;
        keys_of(item)[kWave] = 0xFFFFFFFFu;
    }
    if (tiles == 0) __syncthreads();  // (else the last of the loop's)
    for (int t0 = 0; t0 < tiles; t0 += kMaskTiles) {
        const int t1 = min(t0 + kMaskTiles, tiles);
        // The hits of these tiles, a word a query and tile; a query without a
        // limit takes every reference.
        uint16_t* const masks = reinterpret_cast<uint16_t*>(listed);
        float lim[kU];
        bool wanted[kU], every[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            lim[u] = limit[32 * u + col];
            wanted[u] = (left >> (32 * u + col)) & 1u;
            every[u] = lim[u] == -INFINITY;
        }
        walk(t0, t1, [&](int, int t, const f32x16 (&acc)[kU]) {
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const uint32_t h = hits_of(lim[u], acc[u]);
                if (wanted[u] && t < t1)
                    masks[((32 * u + col) * kMaskStride + t - t0) * 2 + half] = static_cast<uint16_t>(every[u] ? 0xFFFFu : h);
            }
        }, [](int) {});
        __syncthreads();  // masks
        for (int item = wave; item < lefts * shares; item += kScreenWaves) {
            const int qi = uniform(left_q[item / shares]), share = item % shares;
            const float* q = a.query + row_of(qi) * D;
            // Nothing is at a distance from a query that is not finite (dense
            // 3-D searches match at infinite distances).
            bool never = false;
            for (int t = lane; t < D; t += kWave) never = never || (D3 && !FLAT ? q[t] != q[t] : !isfinite(q[t]));
            if (ballot(never) != 0) continue;
            LeftList list;
            list.d[0] = i2f(static_cast<int>(keys_of(item)[0]));
            list.i[0] = static_cast<int>(keys_of(item)[kWave]);
            list.below = static_cast<uint32_t>(uniform(min(f2i(within[qi]), D3 && !FLAT ? 0x7F800000 : 0x7F7FFFFF))) + 1u;
            list.settle(a.K);
            // Lane l looks at tiles 2 l and 2 l + 1; then the pairs with hits
            // one by one, lane l at reference l, their hits queued over the
            // lanes until 64 are there.
            const uint32_t* words = listed + qi * kMaskStride;
            const int pairs = (t1 - t0 + 1) / 2;
            auto word_of = [&](int t) { return t < t1 - t0 ? words[t] : 0u; };
            uint64_t todo = ballot(lane < pairs && lane % shares == share &&
                                   (word_of(2 * lane) | word_of(2 * lane + 1)) != 0);
            int queued = 0, queue = 0;
            auto rank = [&]() {
                const bool in = lane < queued;
                const int at = in ? queue : 0;
                list.offer(in, at, distance(ref0 + at, q), a.K, lane);
                queued = 0;
            };
            while (todo != 0 && list.below != 0) {
                const int pair = static_cast<int>(__builtin_ctzll(todo));
                todo &= todo - 1;
                const int j = (t0 + 2 * pair) * kTileRefs + lane;
                const uint32_t word = word_of(2 * pair + half);
                const int bit = 16 * ((lane >> 2) & 1) + 4 * ((lane >> 3) & 3) + (lane & 3);
                const bool hit = ((word >> bit) & 1u) != 0 && j < n;
                const uint64_t hits = ballot(hit);
                const int more = __popcll(hits);
                // Every lane sends its index to a lane of its own: the hits in
                // order from lane `queued` on, around the end.
                const int to = (queued + (hit ? lanes_below(hits) : more + lanes_below(~hits))) & (kWave - 1);
                const int sent = __builtin_amdgcn_ds_permute(to << 2, j);
                const int place = (lane - queued) & (kWave - 1);
                const bool fits = place < more && place + queued < kWave;
                queue = fits ? sent : queue;
                const int total = queued + more;
                queued = min(total, kWave);
                if (total >= kWave) {
                    rank();
                    queue = sent;  // the others, from lane 0 on
                    queued = total - kWave;
                }
            }
            if (queued != 0 && list.below != 0) rank();
            keys_of(item)[0] = static_cast<uint32_t>(f2i(list.d[0]));
            keys_of(item)[kWave] = static_cast<uint32_t>(list.i[0]);
        }
        __syncthreads();  // masks read, lists written
    }
    for (int r = wave; r < lefts; r += kScreenWaves) {
        const int qi = uniform(left_q[r]);
        LeftList list;
        list.d[0] = i2f(static_cast<int>(keys_of(r * shares)[0]));
        list.i[0] = static_cast<int>(keys_of(r * shares)[kWave]);
        for (int s = 1; s < shares; ++s)
            list.merge(static_cast<uint64_t>(keys_of(r * shares + s)[0]) << 32 | keys_of(r * shares + s)[kWave], lane);
        if (lane >= a.K) continue;
        const float d = list.d[0];
        const int at = list.i[0];
        const int64_t slot = row_of(qi) * a.K + lane;
        if constexpr (FLAT) {
            a.idx[slot] = at < 0 ? int64_t(-1) : ref0 + at;
        } else {
            a.dist[slot] = a.squared ? d : sqrtf(d);
            a.idx[slot] = D3 ? static_cast<int64_t>(static_cast<uint32_t>(at))
                             : (at < 0 ? int64_t(-1) : int64_t(at));
        }
    }
}

template <int KS, bool D3, bool FLAT, bool PREP = true, bool LIST = false>
hipError_t launch_search(const ScreenArgs& a, int64_t blocks, hipStream_t stream) {
    hipLaunchKernelGGL((knn_screen_kernel<KS, D3, FLAT, PREP, LIST>), dim3(static_cast<uint32_t>(blocks)),
                       dim3(kScreenThreads), 0, stream, a);
    return hipGetLastError();
}

// k-steps of the kernel that serves D dimensions.
int screen_kernel_steps(int64_t D) {
    const int s = screen_steps(D);
    return D == 3 ? 1 : s <= 2 ? 2 : s <= 4 ? 4 : s <= 6 ? 6 : 8;
}

size_t screen_workspace(int64_t rows, int64_t batch, int64_t D, ScreenLayout* L = nullptr, void* base = nullptr) {
    return screen_layout(rows, batch, D == 3 ? 3 : 16 * screen_kernel_steps(D), L, static_cast<char*>(base));
}

// The references' fragments (into a.L), which depend on the references alone.
// `lds`: bytes the blocks take without using them.
template <bool FLAT>
hipError_t launch_prep(const ScreenArgs& a, int64_t ref_rows, hipStream_t stream, size_t lds = 0) {
    const int64_t tiles = FLAT ? screen_tiles(ref_rows, a.batch) : a.batch * ((a.N + kTileRefs - 1) / kTileRefs);
    constexpr int kPrepWaves = kPrepThreads / kWave;
    const dim3 grid(static_cast<uint32_t>((tiles + kPrepWaves - 1) / kPrepWaves));
    if (a.D == 3)
        hipLaunchKernelGGL((screen_prep_kernel<true, FLAT>), grid, dim3(kPrepThreads), lds, stream, a.ref,
                           a.ptr_x, a.list_count, a.L, a.batch, a.N, tiles, a.D, 1);
    else
        hipLaunchKernelGGL((screen_prep_kernel<false, FLAT>), grid, dim3(kPrepThreads), lds, stream, a.ref,
                           a.ptr_x, a.list_count, a.L, a.batch, a.N, tiles, a.D, screen_kernel_steps(a.D));
    return hipGetLastError();
}

template <bool FLAT>
hipError_t launch_blocks(const ScreenArgs& a, int64_t blocks, hipStream_t stream) {
    switch (screen_kernel_steps(a.D)) {
        case 1: return launch_search<1, true, FLAT>(a, blocks, stream);
        case 2: return launch_search<2, false, FLAT>(a, blocks, stream);
        case 4: return launch_search<4, false, FLAT>(a, blocks, stream);
        case 6: return launch_search<6, false, FLAT>(a, blocks, stream);
        default: return launch_search<8, false, FLAT>(a, blocks, stream);
    }
}

template <bool FLAT>
hipError_t launch_screen(ScreenArgs a, void* workspace, int64_t ref_rows, int64_t blocks,
                         hipStream_t stream) {
    screen_workspace(ref_rows, a.batch, a.D, &a.L, workspace);
    const hipError_t err = launch_prep<FLAT>(a, ref_rows, stream);
    return err != hipSuccess ? err : launch_blocks<FLAT>(a, blocks, stream);
}

int64_t screen_blocks(int64_t M, int64_t B) { return (M + kScreenQueries - 1) / kScreenQueries * B; }

bool screen_fits(int64_t blocks, int64_t ref_rows, int64_t batch) {
    return blocks <= INT32_MAX && screen_tiles(ref_rows, batch) <= INT32_MAX / 2;
}

}  // namespace
}  // namespace pointops

namespace pointops {

// The dense 3-D search in two launches: knn3_screen_prepare (the references'
// fragments into `workspace`, pointops_knn_screen_workspace_bytes(B, N, 3)
// bytes) and knn3_screen_rows (the queries, over a workspace filled for the same
// references, B and N, or without one).
hipError_t knn3_screen_prepare(const float* ref, void* workspace, int64_t B, int64_t N, hipStream_t stream) {
    if (B < 1 || N < 1 || workspace == nullptr || N > INT32_MAX - kWave || !screen_fits(B, B * N, B))
        return hipErrorInvalidValue;
    ScreenArgs a{};
    a.ref = ref;
    a.batch = B;
    a.N = N;
    a.D = 3;
    screen_workspace(B * N, B, 3, &a.L, workspace);
    // Beside a pipelined FPS, which reserves the LDS of its CUs so that no other
    // block takes issue slots there: this kernel has none of its own.
    return launch_prep<false>(a, B * N, stream, 1024);
}

hipError_t knn3_screen_rows(const float* query, const float* ref, float* dist, int64_t* idx,
                            void* workspace, int64_t B, int64_t M, int64_t N, int64_t K,
                            hipStream_t stream) {
    if (B < 1 || M < 1 || K < 1 || K > kScreenMaxK || K > N || N > INT32_MAX - kWave ||
        !screen_fits(screen_blocks(M, B), B * N, B))
        return hipErrorInvalidValue;
    ScreenArgs a{};
    a.query = query;
    a.ref = ref;
    a.dist = dist;
    a.idx = idx;
    a.batch = B;
    a.M = M;
    a.N = N;
    a.D = 3;
    a.K = static_cast<int>(K);
    if (workspace == nullptr) return launch_search<1, true, false, false>(a, screen_blocks(M, B), stream);
    screen_workspace(B * N, B, 3, &a.L, workspace);
    return launch_blocks<false>(a, screen_blocks(M, B), stream);
}

// The nearest reference (squared distance, smallest index) of the first
// count[b] queries of each cloud's list, M ints a cloud, whose other rows are
// not written; clouds without any cost two empty launches.
hipError_t nearest3_screen_listed(const float* query, const float* ref, const int* count, const int* list,
                                  float* dist2, int64_t* idx, void* workspace, int64_t B, int64_t M,
                                  int64_t N, hipStream_t stream) {
    if (B < 1 || M < 1 || N < 1 || N > INT32_MAX - kWave || workspace == nullptr ||
        !screen_fits(screen_blocks(M, B), B * N, B))
        return hipErrorInvalidValue;
    ScreenArgs a{};
    a.query = query;
    a.ref = ref;
    a.dist = dist2;
    a.idx = idx;
    a.batch = B;
    a.M = M;
    a.N = N;
    a.list = list;
    a.list_count = count;
    a.D = 3;
    a.K = 1;
    a.squared = true;
    screen_workspace(B * N, B, 3, &a.L, workspace);
    const hipError_t err = launch_prep<false>(a, B * N, stream);
    if (err != hipSuccess) return err;
    return launch_search<1, true, false, true, true>(a, screen_blocks(M, B), stream);
}

}  // namespace pointops

using namespace pointops;

extern "C" {

size_t pointops_knn_screen_workspace_bytes(int64_t B, int64_t N, int64_t D) {
    if (B <= 0 || N <= 0 || D < 1 || D > 128) return 0;
    return screen_workspace(B * N, B, D);
}

hipError_t pointops_knn_screen(const float* query, const float* ref, float* dist, int64_t* idx,
                               void* workspace, int64_t B, int64_t M, int64_t N, int64_t D,
                               int64_t K, hipStream_t stream) {
    if (B < 0 || M < 0 || N < 0 || D < 1 || D > 128 || K < 0 || K > kScreenMaxK || K > N)
        return hipErrorInvalidValue;
    if (B == 0 || M == 0 || K == 0) return hipSuccess;
    const int64_t blocks = screen_blocks(M, B);
    if (workspace == nullptr || N > INT32_MAX - kWave || !screen_fits(blocks, B * N, B))
        return hipErrorInvalidValue;
    ScreenArgs a{};
    a.query = query;
    a.ref = ref;
    a.dist = dist;
    a.idx = idx;
    a.batch = B;
    a.M = M;
    a.N = N;
    a.D = static_cast<int>(D);
    a.K = static_cast<int>(K);
    return launch_screen<false>(a, workspace, B * N, blocks, stream);
}

hipError_t pointops_nearest3_screen(const float* query, const float* ref, float* dist2, int64_t* idx,
                                    void* workspace, int64_t B, int64_t M, int64_t N,
                                    hipStream_t stream) {
    if (B < 0 || M < 0 || N < 1) return hipErrorInvalidValue;
    if (B == 0 || M == 0) return hipSuccess;
    const int64_t blocks = screen_blocks(M, B);
    if (workspace == nullptr || N > INT32_MAX - kWave || !screen_fits(blocks, B * N, B))
        return hipErrorInvalidValue;
    ScreenArgs a{};
    a.query = query;
    a.ref = ref;
    a.dist = dist2;
    a.idx = idx;
    a.batch = B;
    a.M = M;
    a.N = N;
    a.D = 3;
    a.K = 1;
    a.squared = true;
    return launch_screen<false>(a, workspace, B * N, blocks, stream);
}

size_t pointops_knn_flat_screen_workspace_bytes(int64_t total_x, int64_t batch, int64_t D) {
    if (total_x < 0 || batch <= 0 || D < 1 || D > 128) return 0;
    return screen_workspace(total_x, batch, D);
}

hipError_t pointops_knn_flat_screen(const float* y, const float* x, const int64_t* ptr_y,
                                    const int64_t* ptr_x, int64_t* out, void* workspace, int64_t Q,
                                    int64_t total_x, int64_t batch, int64_t D, int64_t K,
                                    hipStream_t stream) {
    if (Q < 0 || total_x < 0 || batch < 0 || D < 1 || D > 128 || K < 0 || K > kScreenMaxK)
        return hipErrorInvalidValue;
    if (Q == 0 || K == 0) return hipSuccess;
    const int64_t blocks = Q / kScreenQueries + batch;
    if (batch == 0 || workspace == nullptr || total_x > INT32_MAX - kWave ||
        !screen_fits(blocks, total_x, batch))
        return hipErrorInvalidValue;
    ScreenArgs a{};
    a.query = y;
    a.ref = x;
    a.ptr_y = ptr_y;
    a.ptr_x = ptr_x;
    a.idx = out;
    a.batch = batch;
    a.D = static_cast<int>(D);
    a.K = static_cast<int>(K);
    return launch_screen<true>(a, workspace, total_x, blocks, stream);
}

}  // extern "C"
