// Setup kernels (see setup_kernels.hpp).
#include <cmath>
#include <vector>

#include "setup_kernels.hpp"

#include <algorithm>
#include <mutex>
#include <utility>
#include <vector>

namespace naga_amd {

namespace {

constexpr uint64_t kMaxKey = ~0ull;

__device__ __forceinline__ uint64_t shfl64(uint64_t v, int src) {
    const int lo = __shfl(int(uint32_t(v)), src);
    const int hi = __shfl(int(uint32_t(v >> 32)), src);
    return (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo);
}

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int m) {
    const int lo = __shfl_xor(int(uint32_t(v)), m);
    const int hi = __shfl_xor(int(uint32_t(v >> 32)), m);
    return (uint64_t(uint32_t(hi)) << 32) | uint32_t(lo);
}

// FP32 squared distance, fixed order, no contraction (the kNN key).
__device__ __forceinline__ float dist2_f32(int D, const float* a, const float* b) {
#pragma clang fp contract(off)
    float s = (a[0] - b[0]) * (a[0] - b[0]);
    for (int d = 1; d < D; ++d) {
        const float t = (a[d] - b[d]) * (a[d] - b[d]);
        s = t + s;
    }
    return s;
}

// bitonic sort of one key per lane across the wavefront, ascending
__device__ __forceinline__ uint64_t wave_sort64(uint64_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int kk = 2; kk <= 64; kk <<= 1)
#pragma unroll
        for (int j = kk >> 1; j > 0; j >>= 1) {
            const uint64_t p = shfl_xor64(v, j);
            const bool up = (lane & kk) == 0, lower = (lane & j) == 0;
            v = (lower == up) ? (p < v ? p : v) : (p > v ? p : v);
        }
    return v;
}

// sort a bitonic sequence ascending
__device__ __forceinline__ uint64_t wave_merge64(uint64_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 32; j > 0; j >>= 1) {
        const uint64_t p = shfl_xor64(v, j);
        const bool lower = (lane & j) == 0;
        v = lower ? (p < v ? p : v) : (p > v ? p : v);
    }
    return v;
}

// Merge the candidates of one 64-wide batch into the running top list
// (lane t holds the t-th smallest key).
__device__ __forceinline__ void knn_merge(uint64_t key, uint64_t& top, uint64_t& kth, int k) {
    if (!__any(key < kth)) return;
    const int lane = threadIdx.x & 63;
    const uint64_t sorted = wave_sort64(key);
    const uint64_t rev = shfl64(sorted, 63 - lane);
    top = wave_merge64(top < rev ? top : rev);
    kth = shfl64(top, k - 1);
}

// The kNN key of a binned point: FP32 squared distance, then index.
template <int D>
__device__ __forceinline__ uint64_t knn_key(const float* x, const float4& c) {
    const float p[3] = {c.x, c.y, c.z};
    return (uint64_t(__float_as_uint(dist2_f32(D, x, p))) << 32) | __float_as_uint(c.w);
}

// One query by rings of cells around its own: the ring's rows of cells are
// looked up 64 at a time, one per lane, and those that hold points are
// merged, 64 points at a time, into the running list, until the k-th distance
// is inside the searched box.  Takes any cloud; knn_box serves most queries.
// (Queries far from a hollow cloud pass many empty rings: visiting every row
// by the whole wavefront made the nodes' distance to the boundary most of a
// grid's set-up.)
template <int D>
__device__ void knn_rings(const CellGrid& G, const float4* cpts, const uint32_t* start,
                          const float* x, int64_t q, int k, float* d2o, uint32_t* idxo) {
    const int lane = threadIdx.x & 63;
    int64_t qc[3] = {0, 0, 0};
    for (int d = 0; d < D; ++d) {
        int64_t c = int64_t(floor((double(x[d]) - G.lo[d]) / G.w));
        qc[d] = c < 0 ? 0 : c >= G.dims[d] ? G.dims[d] - 1 : c;
    }
    uint64_t top = kMaxKey, kth = kMaxKey;
    for (int64_t r = 0;; ++r) {
        // rows of the ring inside the grid
        const int64_t y0 = qc[1] - r < 0 ? 0 : qc[1] - r;
        const int64_t y1 = qc[1] + r >= G.dims[1] ? G.dims[1] - 1 : qc[1] + r;
        const int64_t z0 = D == 2 ? 0 : qc[2] - r < 0 ? 0 : qc[2] - r;
        const int64_t z1 = D == 2 ? 0 : qc[2] + r >= G.dims[2] ? G.dims[2] - 1 : qc[2] + r;
        const int64_t ny = y1 - y0 + 1, nrow = ny * (z1 - z0 + 1);
        const int64_t xa = qc[0] - r, xb = qc[0] + r;
        const int64_t xl = xa < 0 ? 0 : xa, xr = xb >= G.dims[0] ? G.dims[0] - 1 : xb;
        for (int64_t b0 = 0; b0 < nrow; b0 += 64) {
            // the row's points: a whole row of cells on the ring's faces in
            // y and z, else the cells at its two ends
            uint32_t p0 = 0, p1 = 0, s0 = 0, s1 = 0;
            if (b0 + lane < nrow) {
                const int64_t cz = z0 + (b0 + lane) / ny, cy = y0 + (b0 + lane) % ny;
                const int64_t row = G.dims[0] * (cy + G.dims[1] * cz);
                const bool face = cy == qc[1] - r || cy == qc[1] + r ||
                                  (D == 3 && (cz == qc[2] - r || cz == qc[2] + r));
                if (face) {
                    p0 = start[row + xl];
                    p1 = start[row + xr + 1];
                } else {
                    if (xa >= 0) {
                        p0 = start[row + xa];
                        p1 = start[row + xa + 1];
                    }
                    if (xb < G.dims[0]) {
                        s0 = start[row + xb];
                        s1 = start[row + xb + 1];
                    }
                }
            }
            for (uint64_t has = __ballot(p0 < p1 || s0 < s1); has; has &= has - 1) {
                const int l = int(__ffsll((unsigned long long)has)) - 1;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const uint32_t a = __builtin_amdgcn_readlane(int(t ? s0 : p0), l);
                    const uint32_t e = __builtin_amdgcn_readlane(int(t ? s1 : p1), l);
                    for (uint32_t base = a; base < e; base += 64) {
                        const uint64_t key =
                            base + lane < e ? knn_key<D>(x, cpts[base + lane]) : kMaxKey;
                        knn_merge(key, top, kth, k);
                    }
                }
            }
        }
        double bound = 1e300;
        bool all = true;
        for (int d = 0; d < D; ++d) {
            if (qc[d] - r > 0) {
                const double t = double(x[d]) - (G.lo[d] + double(qc[d] - r) * G.w);
                bound = t < bound ? t : bound;
                all = false;
            }
            if (qc[d] + r < G.dims[d] - 1) {
                const double t = (G.lo[d] + double(qc[d] + r + 1) * G.w) - double(x[d]);
                bound = t < bound ? t : bound;
                all = false;
            }
        }
        if (all) break;
        if (kth != kMaxKey && bound > 0.0) {
            const double kd = double(__uint_as_float(uint32_t(kth >> 32)));
            if (kd < bound * bound * (1.0 - 1e-5)) break;
        }
    }
    if (lane < k) {
        d2o[q * k + lane] = __uint_as_float(uint32_t(top >> 32));
        idxo[q * k + lane] = uint32_t(top);
    }
}

// One query by the box of cells within R of its own: the points closer than
// a filter radius (the radius expected to hold about 1.75 k + 8 of them at
// the box's density, at most the distance to the box's nearest open side)
// are compacted into LDS, a bound that leaves k to 64 of them is found by
// ballots, and those are ranked by counting.  More points than fit are
// filtered again, below a bound taken from those kept.  Returns false, having
// written nothing, where the box cannot decide (too few points inside up to
// R = 3, more than kKnnKeep left after the retries): the caller then searches
// by rings.
//
// Bound by VALU issue, not bytes (1M points: 0.28 GB in and out, 0.05 ms at
// the card's copy rate).  Merging every cell row into a sorted list of 64-bit
// keys took 11 wavefront sorts per query; here a candidate costs about 20
// instructions once and only 64 keys are ordered, by counting smaller ones
// (broadcast LDS reads, no shuffles).  1,030,301 cube nodes, k = 32: 14.4 ->
// 1.4 ms; 1M random points 1.7 ms; 1M square nodes, k = 16: 0.8 ms.  200,000
// points that repeat 300-fold, k = 16: 0.55 ms in 2D (by rings 1.9).
constexpr int kKnnKeep = 256;   // points kept of one query (four per lane)
constexpr int kKnnMaxBox = 4096;  // points of a box visited by one wavefront
constexpr int kKnnBlockQueries = 16;  // queries per block: four per wavefront

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int D>
__device__ bool knn_box(const CellGrid& G, double inv_w, const float4* __restrict__ cpts,
                        const uint32_t* __restrict__ start, const float* x, int64_t q, int k,
                        uint64_t* keep, float* d2o, uint32_t* idxo) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (uint64_t(1) << lane) - 1;
    int dims[3], qc[3] = {0, 0, 0};  // at most 2^20 cells per dimension
#pragma unroll
    for (int d = 0; d < 3; ++d) dims[d] = int(G.dims[d]);
#pragma unroll
    for (int d = 0; d < D; ++d) {
        // within rounding of the cell's edge either cell serves: the bounds
        // below are taken from this one
        const double c = floor((double(x[d]) - G.lo[d]) * inv_w);
        qc[d] = __builtin_amdgcn_readfirstlane(
            c >= double(dims[d] - 1) ? dims[d] - 1 : c > 0.0 ? int(c) : 0);
    }
    for (int R = 1; R <= 3; ++R) {
        // the box's rows of cells (x fastest), one per lane
        const int side = 2 * R + 1, nrows = D == 3 ? side * side : side;
        int xa = qc[0] - R, xb = qc[0] + R;
        xa = xa < 0 ? 0 : xa;
        xb = xb >= dims[0] ? dims[0] - 1 : xb;
        const int cy = qc[1] + lane % side - R, cz = D == 3 ? qc[2] + lane / side - R : 0;
        const bool in = lane < nrows && cy >= 0 && cy < dims[1] && cz >= 0 &&
                        (D == 2 || cz < dims[2]);
        uint32_t p0 = 0, p1 = 0;
        if (in) {
            const int64_t row = int64_t(dims[0]) * (cy + int64_t(dims[1]) * cz);
            p0 = start[row + xa];
            p1 = start[row + xb + 1];
        }
        int T = int(p1 - p0);
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) T += __shfl_xor(T, o);
        T = __builtin_amdgcn_readfirstlane(T);
        // squared distance within which every point lies in the box
        double bound = 1e300;
        bool open = false;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (qc[d] - R > 0) {
                const double t = double(x[d]) - (G.lo[d] + double(qc[d] - R) * G.w);
                bound = t < bound ? t : bound;
                open = true;
            }
            if (qc[d] + R < dims[d] - 1) {
                const double t = (G.lo[d] + double(qc[d] + R + 1) * G.w) - double(x[d]);
                bound = t < bound ? t : bound;
                open = true;
            }
        }
        if (T == 0) return false;  // far from the cloud
        if (T < k || (open && bound <= 0.0)) {
            if (!open) return false;
            continue;
        }
        if (T > kKnnMaxBox) return false;
        const float b2 = open ? float(bound * bound * (1.0 - 1e-5)) : __builtin_inff();
        const float cells = float((xb - xa + 1) * __popcll(__ballot(in)));
        const float vol = cells * float(G.w) * float(G.w) * (D == 3 ? float(G.w) : 1.0f) *
                          (1.75f * float(k) + 8.0f) / float(T);
        float f2 = D == 3 ? exp2f(log2f(vol * 0.238732f) * (2.0f / 3.0f)) : vol * 0.318310f;
        if (!(f2 < b2)) f2 = b2;
        // points are kept whose key is below lim (their distance below f2, or
        // past a key known to have at least k below it); none above `most`
        uint64_t most = uint64_t(__float_as_uint(b2)) << 32;
        uint64_t lim = uint64_t(__float_as_uint(f2)) << 32;
        bool shrink = true;  // the radius may still be guessed from the count
        for (int attempt = 0; attempt < 6; ++attempt) {
            // keys of the box's points below lim, compacted
            int M = 0;
            for (int r0 = 0; r0 < nrows; r0 += 3) {
                uint32_t a[3], e[3];
                float4 c[3];
#pragma unroll
                for (int u = 0; u < 3; ++u) {
                    const int r = r0 + u < 64 ? r0 + u : 63;  // past the rows: empty
                    a[u] = __builtin_amdgcn_readlane(p0, r);
                    e[u] = __builtin_amdgcn_readlane(p1, r);
                    c[u] = a[u] + lane < e[u] ? cpts[a[u] + lane] : make_float4(0.f, 0.f, 0.f, 0.f);
                }
#pragma unroll
                for (int u = 0; u < 3; ++u)
                    while (a[u] < e[u]) {
                        const uint64_t key = knn_key<D>(x, c[u]);
                        const bool hit = a[u] + lane < e[u] && key < lim;
                        const uint64_t m = __ballot(hit);
                        const int at = M + __popcll(m & below);
                        if (hit && at < kKnnKeep) keep[at] = key;
                        M += __popcll(m);
                        a[u] += 64;
                        if (a[u] + lane < e[u]) c[u] = cpts[a[u] + lane];
                    }
            }
            if (M < k) {  // the radius was too small; the whole bound, then a larger box
                if (lim >= most) break;
                lim = most;
                shrink = false;
                continue;
            }
            wave_lds_fence();
            uint64_t key[kKnnKeep / 64];
#pragma unroll
            for (int e = 0; e < kKnnKeep / 64; ++e)
                key[e] = lane + 64 * e < M ? keep[lane + 64 * e] : kMaxKey;
            int C = M;
            uint64_t t = lim;  // C of the kept keys are below t
            if (M > 64) {
                // bounds with fewer than k (lo) and more than 64 (hi) kept
                // keys below them; the middle by distance, then one of the
                // keys between them: they are distinct, so that some bound
                // leaves k to 64 also where distances are equal
                uint64_t lo = 0, hi = lim;
                const float s = (float(k) + 0.5f * float(64 - k)) /
                                float(M < kKnnKeep ? M : kKnnKeep);
                float v = fminf(f2, 3.4e38f) * (D == 3 ? exp2f(log2f(s) * (2.0f / 3.0f)) : s);
                for (int step = 0;; ++step) {
                    if (step < 6) {
                        t = uint64_t(__float_as_uint(v)) << 32;
                    } else if (step < 64) {
                        uint64_t p = 0;
#pragma unroll
                        for (int e = 0; e < kKnnKeep / 64; ++e) {
                            const uint64_t m = __ballot(key[e] >= lo && key[e] < hi);
                            if (m == 0) continue;
                            const uint64_t r = m >> ((23 * step) & 63);  // any of them
                            const int l = int(__ffsll((unsigned long long)(r ? r : m))) - 1 +
                                          (r ? (23 * step) & 63 : 0);
                            p = (uint64_t(uint32_t(__builtin_amdgcn_readlane(
                                     int(uint32_t(key[e] >> 32)), l)))
                                 << 32) |
                                uint32_t(__builtin_amdgcn_readlane(int(uint32_t(key[e])), l));
                        }
                        t = p + 1 == hi ? p : p + 1;
                    } else {
                        return false;
                    }
                    C = 0;
#pragma unroll
                    for (int e = 0; e < kKnnKeep / 64; ++e) C += __popcll(__ballot(key[e] < t));
                    if (C >= k && C <= 64) break;
                    if (C < k) lo = t;
                    else hi = t;
                    v = 0.5f * (__uint_as_float(uint32_t(lo >> 32)) +
                                __uint_as_float(uint32_t(hi >> 32)));
                }
            }
            if (M > kKnnKeep) {  // denser here than over the box: t has k below it
                most = t;
                // (of up to four times the keys kept, about 256 lie below t)
                if (shrink && M > 4 * kKnnKeep) {
                    const float s = (1.75f * float(k) + 8.0f) / float(M);
                    f2 = fminf(f2, 3.0e38f) * (D == 3 ? exp2f(log2f(s) * (2.0f / 3.0f)) : s);
                    const uint64_t by_count = uint64_t(__float_as_uint(f2)) << 32;
                    lim = by_count < most ? by_count : most;
                    shrink = false;
                } else {
                    lim = most;
                }
                f2 = fminf(f2, __uint_as_float(uint32_t(lim >> 32)));
                continue;
            }
            if (M > 64) {
                wave_lds_fence();  // the keys are in registers
                int at = 0;
#pragma unroll
                for (int e = 0; e < kKnnKeep / 64; ++e) {
                    const bool hit = key[e] < t;
                    const uint64_t m = __ballot(hit);
                    if (hit) keep[at + __popcll(m & below)] = key[e];
                    at += __popcll(m);
                }
                wave_lds_fence();
                key[0] = lane < C ? keep[lane] : kMaxKey;
            }
            if (lane == 0 && (C & 1)) keep[C] = kMaxKey;  // whole pairs below
            wave_lds_fence();
            // keys are distinct: a key's rank is the number of smaller ones
            int rank = 0;
            const ulonglong2* pairs = reinterpret_cast<const ulonglong2*>(keep);
            for (int t = 0; 2 * t < C; ++t) {
                const ulonglong2 o = pairs[t];
                rank += (uint64_t(o.x) < key[0] ? 1 : 0) + (uint64_t(o.y) < key[0] ? 1 : 0);
            }
            if (lane < C && rank < k) {
                d2o[q * k + rank] = __uint_as_float(uint32_t(key[0] >> 32));
                idxo[q * k + rank] = uint32_t(key[0]);
            }
            wave_lds_fence();  // before the next query's keys
            return true;
        }
        if (!open) return false;
    }
    return false;
}

// Exact kNN, one wavefront per query at a time.
template <int D>
__global__ __launch_bounds__(256) void k_knn(const CellGrid* __restrict__ gp,
                                             const float4* __restrict__ cpts,
                                             const uint32_t* __restrict__ start,
                                             const float* __restrict__ query, int64_t n_q, int k,
                                             float* __restrict__ d2o,
                                             uint32_t* __restrict__ idxo) {
    __shared__ ulonglong2 keep[4][kKnnKeep / 2 + 1];
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    uint64_t* mine = reinterpret_cast<uint64_t*>(keep[wave]);
    const CellGrid G = *gp;
    const double inv_w = 1.0 / G.w;
    const int64_t q0 = int64_t(blockIdx.x) * kKnnBlockQueries + wave;
    for (int64_t q = q0; q < q0 + kKnnBlockQueries && q < n_q; q += 4) {
        float x[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < D; ++d) x[d] = query[q * D + d];
        if (!knn_box<D>(G, inv_w, cpts, start, x, q, k, mine, d2o, idxo))
            knn_rings<D>(G, cpts, start, x, q, k, d2o, idxo);
    }
}

// ---------------------------------------------------------------------------
// Wavefront LU with partial pivoting (Golub & Van Loan, Alg. 3.4.1).  Lane r
// holds row r of A in registers and its right-hand sides.  Rows stay in
// their lanes: the pivot row reaches the others through v_readlane (scalar
// operands of the update).  Every step works on register 0 and shifts the
// row down by one, so the steps are a loop with constant register indices;
// the loop's width drops by four columns every four steps.  A pivot row's
// entries right of its pivot are dropped by the shift one per step and kept
// in LDS, packed by column, for the back substitution.  Row swaps are
// tracked as positions, ties in |pivot| going to the smallest current
// position, as a row-swapping LU scanning downwards picks.
//
// With the rows in LDS (two reads and a write per element and lane, two
// barriers per step) and a 64-bit pivot search by shuffles the steps were
// bound by LDS latency at 13 wavefronts per CU; the pivot is now found on
// the high words by DPP, the low words only deciding between equal ones.
// Weights of 132,651 cube nodes, k = 32 (36 x 36 systems): 6.85 -> 2.66 ms.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
    const uint64_t b = uint64_t(__double_as_longlong(v));
    const uint32_t lo = __builtin_amdgcn_readlane(int(uint32_t(b)), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(int(uint32_t(b >> 32)), lane);
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}
// |v| in order as unsigned words: the high one first
__device__ __forceinline__ uint32_t abs_high(float v) { return __float_as_uint(v) & 0x7fffffffu; }
__device__ __forceinline__ uint32_t abs_low(float) { return 0; }
__device__ __forceinline__ uint32_t abs_high(double v) {
    return uint32_t(uint64_t(__double_as_longlong(v)) >> 32) & 0x7fffffffu;
}
__device__ __forceinline__ uint32_t abs_low(double v) {
    return uint32_t(uint64_t(__double_as_longlong(v)));
}

// Largest v over the wavefront (uniform).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#define NAGA_DPP_MAX(ctrl)                                                                  \
    v = max(v, uint32_t(__builtin_amdgcn_update_dpp(int(v), int(v), ctrl, 0xf, 0xf, false)))
    NAGA_DPP_MAX(0xb1);   // quad_perm [1, 0, 3, 2]
    NAGA_DPP_MAX(0x4e);   // quad_perm [2, 3, 0, 1]
    NAGA_DPP_MAX(0x141);  // row_half_mirror
    NAGA_DPP_MAX(0x140);  // row_mirror: every lane of a row holds its maximum
    NAGA_DPP_MAX(0x142);  // row_bcast15
    NAGA_DPP_MAX(0x143);  // row_bcast31: lane 63 holds the wavefront's
#undef NAGA_DPP_MAX
    return uint32_t(__builtin_amdgcn_readlane(int(v), 63));
}

// a / b given y ~ 1 / b.  Quick: y from v_rcp_f64 by two Newton steps, the
// quotient corrected by its residual (Markstein), for systems whose entries
// stay far from the ends of the exponent range; else the plain division.
template <bool QUICK>
struct Divisor {
    double b, y;
    __device__ explicit Divisor(double v) : b(v), y(0.0) {
        if (QUICK) {
            y = __builtin_amdgcn_rcp(v);
            y = fma(fma(-v, y, 1.0), y, y);
            y = fma(fma(-v, y, 1.0), y, y);
        }
    }
    __device__ double of(double a) const {
        if (!QUICK) return a / b;
        const double q = a * y;
        return fma(fma(-q, b, a), y, q);
    }
};

// LDS of one factorisation: the entries right of the diagonal, column j from
// j (j - 1) / 2.
constexpr int lu_upper(int nmax) { return nmax * (nmax - 1) / 2; }

// QUICK: entries are finite and far from the ends of the exponent range
// (quotients by reciprocals; finished rows take part in the shift with a
// zero multiplier instead of a branch).
template <int NMAX, int NR, bool QUICK, class T>
struct WaveLu {
    T (&row)[NMAX];
    T (&rhs)[NR];
    T* upper;
    const int n, lane;
    int j = 0, pos, col = 64;
    bool open;                 // not yet a pivot row
    bool singular = false;
    T own = T(0);              // this row's pivot
    double recip = 0.0;        // quick: its reciprocal

    __device__ __forceinline__ WaveLu(T (&r)[NMAX], T (&b)[NR], T* u, int n_)
        : row(r), rhs(b), upper(u), n(n_), lane(threadIdx.x & 63), pos(lane), open(lane < n_) {}

    // Steps while more than W0 - 4 columns are left, on the first W0 registers.
    template <int W0>
    __device__ __forceinline__ void steps() {
        constexpr int W = W0 < NMAX ? W0 : NMAX;
        while (n - j > W0 - 4 && j < n && !singular) {
            const uint32_t hi = abs_high(row[0]);
            const uint32_t most = wave_max_u32(open ? hi : 0u);
            uint64_t same = __ballot(open && hi == most);
            int p = int(__ffsll((unsigned long long)same)) - 1;
            if (same & (same - 1)) {  // equal high words: low words, then positions
                uint32_t plo = __builtin_amdgcn_readlane(int(abs_low(row[0])), p);
                int ppos = __builtin_amdgcn_readlane(pos, p);
                for (same &= same - 1; same; same &= same - 1) {
                    const int l = int(__ffsll((unsigned long long)same)) - 1;
                    const uint32_t llo = __builtin_amdgcn_readlane(int(abs_low(row[0])), l);
                    const int lpos = __builtin_amdgcn_readlane(pos, l);
                    if (llo > plo || (llo == plo && lpos < ppos)) {
                        p = l;
                        plo = llo;
                        ppos = lpos;
                    }
                }
            }
            p = __builtin_amdgcn_readfirstlane(p);
            const T piv = lane_value(row[0], p);
            if (!(fabs(piv) > T(0))) {
                singular = true;
                break;
            }
            const int pos_p = __builtin_amdgcn_readlane(pos, p);
            if (pos == j) pos = pos_p;
            if (col < j) upper[j * (j - 1) / 2 + col] = row[0];
            T l;
            if constexpr (sizeof(T) == 8) {
                const Divisor<QUICK> d(piv);
                l = d.of(row[0]);
                if (lane == p) recip = d.y;
            } else {
                l = row[0] / piv;
            }
            if (lane == p) {
                pos = j;
                col = j;
                own = piv;
                open = false;
            }
            if constexpr (QUICK) {
                l = open ? l : T(0);
#pragma unroll
                for (int c = 1; c < W; ++c) row[c - 1] = row[c] - l * lane_value(row[c], p);
#pragma unroll
                for (int m = 0; m < NR; ++m) rhs[m] -= l * lane_value(rhs[m], p);
            } else {
#pragma unroll
                for (int c = 1; c < W; ++c) {
                    const T pr = lane_value(row[c], p);
                    row[c - 1] = open ? row[c] - l * pr : row[c];
                }
#pragma unroll
                for (int m = 0; m < NR; ++m) {
                    const T b = lane_value(rhs[m], p);
                    rhs[m] = open ? rhs[m] - l * b : rhs[m];
                }
            }
            ++j;
        }
    }
    template <int... I>
    __device__ __forceinline__ void all_steps(std::integer_sequence<int, I...>) {
        (steps<(NMAX + 3) / 4 * 4 - 4 * I>(), ...);
    }

    // Unknown c lives in the lane whose pivot step was c.
    __device__ __forceinline__ void back() {
        const int mine = col < 64 ? col : 0;
#pragma unroll 4
        for (int c = n - 1; c >= 0; --c) {
            const T u = upper[c * (c - 1) / 2 + (mine < c ? mine : 0)];
            const int p = int(__ffsll((unsigned long long)__ballot(col == c))) - 1;
#pragma unroll
            for (int m = 0; m < NR; ++m) {
                T q;  // of the pivot lane's own values
                if constexpr (sizeof(T) == 8 && QUICK) {
                    q = rhs[m] * recip;
                    q = fma(fma(-q, own, rhs[m]), recip, q);
                } else {
                    q = rhs[m] / own;
                }
                const T x = lane_value(q, p);
                rhs[m] = col == c ? x : col < c ? rhs[m] - u * x : rhs[m];
            }
        }
    }
};

// Solves for NR right-hand sides; upper: lu_upper(NMAX) values of LDS (at
// least one).  Returns the unknown that the lane then holds in rhs[] (64:
// none), or -1 in every lane for a zero pivot.
template <int NMAX, int NR, bool QUICK, class T>
__device__ __forceinline__ int wave_lu_solve(T (&row)[NMAX], T (&rhs)[NR], T* upper, int n) {
    WaveLu<NMAX, NR, QUICK, T> w(row, rhs, upper, __builtin_amdgcn_readfirstlane(n));
    w.all_steps(std::make_integer_sequence<int, (NMAX + 3) / 4>());
    if (w.singular) return -1;
    __syncthreads();  // the entries kept in LDS
    w.back();
    return w.col;
}

// unscaled quadrature points, [0]: 2D (16 used), [1]: 3D (64); both
// tables are written once per device and never change afterwards, so
// scenes of either dimension can be set up concurrently
__constant__ double c_quad_unit[2][64][3];
__constant__ double c_quad_rw[4];        // radial Gauss weights

__device__ __forceinline__ double dist2_f64(int D, const double* a, const double* b) {
    double s = (a[0] - b[0]) * (a[0] - b[0]);
    for (int d = 1; d < D; ++d) s = (a[d] - b[d]) * (a[d] - b[d]) + s;
    return s;
}

// Square root of x = 0 or 2^-700 < x < 2^700 (squared distances of FP32
// points): v_rsq_f64 refined by one Goldschmidt step and the residual of the
// result; without the scaling a full-range square root needs.
__device__ __forceinline__ double sqrt_mid(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, x), h, g);
    return x > 0.0 ? g : 0.0;
}

__device__ __forceinline__ double rbf_eval(int rbf, double r2, double spacing) {
    if (rbf == 1) return r2 * sqrt_mid(r2);
    const double c = spacing * 0.1;
    return sqrt_mid(r2 + c * c);
}

// Row `lane` of the augmented RBF matrix [[Phi, P], [P^T, 0]] in raw
// coordinates (interpolation/detail/radial_point_method.cuh:349-398), zeros
// past its n = k + D + 1 columns.
template <int NMAX, int D, class T>
__device__ __forceinline__ void g0_row(const double (*xs)[4], int k, int rbf, double spacing,
                                       T (&row)[NMAX]) {
    const int lane = threadIdx.x & 63;
    const int n = k + D + 1;
    const int axis = lane > k && lane < n ? lane - k - 1 : 0;
    double mine[D];
#pragma unroll
    for (int d = 0; d < D; ++d) mine[d] = xs[lane][d];
#pragma unroll
    for (int c = 0; c < NMAX; ++c) {
        double v = 0.0;
        if (c < k) {
            double o[D];
#pragma unroll
            for (int d = 0; d < D; ++d) o[d] = xs[c][d];
            v = rbf_eval(rbf, dist2_f64(D, mine, o), spacing);
            v = lane < k ? v : lane == k ? 1.0 : xs[c][axis];
        } else if (c == k) {
            v = lane < k ? 1.0 : 0.0;
        } else if (c < n) {
            v = lane < k ? xs[lane][c - k - 1] : 0.0;
        }
        row[c] = lane < n ? T(v) : T(0);
    }
}

// entry `lane` of G_x (:400-433)
template <int D>
__device__ __forceinline__ double gx_entry(const double (*xs)[4], const double* mine, int k,
                                           int rbf, double spacing, const double* xq) {
    const int lane = threadIdx.x & 63;
    double v = rbf_eval(rbf, dist2_f64(D, mine, xq), spacing);
#pragma unroll
    for (int d = 0; d < D; ++d) v = lane == k + 1 + d ? xq[d] : v;
    return lane == k ? 1.0 : v;
}

// antisymmetric w4 B-spline kernel times the quadrature weight
// (nonlocal_calculus/detail/divergence.inl:55-133, :167-201)
__device__ void quad_term(int D, double delta, const double* xi, const double* xq,
                          int q, double* aw) {
    double dx[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < D; ++d) dx[d] = xq[d] - xi[d];
    const double rxy = sqrt(dx[1] * dx[1] + dx[0] * dx[0]);
    const double r = D == 3 ? sqrt(dx[2] * dx[2] + (dx[1] * dx[1] + dx[0] * dx[0])) : rxy;
    double g;
    if (2.0 * r / delta < 1.0)
        g = r * (2.0 * delta - 3.0 * r);
    else if (2.0 * r / delta < 2.0)
        g = (delta - r) * (delta - r);
    else
        g = 0.0;
    double qw = c_quad_rw[q % 4] * delta / 2.0;
    qw *= 2.0 * M_PI / 4.0;
    if (D == 3) qw *= M_PI / 4.0;
    if (D == 2) {
        const double C = (240.0 / 7.0) / (M_PI * pow(delta, 5.0));
        qw *= r;
        aw[0] = C * g * (dx[0] / r) * qw;
        aw[1] = C * g * (dx[1] / r) * qw;
    } else {
        const double C = 48.0 / (M_PI * pow(delta, 6.0));
        const double sp = rxy / r, cp = dx[2] / r;
        const double ct = rxy != 0.0 ? dx[0] / rxy : 0.0;
        const double st = rxy != 0.0 ? dx[1] / rxy : 0.0;
        qw *= r * rxy;
        aw[0] = C * g * sp * ct * qw;
        aw[1] = C * g * sp * st * qw;
        aw[2] = C * g * cp * qw;
    }
}

// One wavefront per query node: assemble G0, the D quadrature right-hand
// sides b_d = sum_q alpha_d(q) w(q) G_x(q), solve G0 y_d = b_d in FP64 and
// write W(d, s) = y_d[s] (+ sum_q alpha_d w for s = 0).  By linearity this
// equals the reference's per-quadrature-point RPIM weights summed against
// the kernel (detail/divergence.inl:203-215) with D solves instead of Nq.
// Lane q forms quadrature point q and its kernel weights once; the points
// then reach every lane (a row of the system each) as broadcast LDS reads.
template <int NMAX, int D, class T>
__global__ __launch_bounds__(64) void k_divw(const float* __restrict__ src,
                                             const float* __restrict__ query, int64_t n_q,
                                             const uint32_t* __restrict__ idx,
                                             const float* __restrict__ d2, int kmax, int rbf,
                                             const double* __restrict__ hbar,
                                             const uint8_t* __restrict__ kvar,
                                             float* __restrict__ W, double* __restrict__ W64,
                                             int* __restrict__ info) {
    constexpr int Nq = D == 2 ? 16 : 64;
    __shared__ double xs[64][4];
    // quadrature points and their kernel weights, then the factorisation
    constexpr size_t kQuad = sizeof(double) * Nq * 2 * D, kUpper = sizeof(T) * lu_upper(NMAX);
    __shared__ double pool[((kQuad > kUpper ? kQuad : kUpper) + 7) / 8];
    double(*quad)[2 * D] = reinterpret_cast<double(*)[2 * D]>(pool);
    const int lane = threadIdx.x;
    const int64_t i = blockIdx.x;
    if (i >= n_q) return;
    // per-node stencil width k <= kmax (entries past k get zero weights)
    const int k = kvar ? int(kvar[i]) : kmax;
    const int n = k + D + 1;
    if (lane >= k && lane < kmax)
        for (int d = 0; d < D; ++d) {
            W[(i * kmax + lane) * D + d] = 0.0f;
            if (W64) W64[(i * kmax + lane) * D + d] = 0.0;
        }
    double mine[3] = {0.0, 0.0, 0.0};
    if (lane < k) {
        const int64_t j = idx[i * kmax + lane];
        for (int d = 0; d < D; ++d) mine[d] = double(src[j * D + d]);
    }
    for (int d = 0; d < D; ++d) xs[lane][d] = mine[d];
    double xi[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < D; ++d) xi[d] = double(query[i * D + d]);
    const double delta = 0.05 * sqrt(double(d2[i * kmax + 1]));
    const double spacing = hbar[i / 16384];
    if (lane < Nq) {
        double xq[3] = {0.0, 0.0, 0.0}, aw[3];
        for (int d = 0; d < D; ++d) xq[d] = c_quad_unit[D - 2][lane][d] * delta + xi[d];
        quad_term(D, delta, xi, xq, lane, aw);
        for (int d = 0; d < D; ++d) {
            quad[lane][d] = xq[d];
            quad[lane][D + d] = aw[d];
        }
    }
    __syncthreads();
    double b64[D], S[D];
    for (int d = 0; d < D; ++d) b64[d] = S[d] = 0.0;
#pragma unroll 4
    for (int q = 0; q < Nq; ++q) {
        const double gx = gx_entry<D>(xs, mine, k, rbf, spacing, quad[q]);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            b64[d] += quad[q][D + d] * gx;
            S[d] += quad[q][D + d];
        }
    }
    T b[D], row[NMAX];
    for (int d = 0; d < D; ++d) b[d] = T(b64[d]);
    g0_row<NMAX, D>(xs, k, rbf, spacing, row);
    __syncthreads();  // every lane is done with the quadrature points
    const int col = wave_lu_solve<NMAX, D, true, T>(row, b, reinterpret_cast<T*>(pool), n);
    if (lane == 0) info[i] = col < 0 ? 1 : 0;
    if (col < 0 || col >= k) return;
    for (int d = 0; d < D; ++d) {
        const double v = double(b[d]) + (col == 0 ? S[d] : 0.0);
        W[(i * kmax + col) * D + d] = float(v);
        if (W64) W64[(i * kmax + col) * D + d] = v;
    }
}

template <int NMAX, int D, class T>
__global__ __launch_bounds__(64) void k_rpim(const float* __restrict__ src,
                                             const float* __restrict__ query, int64_t n_q,
                                             const uint32_t* __restrict__ idx, int k, int rbf,
                                             double spacing, float* __restrict__ w,
                                             double* __restrict__ w64, int* __restrict__ info,
                                             int group) {
    __shared__ double xs[64][4];
    const int lane = threadIdx.x;
    const int64_t i = blockIdx.x;
    if (i >= n_q) return;
    double mine[3] = {0.0, 0.0, 0.0};
    if (lane < k) {  // the queries of a group share their group's stencil
        const int64_t j = idx[(i / group) * k + lane];
        for (int d = 0; d < D; ++d) mine[d] = double(src[j * D + d]);
    }
    for (int d = 0; d < D; ++d) xs[lane][d] = mine[d];
    __syncthreads();
    double xq[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < D; ++d) xq[d] = double(query[i * D + d]);
    __shared__ T upper[lu_upper(NMAX)];
    T row[NMAX];
    g0_row<NMAX, D>(xs, k, rbf, spacing, row);
    T b[1] = {T(gx_entry<D>(xs, mine, k, rbf, spacing, xq))};
    const int col = wave_lu_solve<NMAX, 1, true, T>(row, b, upper, k + D + 1);
    if (lane == 0) info[i] = col < 0 ? 1 : 0;
    if (col < 0 || col >= k) return;
    w[i * k + col] = float(b[0]);
    if (w64) w64[i * k + col] = double(b[0]);
}

template <int NMAX>
__global__ __launch_bounds__(64) void k_batched_lu(int n, int nrhs, int64_t batch,
                                                   double* A, double* B, int* info) {
    const int lane = threadIdx.x;
    const int64_t b = blockIdx.x;
    if (b >= batch) return;
    const double* Ab = A + b * int64_t(n) * n;
    double* Bb = B + b * int64_t(n) * nrhs;
    __shared__ double upper[lu_upper(NMAX)];
    // right-hand sides are processed four at a time, each group against a
    // fresh copy of the matrix
    for (int m0 = 0; m0 < nrhs; m0 += 4) {
        double row[NMAX], rhs[4];
#pragma unroll
        for (int c = 0; c < NMAX; ++c)
            row[c] = (lane < n && c < n) ? Ab[lane + int64_t(c) * n] : 0.0;
#pragma unroll
        for (int m = 0; m < 4; ++m)
            rhs[m] = (lane < n && m0 + m < nrhs) ? Bb[lane + int64_t(m0 + m) * n] : 0.0;
        const int col = wave_lu_solve<NMAX, 4, false, double>(row, rhs, upper, n);
        if (col < 0) {
            if (lane == 0) info[b] = 1;
            return;
        }
        if (col < n)
#pragma unroll
            for (int m = 0; m < 4; ++m)
                if (m0 + m < nrhs) Bb[col + int64_t(m0 + m) * n] = rhs[m];
        __syncthreads();  // before the next group's factorisation
    }
    if (lane == 0) info[b] = 0;
}

__global__ void k_filter(int D, const float* pts, int64_t n, const uint32_t* idx,
                         int kmax, double sg, const uint8_t* kvar, float* wf) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int k = kvar ? int(kvar[i]) : kmax;
    double xi[3] = {0.0, 0.0, 0.0};
    for (int d = 0; d < D; ++d) xi[d] = double(pts[i * D + d]);
    double sum = 0.0;
    for (int s = 0; s < k; ++s) {
        double xj[3] = {0.0, 0.0, 0.0};
        const int64_t j = idx[i * kmax + s];
        for (int d = 0; d < D; ++d) xj[d] = double(pts[j * D + d]);
        const double r = sqrt(dist2_f64(D, xi, xj)) / sg;
        sum += exp(-0.5 * r * r);
    }
    for (int s = 0; s < kmax; ++s) {
        double wv = 0.0;
        if (s < k) {
            double xj[3] = {0.0, 0.0, 0.0};
            const int64_t j = idx[i * kmax + s];
            for (int d = 0; d < D; ++d) xj[d] = double(pts[j * D + d]);
            const double r = sqrt(dist2_f64(D, xi, xj)) / sg;
            wv = exp(-0.5 * r * r) / sum;
        }
        wf[i * kmax + s] = float(wv);
    }
}

__global__ void k_pad_entries(int64_t n, int k, int ks, int nc, const uint32_t* idx,
                              const float* w, uint32_t* idx_out, float* w_out) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n * ks) return;
    const int64_t i = e / ks;
    const int s = int(e - i * ks);
    idx_out[e] = idx[i * k + (s < k ? s : 0)];
    for (int c = 0; c < nc; ++c) w_out[e * nc + c] = s < k ? w[(i * k + s) * nc + c] : 0.0f;
}

__global__ void k_make_slab(int64_t n, int k, int nc, const uint32_t* idx,
                            const float* w, float* slab) {
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n * k) return;
    float* r = slab + t * (1 + nc);
    r[0] = __uint_as_float(idx[t]);
    for (int c = 0; c < nc; ++c) r[1 + c] = w[t * nc + c];
}

// One thread per (node, 32-bit word) of the D2Q9 records.
__global__ void k_make_slab_q9(int64_t n, int k, int nc, const uint32_t* idx, const float* w,
                               uint32_t* slab) {
    const int words = 4 * q9_units(k, nc);
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n * words) return;
    const int64_t i = t / words;
    const int u = int(t - i * words) / 4, f = u % (1 + nc);  // field: index, weights
    const int s = u / (1 + nc) * 4 + int(t % 4);             // record (words is a multiple of 4)
    uint32_t v = 0u;
    if (f == 0) v = idx[i * k + (s < k ? s : 0)];
    else if (s < k) v = __float_as_uint(w[(i * k + s) * nc + f - 1]);
    slab[t] = v;
}

// One thread per (node, 32-bit word) of the packed divergence records.
__global__ void k_pack_div_records(int64_t n, int k, const float* src, uint32_t* dst) {
    const int units = packed_div_units(k);
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n * units * 4) return;
    const int64_t i = t / (int64_t(units) * 4);
    const int word = int(t - i * units * 4);
    const int u = word / 4, g = u / 7, w = u % 7;
    const float* rec = src + (i * k + 8 * g) * 4;  // the group's 8 records
    uint32_t v = 0;
    if (u >= 7 * (k / 8)) {
        v = 0;  // padding units
    } else if (w < 6) {
        const int f = 4 * w + word % 4;  // float f of the group's 24 weights
        v = __float_as_uint(rec[(f / 3) * 4 + 1 + f % 3]);
    } else {
        const int m = word % 4;  // records 2m, 2m + 1
        const uint32_t lo = __float_as_uint(rec[(2 * m) * 4]);
        const uint32_t hi = __float_as_uint(rec[(2 * m + 1) * 4]);
        v = (lo & 0xffffu) | (hi << 16);
    }
    dst[t] = v;
}

// One thread per (node, 32-bit word) of the packed filter records.
__global__ void k_pack_filter_records(int64_t n, int k, const float* src, uint32_t* dst) {
    const int units = packed_filter_units(k);
    const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n * units * 4) return;
    const int64_t i = t / (int64_t(units) * 4);
    const int word = int(t - i * units * 4);
    const int u = word / 4, g = u / 3, w = u % 3;
    const float* rec = src + (i * k + 8 * g) * 2;  // the group's 8 {position, weight}
    uint32_t v = 0;
    if (u >= 3 * (k / 8)) {
        v = 0;  // padding units
    } else if (w < 2) {
        v = __float_as_uint(rec[(4 * w + word % 4) * 2 + 1]);
    } else {
        const int m = word % 4;  // records 2m, 2m + 1
        const uint32_t lo = __float_as_uint(rec[(2 * m) * 2]);
        const uint32_t hi = __float_as_uint(rec[(2 * m + 1) * 2]);
        v = (lo & 0xffffu) | (hi << 16);
    }
    dst[t] = v;
}

// One block per tile: the tile's k * tile_nodes (<= 4096) neighbour indices
// are sorted in LDS (bitonic), flagged where they differ from their
// predecessor and compacted by a block-wide scan of the flags.
constexpr int kUnionMax = 4096;

__device__ __forceinline__ int block_exclusive_scan(int* v, int n, int* tmp) {
    // v[0..n) in LDS, n <= kUnionMax, blockDim.x == 256: per-thread chunks of
    // n / 256 (n is a power of two >= 256 here), then a scan of the chunk sums.
    const int per = n / 256, t = threadIdx.x;
    int sum = 0;
    for (int e = 0; e < per; ++e) sum += v[t * per + e];
    tmp[t] = sum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const int add = t >= off ? tmp[t - off] : 0;
        __syncthreads();
        tmp[t] += add;
        __syncthreads();
    }
    int run = tmp[t] - sum;  // exclusive prefix of this chunk
    for (int e = 0; e < per; ++e) {
        const int f = v[t * per + e];
        v[t * per + e] = run;
        run += f;
    }
    __syncthreads();
    const int total = tmp[255];
    __syncthreads();
    return total;
}

// Sorted distinct keys of src[0..M) (M <= kUnionMax) into uniq[0..U) by
// the whole block; returns U.
__device__ int block_union(const uint32_t* src, int M, uint32_t* keys, uint32_t* uniq,
                           int* rank, int* tmp) {
    int P = 256;
    while (P < M) P <<= 1;
    for (int e = threadIdx.x; e < P; e += 256) keys[e] = e < M ? src[e] : 0xffffffffu;
    __syncthreads();
    for (int size = 2; size <= P; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int e = threadIdx.x; e < P / 2; e += 256) {
                const int i = 2 * stride * (e / stride) + (e % stride), j = i + stride;
                const bool up = (i & size) == 0;
                const uint32_t a = keys[i], b = keys[j];
                if ((a > b) == up) {
                    keys[i] = b;
                    keys[j] = a;
                }
            }
            __syncthreads();
        }
    for (int e = threadIdx.x; e < P; e += 256)
        rank[e] = (e < M && (e == 0 || keys[e] != keys[e - 1])) ? 1 : 0;
    __syncthreads();
    const int U = block_exclusive_scan(rank, P, tmp);
    // compact the distinct keys (rank is the exclusive scan of the flags)
    for (int e = threadIdx.x; e < M; e += 256)
        if (e == 0 || keys[e] != keys[e - 1]) uniq[rank[e]] = keys[e];
    __syncthreads();
    return U;
}

// Writes uniq[0..U) to out and, for the M stencil entries src[0..M), the
// entry's position in uniq into the index field of the slab records.
__device__ void write_union(const uint32_t* src, int M, const uint32_t* uniq, int U,
                            uint32_t* out, float* slab_a, int nca, float* slab_b, int ncb) {
    for (int e = threadIdx.x; e < U; e += 256) out[e] = uniq[e];
    for (int r = threadIdx.x; r < M; r += 256) {
        const uint32_t j = src[r];
        int lo = 0, hi = U;  // first position with uniq[pos] >= j
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (uniq[mid] < j) lo = mid + 1;
            else hi = mid;
        }
        const float slot = __uint_as_float(uint32_t(lo));
        slab_a[r * (1 + nca)] = slot;
        if (slab_b) slab_b[r * (1 + ncb)] = slot;
    }
    __syncthreads();
}

// One block per tile: the tile's k * tile_nodes (<= 4096) neighbour indices
// are sorted in LDS (bitonic), flagged where they differ from their
// predecessor and compacted by a block-wide scan of the flags.  A tile
// whose union exceeds cap (> 0) while each half-tile's union fits is
// split: its list is the first half's union followed by the second
// half's, each half's records hold positions in its own part, and
// usplit[t] is the first part's length (0 for tiles not split).
// Counting pass (ulist == nullptr): counts[t] = list length, usplit[t].
__global__ __launch_bounds__(256) void k_tile_union(int64_t nfluid, int k, int tile_nodes,
                                                    const uint32_t* idx, int cap,
                                                    int32_t* counts, int32_t* usplit,
                                                    const int64_t* uoff,
                                                    uint32_t* ulist, float* slab_a, int nca,
                                                    float* slab_b, int ncb) {
    __shared__ uint32_t keys[kUnionMax];
    __shared__ uint32_t uniq[kUnionMax];
    __shared__ int rank[kUnionMax];
    __shared__ int tmp[256];
    const int64_t node0 = int64_t(blockIdx.x) * tile_nodes;
    const int64_t left = nfluid - node0;
    const int cnt = left < tile_nodes ? int(left) : tile_nodes;
    const int M = cnt * k;
    const int h = tile_nodes / 2;  // nodes of the first half
    const uint32_t* src = idx + node0 * k;
    if (!ulist) {
        const int U = block_union(src, M, keys, uniq, rank, tmp);
        int total = U, first = 0;
        if (cap > 0 && U > cap && cnt > h) {
            const int UA = block_union(src, h * k, keys, uniq, rank, tmp);
            const int UB = block_union(src + h * k, (cnt - h) * k, keys, uniq, rank, tmp);
            if (UA <= cap && UB <= cap) {
                total = UA + UB;
                first = UA;
            }
        }
        if (threadIdx.x == 0) {
            counts[blockIdx.x] = total;
            if (usplit) usplit[blockIdx.x] = first;
        }
        return;
    }
    uint32_t* out = ulist + uoff[blockIdx.x];
    float* sa = slab_a + node0 * k * (1 + nca);
    float* sb = slab_b ? slab_b + node0 * k * (1 + ncb) : nullptr;
    const int first = usplit ? usplit[blockIdx.x] : 0;
    if (first == 0) {
        const int U = block_union(src, M, keys, uniq, rank, tmp);
        write_union(src, M, uniq, U, out, sa, nca, sb, ncb);
        return;
    }
    const int UA = block_union(src, h * k, keys, uniq, rank, tmp);
    write_union(src, h * k, uniq, UA, out, sa, nca, sb, ncb);
    const int MB = (cnt - h) * k;
    const int UB = block_union(src + h * k, MB, keys, uniq, rank, tmp);
    write_union(src + h * k, MB, uniq, UB, out + UA, sa + int64_t(h) * k * (1 + nca), nca,
                sb ? sb + int64_t(h) * k * (1 + ncb) : nullptr, ncb);
}

// Ragged record rows: node i of tile t = i / T keeps the first upg *
// ng[t] units of its full row (KP units) and pads to `ragged(ng[t])` units
// with zeros; tile t's rows start at unit off[t].
__global__ void k_ragged_records(int64_t n, int T, int KP, int upg, const int32_t* ng,
                                 const int64_t* off, const float4* src, float4* dst) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n * KP) return;
    const int64_t i = e / KP;
    const int u = int(e - i * KP);
    const int64_t t = i / T;
    const int g = ng[t];
    const int kpt = upg == 7 ? ragged_div_units(g) : ragged_filter_units(g);
    if (u >= kpt) return;
    dst[off[t] + (i - t * T) * kpt + u] = u < upg * g ? src[e] : make_float4(0.f, 0.f, 0.f, 0.f);
}

// flag stays 1 if idx[i * k] == i for every i < n, else becomes 0.
__global__ void k_self_first(int64_t n, int k, const uint32_t* idx, int* flag) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n && idx[i * k] != uint32_t(i)) atomicAnd(flag, 0);
}

// Stencil entries s >= kvar[i] (zero weights) of node i point at i itself.
__global__ void k_self_past_k(int64_t n, int k, const uint8_t* kvar, uint32_t* idx) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n * k) return;
    const int64_t i = e / k;
    if (int(e - i * k) >= int(kvar[i])) idx[e] = uint32_t(i);
}

// out[e] = idx[e] if it is in [lo, hi), else zero_row.
__global__ void k_layer_only(int64_t n, const uint32_t* idx, uint32_t lo, uint32_t hi,
                             uint32_t zero_row, uint32_t* out) {
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const uint32_t j = idx[e];
    out[e] = (j >= lo && j < hi) ? j : zero_row;
}

__global__ void k_flag(int64_t n, int k, const uint32_t* idx, int64_t lo,
                       int64_t hi, uint8_t* flag) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint8_t f = 0;
    for (int s = 0; s < k; ++s) {
        const int64_t j = idx[i * k + s];
        f |= (j >= lo && j < hi) ? 1 : 0;
    }
    flag[i] = f;
}

__global__ void k_div_apply(int D, int64_t n, int k, const uint32_t* idx,
                            const float* W, const float* F, float off, float* out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float acc = 0.0f;
    for (int s = 0; s < k; ++s) {
        const int64_t j = idx[i * k + s];
        float v = 0.0f;
        for (int d = 0; d < D; ++d) v += W[(i * k + s) * D + d] * (F[j * D + d] - off);
        acc += v;
    }
    out[i] = acc;
}

// ---------------------------------------------------------------------------
// Cell binning on the device (segmentation/detail/nd_cubic_segmentation.inl:
// 38-273: bounds, partition sizes, offsets by a scan, indices by a scatter).
// The order of indices within a cell follows the scatter's atomics, as in
// the reference; the kNN over the cells is exact whatever that order.
// ---------------------------------------------------------------------------
// Per-block bounds of the points (grid-stride), partial[b][0..3) minima and
// [3..6) maxima.
// Per-block bounds of the points; zeroes the M cell counts.
__global__ __launch_bounds__(256) void k_bounds(const float* pts, int64_t n, int D,
                                                double* partial, uint32_t* counts, int64_t M) {
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < M; i += int64_t(gridDim.x) * 256)
        counts[i] = 0u;
    __shared__ float lo[3][256], hi[3][256];
    float l[3] = {3.0e38f, 3.0e38f, 3.0e38f}, h[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
    for (int64_t j = int64_t(blockIdx.x) * 256 + threadIdx.x; j < n;
         j += int64_t(gridDim.x) * 256)
        for (int d = 0; d < D; ++d) {
            const float v = pts[j * D + d];
            l[d] = fminf(l[d], v);
            h[d] = fmaxf(h[d], v);
        }
    for (int d = 0; d < 3; ++d) {
        lo[d][threadIdx.x] = l[d];
        hi[d][threadIdx.x] = h[d];
    }
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int d = 0; d < 3; ++d) {
                lo[d][threadIdx.x] = fminf(lo[d][threadIdx.x], lo[d][threadIdx.x + w]);
                hi[d][threadIdx.x] = fmaxf(hi[d][threadIdx.x], hi[d][threadIdx.x + w]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 3) {
        partial[blockIdx.x * 6 + threadIdx.x] = double(lo[threadIdx.x][0]);
        partial[blockIdx.x * 6 + 3 + threadIdx.x] = double(hi[threadIdx.x][0]);
    }
}

// Cells of width w over the grid's extents, w grown until they fit the capacity.
__device__ void size_grid(CellGrid& G, double w, int64_t cap) {
    int64_t nc = 1;
    for (int it = 0; it < 4096; ++it) {
        nc = 1;
        for (int d = 0; d < 3; ++d) {
            double m = d < G.D ? ceil(G.ext[d] / w) : 1.0;
            m = m < 1.0 ? 1.0 : (m > 1048576.0 ? 1048576.0 : m);
            G.dims[d] = int64_t(m);
            nc *= G.dims[d];
        }
        if (nc <= cap) break;
        w *= 1.25;
    }
    if (nc > cap) {  // unreachable for finite input: one cell then
        G.dims[0] = G.dims[1] = G.dims[2] = 1;
        nc = 1;
        w = 1e300;
    }
    G.w = w;
    G.ncell = nc;
}

// The grid from the per-block bounds (nd_cubic_segmentation.cuh:241-279).
__global__ __launch_bounds__(256) void k_grid(const double* partial, int D, int64_t n,
                                              double per_cell, double width, int64_t cap,
                                              CellGrid* g) {
    __shared__ double lo[3][kBoundBlocks], hi[3][kBoundBlocks];
    const int t = threadIdx.x;
    for (int d = 0; d < 3; ++d) {
        lo[d][t] = partial[t * 6 + d];
        hi[d][t] = partial[t * 6 + 3 + d];
    }
    __syncthreads();
    for (int w = kBoundBlocks / 2; w > 0; w >>= 1) {
        if (t < w)
            for (int d = 0; d < 3; ++d) {
                lo[d][t] = fmin(lo[d][t], lo[d][t + w]);
                hi[d][t] = fmax(hi[d][t], hi[d][t + w]);
            }
        __syncthreads();
    }
    if (t != 0) return;
    CellGrid G{};
    G.D = D;
    double vol = 1.0;
    for (int d = 0; d < 3; ++d) {
        G.lo[d] = d < D ? lo[d][0] : 0.0;
        G.ext[d] = 1.0;
        if (d < D) {
            G.ext[d] = hi[d][0] - lo[d][0];
            if (G.ext[d] < 1e-3) G.ext[d] = 1e-3;  // the reference's tolerance
            vol *= G.ext[d];
        }
    }
    size_grid(G, width > 0.0 ? width : pow(per_cell * vol / double(n), 1.0 / double(D)), cap);
    *g = G;
}

// Cell of a point: floor((x - lo) / w) per axis, clamped to the grid;
// linear index with x fastest (the kNN's cell rows).
__device__ __forceinline__ int64_t cell_of(const CellGrid& G, const float* p) {
    int64_t c = 0, mul = 1;
#pragma unroll  // (indexed at run time the grid would be copied to scratch memory)
    for (int d = 0; d < 3; ++d)
        if (d < G.D) {
            int64_t ci = int64_t(floor((double(p[d]) - G.lo[d]) / G.w));
            ci = ci < 0 ? 0 : ci >= G.dims[d] ? G.dims[d] - 1 : ci;
            c += ci * mul;
            mul *= G.dims[d];
        }
    return c;
}

__global__ __launch_bounds__(256) void k_count_cells(const float* pts, int64_t n,
                                                     const CellGrid* gp, uint32_t* counts) {
    const int64_t j = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (j >= n) return;
    const CellGrid G = *gp;
    atomicAdd(&counts[cell_of(G, pts + j * G.D)], 1u);
}

// Exclusive scan of in[0..M) into out, block b covering [b * 2048, ..); its
// total goes to bsum[b] and, with pairs, the sum of in (in - 1) / 2 to
// pairs[b].  in is left zero.
__device__ __forceinline__ uint32_t block_scan_256(uint32_t v, uint32_t* tmp, uint32_t& total) {
    const int t = threadIdx.x;
    tmp[t] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const uint32_t a = t >= off ? tmp[t - off] : 0u;
        __syncthreads();
        tmp[t] += a;
        __syncthreads();
    }
    total = tmp[255];
    const uint32_t incl = tmp[t];
    __syncthreads();
    return incl - v;
}

// Sum over the block's 256 threads, in every thread.
__device__ __forceinline__ uint64_t block_sum_256(uint64_t v, uint64_t* tmp) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += shfl_xor64(v, o);
    if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
    __syncthreads();
    return tmp[0] + tmp[1] + tmp[2] + tmp[3];
}

__device__ __forceinline__ void scan_chunk(uint32_t* in, int64_t M, uint32_t* out, uint32_t* bsum,
                                           uint64_t* pairs) {
    __shared__ uint32_t tmp[256];
    __shared__ uint64_t ptmp[4];
    const int64_t base = int64_t(blockIdx.x) * kScanChunk + threadIdx.x * 8;
    uint32_t v[8], s = 0;
    uint64_t mates = 0;
    for (int e = 0; e < 8; ++e) {
        v[e] = base + e < M ? in[base + e] : 0u;
        s += v[e];
        if (v[e]) mates += uint64_t(v[e]) * (v[e] - 1) / 2;
    }
    uint32_t total;
    uint32_t run = block_scan_256(s, tmp, total);
    for (int e = 0; e < 8; ++e) {
        if (base + e < M) {
            out[base + e] = run;
            if (v[e]) in[base + e] = 0u;
        }
        run += v[e];
    }
    if (pairs) mates = block_sum_256(mates, ptmp);
    if (threadIdx.x == 0) {
        bsum[blockIdx.x] = total;
        if (pairs) pairs[blockIdx.x] = mates;
    }
}

__global__ __launch_bounds__(256) void k_scan_local(uint32_t* in, int64_t M, uint32_t* out,
                                                    uint32_t* bsum, uint64_t* pairs) {
    scan_chunk(in, M, out, bsum, pairs);
}

// Whether the cloud is crowded (a point has on average more than kCrowded
// times per_cell others in its cell), and its grid of narrower cells then.
// The cells sized for k points are best for evenly spread clouds (2 points per
// cell, k = 32: 1M random points take 3.8 ms instead of 1.7 in 3D, 1.7 instead
// of 1.0 in 2D), but where they hold many times that each query visits
// hundreds of points too many: 200,000 points on a circle, k = 32, 1.08 ms
// against 0.43.  Between the two, gains of two and losses of a fifth lie at 6
// to 9 times the points per cell.  Every block decides by itself, from the
// same sums; the narrow grid takes the other's place in k_scan_sums.
struct Crowding {
    const uint64_t* pairs;  // null: never
    int64_t nblocks, n, cap;
    double per_cell, narrow;
};
__device__ __forceinline__ bool is_crowded(const Crowding& c) {
    __shared__ uint64_t tmp[4];
    if (!c.pairs) return false;
    uint64_t mates = 0;
    for (int64_t i = threadIdx.x; i < c.nblocks; i += 256) mates += c.pairs[i];
    mates = block_sum_256(mates, tmp);
    return 2.0 * double(mates) > kCrowded * c.per_cell * double(c.n);
}
__device__ CellGrid narrow_grid(const Crowding& c, CellGrid G) {
    double vol = 1.0;
    for (int d = 0; d < G.D; ++d) vol *= G.ext[d];
    size_grid(G, pow(c.narrow * vol / double(c.n), 1.0 / double(G.D)), c.cap);
    return G;
}

__global__ __launch_bounds__(256) void k_recount_cells(const float* pts, const CellGrid* g,
                                                       Crowding c, uint32_t* counts) {
    __shared__ CellGrid G;
    if (!is_crowded(c)) return;
    if (threadIdx.x == 0) G = narrow_grid(c, *g);
    __syncthreads();
    for (int64_t j = int64_t(blockIdx.x) * 256 + threadIdx.x; j < c.n;
         j += int64_t(gridDim.x) * 256)
        atomicAdd(&counts[cell_of(G, pts + j * G.D)], 1u);
}

__global__ __launch_bounds__(256) void k_rescan_local(Crowding c, uint32_t* in, int64_t M,
                                                      uint32_t* out, uint32_t* bsum) {
    if (is_crowded(c)) scan_chunk(in, M, out, bsum, nullptr);
}

__global__ __launch_bounds__(256) void k_scan_sums(uint32_t* bsum, int64_t nb, CellGrid* g,
                                                   Crowding c) {
    __shared__ uint32_t tmp[256];
    if (is_crowded(c) && threadIdx.x == 0) *g = narrow_grid(c, *g);
    uint32_t carry = 0;
    for (int64_t c0 = 0; c0 < nb; c0 += 256) {
        const int64_t i = c0 + threadIdx.x;
        const uint32_t v = i < nb ? bsum[i] : 0u;
        uint32_t total;
        const uint32_t ex = block_scan_256(v, tmp, total);
        if (i < nb) bsum[i] = carry + ex;
        carry += total;
    }
}

__global__ __launch_bounds__(256) void k_scan_add(uint32_t* out, int64_t M, const uint32_t* bsum) {
    const int64_t base = int64_t(blockIdx.x) * kScanChunk;
    const uint32_t add = bsum[blockIdx.x];
    for (int e = threadIdx.x; e < kScanChunk; e += 256)
        if (base + e < M) out[base + e] += add;
}

__global__ __launch_bounds__(256) void k_scatter_cells(const float* pts, int64_t n,
                                                       const CellGrid* gp, const uint32_t* start,
                                                       uint32_t* fill, uint32_t* sorted,
                                                       float4* cpts) {
    const int64_t j = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (j >= n) return;
    const CellGrid G = *gp;
    float p[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (d < G.D) p[d] = pts[j * G.D + d];
    const int64_t c = cell_of(G, p);
    const uint32_t at = start[c] + atomicAdd(&fill[c], 1u);
    sorted[at] = uint32_t(j);
    cpts[at] = make_float4(p[0], p[1], p[2], __uint_as_float(uint32_t(j)));
}

int pick_nmax(int n) {
    const int opts[] = {20, 28, 36, 44, 52, 64};
    for (int o : opts)
        if (n <= o) return o;
    return -1;
}

void fill_quadrature(int D, double (&tab)[64][3]) {
    static const double xr[4] = {0.339981, -0.339981, 0.861136, -0.861136};
    const int Nq = D == 2 ? 16 : 64;
    for (int q = 0; q < 64; ++q)
        for (int d = 0; d < 3; ++d) tab[q][d] = 0.0;
    for (int q = 0; q < Nq; ++q) {
        // nonlocal_calculus/detail/quadrature_points.cuh:74-91, :127-152
        const double r = (xr[q % 4] + 1.0) / 2.0;
        const double ts = 3.0 * M_PI / 2.0 / 3.0;
        if (D == 2) {
            const double th = (q / 4) * ts;
            tab[q][0] = r * cos(th);
            tab[q][1] = r * sin(th);
        } else {
            const double th = ((q / 4) % 4) * ts;
            const double ph = (q / 16) * (ts / 2.0) + M_PI / 4.0 / 2.0;
            tab[q][0] = r * sin(ph) * cos(th);
            tab[q][1] = r * sin(ph) * sin(th);
            tab[q][2] = r * cos(ph);
        }
    }
}

// Uploads both quadrature tables once per device (thread-safe).
void upload_quadrature(int /*D*/) {
    static std::mutex mu;
    static std::vector<int> done;  // devices already holding the tables
    int dev = 0;
    NAGA_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    if (std::find(done.begin(), done.end(), dev) != done.end()) return;
    static const double wr[4] = {0.652145, 0.652145, 0.347855, 0.347855};
    double tab[2][64][3];
    fill_quadrature(2, tab[0]);
    fill_quadrature(3, tab[1]);
    NAGA_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_quad_unit), tab, sizeof(tab)));
    NAGA_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_quad_rw), wr, sizeof(wr)));
    done.push_back(dev);
}

template <int D, class T>
void launch_divw_d(int nmax, const float* src, const float* query, int64_t n_q,
                   const uint32_t* idx, const float* d2, int k, int rbf,
                   const double* hbar, const uint8_t* kvar, float* W, double* W64, int* info,
                   hipStream_t st) {
#define NAGA_DIVW(NM)                                                                 \
    case NM:                                                                          \
        k_divw<NM, D, T><<<n_q, 64, 0, st>>>(src, query, n_q, idx, d2, k, rbf, hbar, \
                                              kvar, W, W64, info);                    \
        break;
    switch (nmax) {
        NAGA_DIVW(20) NAGA_DIVW(28) NAGA_DIVW(36) NAGA_DIVW(44) NAGA_DIVW(52) NAGA_DIVW(64)
        default: fail(kInvalidArgument, "stencil too wide");
    }
#undef NAGA_DIVW
}

template <int D, class T>
void launch_rpim_d(int nmax, const float* src, const float* query, int64_t n_q,
                   const uint32_t* idx, int k, int rbf, double spacing, float* w,
                   double* w64, int* info, hipStream_t st, int group) {
#define NAGA_RPIM(NM)                                                                  \
    case NM:                                                                           \
        k_rpim<NM, D, T><<<n_q, 64, 0, st>>>(src, query, n_q, idx, k, rbf, spacing, w, \
                                              w64, info, group);                       \
        break;
    switch (nmax) {
        NAGA_RPIM(20) NAGA_RPIM(28) NAGA_RPIM(36) NAGA_RPIM(44) NAGA_RPIM(52) NAGA_RPIM(64)
        default: fail(kInvalidArgument, "stencil too wide");
    }
#undef NAGA_RPIM
}

}  // namespace

size_t cell_bins_bytes(int64_t n) { return bin_layout(n).total; }

CellBins launch_bin_points(int D, const float* pts, int64_t n, double per_cell, double width,
                           void* scratch_mem, size_t bytes, hipStream_t st,
                           double crowded_per_cell) {
    require(D >= 1 && D <= 3, "dimension must be 1, 2 or 3");
    require(n > 0, "no reference points");
    require(n < (int64_t(1) << 31), "at most 2^31 - 1 points");
    require(per_cell > 0.0 || width > 0.0, "cell size must be positive");
    const BinLayout L = bin_layout(n);
    require(scratch_mem != nullptr && bytes >= L.total, "cell binning scratch too small");
    char* base = static_cast<char*>(scratch_mem);
    CellBins b{};
    b.grid = reinterpret_cast<CellGrid*>(base + L.grid);
    b.start = reinterpret_cast<uint32_t*>(base + L.start);
    b.counts = reinterpret_cast<uint32_t*>(base + L.counts);
    b.sorted = reinterpret_cast<uint32_t*>(base + L.sorted);
    b.pts = reinterpret_cast<float4*>(base + L.pts);
    b.cap = L.cap;
    b.n = n;
    double* partial = reinterpret_cast<double*>(base + L.partial);
    uint32_t* bsum = reinterpret_cast<uint32_t*>(base + L.bsum);
    const int64_t M = L.cap + 1;
    const int64_t nbn = (n + 255) / 256;
    Crowding c{nullptr, L.nblocks, n, L.cap, per_cell, crowded_per_cell};
    uint64_t* pairs = nullptr;
    if (per_cell > 0.0 && crowded_per_cell > 0.0 && crowded_per_cell < per_cell)
        c.pairs = pairs = reinterpret_cast<uint64_t*>(base + L.pairs);
    k_bounds<<<kBoundBlocks, 256, 0, st>>>(pts, n, D, partial, b.counts, M);
    k_grid<<<1, kBoundBlocks, 0, st>>>(partial, D, n, per_cell > 0.0 ? per_cell : 0.0,
                                       per_cell > 0.0 ? 0.0 : width, L.cap, b.grid);
    k_count_cells<<<nbn, 256, 0, st>>>(pts, n, b.grid, b.counts);
    k_scan_local<<<L.nblocks, 256, 0, st>>>(b.counts, M, b.start, bsum, pairs);
    if (pairs) {  // again in narrower cells where the cloud is crowded
        k_recount_cells<<<std::min<int64_t>(nbn, 1024), 256, 0, st>>>(pts, b.grid, c, b.counts);
        k_rescan_local<<<L.nblocks, 256, 0, st>>>(c, b.counts, M, b.start, bsum);
    }
    k_scan_sums<<<1, 256, 0, st>>>(bsum, L.nblocks, b.grid, c);
    k_scan_add<<<L.nblocks, 256, 0, st>>>(b.start, M, bsum);
    // the scatter counts each cell up from the scan's zeros, leaving the sizes
    k_scatter_cells<<<nbn, 256, 0, st>>>(pts, n, b.grid, b.start, b.counts, b.sorted,
                                          b.pts);
    hip_check(hipGetLastError(), "cell binning");
    return b;
}

DeviceCells bin_points_device(int D, const float* pts, int64_t n, hipStream_t st,
                              double per_cell, double width, double crowded_per_cell) {
    DeviceCells c;
    const size_t bytes = cell_bins_bytes(n);
    c.mem.allocate(bytes);
    c.bins = launch_bin_points(D, pts, n, per_cell, width, c.mem.get(), bytes, st,
                               crowded_per_cell);
    return c;
}

// Wider cells waste candidates, narrower ones fail the R = 1 box more often
// (2 points per cell, as before, needs R = 3 and 49 rows for k = 32).
double knn_points_per_cell(int D, int k) {
    // 1.1^D times the points over the unit ball's volume (pi, 4 pi / 3)
    const double c = D == 3 ? 1.331 / 4.18879 : 1.21 / 3.14159;
    return std::max(2.0, c * double(k));
}

DeviceCells knn_bins_device(int D, const float* pts, int64_t n, int k, hipStream_t st) {
    return bin_points_device(D, pts, n, st, knn_points_per_cell(D, k), 0.0, kKnnCrowdedPerCell);
}

void launch_knn(int D, const CellBins& bins, const float* query, int64_t n_q, int k,
                float* d2_out, uint32_t* idx_out, hipStream_t st) {
    require(D == 2 || D == 3, "dimension must be 2 or 3");
    require(k >= 1 && k <= 64, "k must be in [1, 64]");
    require(bins.n >= k, "fewer reference points than neighbours requested");
    if (n_q == 0) return;
    const int64_t blocks = (n_q + kKnnBlockQueries - 1) / kKnnBlockQueries;
    if (D == 3)
        k_knn<3><<<blocks, 256, 0, st>>>(bins.grid, bins.pts, bins.start, query, n_q, k, d2_out,
                                         idx_out);
    else
        k_knn<2><<<blocks, 256, 0, st>>>(bins.grid, bins.pts, bins.start, query, n_q, k, d2_out,
                                         idx_out);
    hip_check(hipGetLastError(), "knn");
}

void launch_batched_lu_solve(int n, int nrhs, int64_t batch, double* A, double* B,
                             int* info, hipStream_t st) {
    const int nmax = pick_nmax(n);
    require(nmax > 0 && n >= 1, "n must be in [1, 64]");
    require(nrhs >= 1, "nrhs must be >= 1");
    if (batch == 0) return;
#define NAGA_LU(NM) \
    case NM: k_batched_lu<NM><<<batch, 64, 0, st>>>(n, nrhs, batch, A, B, info); break;
    switch (nmax) { NAGA_LU(20) NAGA_LU(28) NAGA_LU(36) NAGA_LU(44) NAGA_LU(52) NAGA_LU(64) }
#undef NAGA_LU
    hip_check(hipGetLastError(), "batched lu");
}

void launch_divergence_weights(int D, const float* src, const float* query,
                               int64_t n_q, const uint32_t* idx, const float* d2,
                               int k, int rbf, const double* hbar, float* W,
                               double* W64, int* info, hipStream_t st, const uint8_t* kvar,
                               int solve_bits) {
    const int nmax = pick_nmax(k + D + 1);
    require(nmax > 0, "stencil too wide (k + D + 1 must be <= 64)");
    require(k >= 2, "k must be >= 2");
    require(solve_bits == 64 || solve_bits == 32, "solve precision must be 64 or 32 bits");
    if (n_q == 0) return;
    upload_quadrature(D);
    const bool f32 = solve_bits == 32;
    if (D == 2 && f32)
        launch_divw_d<2, float>(nmax, src, query, n_q, idx, d2, k, rbf, hbar, kvar, W, W64, info,
                                st);
    else if (D == 2)
        launch_divw_d<2, double>(nmax, src, query, n_q, idx, d2, k, rbf, hbar, kvar, W, W64,
                                 info, st);
    else if (f32)
        launch_divw_d<3, float>(nmax, src, query, n_q, idx, d2, k, rbf, hbar, kvar, W, W64, info,
                                st);
    else
        launch_divw_d<3, double>(nmax, src, query, n_q, idx, d2, k, rbf, hbar, kvar, W, W64,
                                 info, st);
    hip_check(hipGetLastError(), "divergence weights");
}

void launch_rpim_weights(int D, const float* src, const float* query, int64_t n_q,
                         const uint32_t* idx, int k, int rbf, double spacing,
                         float* w, double* w64, int* info, hipStream_t st, int solve_bits,
                         int group) {
    const int nmax = pick_nmax(k + D + 1);
    require(nmax > 0, "stencil too wide (k + D + 1 must be <= 64)");
    require(group >= 1, "group size must be >= 1");
    require(solve_bits == 64 || solve_bits == 32, "solve precision must be 64 or 32 bits");
    if (n_q == 0) return;
    const bool f32 = solve_bits == 32;
    if (D == 2 && f32)
        launch_rpim_d<2, float>(nmax, src, query, n_q, idx, k, rbf, spacing, w, w64, info, st, group);
    else if (D == 2)
        launch_rpim_d<2, double>(nmax, src, query, n_q, idx, k, rbf, spacing, w, w64, info, st, group);
    else if (f32)
        launch_rpim_d<3, float>(nmax, src, query, n_q, idx, k, rbf, spacing, w, w64, info, st, group);
    else
        launch_rpim_d<3, double>(nmax, src, query, n_q, idx, k, rbf, spacing, w, w64, info, st, group);
    hip_check(hipGetLastError(), "rpim weights");
}

void launch_filter_weights(int D, const float* pts, int64_t n, const uint32_t* idx,
                           int k, double h, float* wf, hipStream_t st, const uint8_t* kvar) {
    if (n == 0) return;
    k_filter<<<(n + 255) / 256, 256, 0, st>>>(D, pts, n, idx, k, h / 2.5, kvar, wf);
    hip_check(hipGetLastError(), "filter weights");
}

void launch_pad_entries(int64_t n, int k, int ks, int nc, const uint32_t* idx, const float* w,
                        uint32_t* idx_out, float* w_out, hipStream_t st) {
    if (n == 0) return;
    k_pad_entries<<<(n * ks + 255) / 256, 256, 0, st>>>(n, k, ks, nc, idx, w, idx_out, w_out);
    hip_check(hipGetLastError(), "stencil padding");
}

void launch_make_slab(int64_t n, int k, int nc, const uint32_t* idx, const float* w,
                      float* slab, hipStream_t st) {
    if (n == 0) return;
    k_make_slab<<<(n * k + 255) / 256, 256, 0, st>>>(n, k, nc, idx, w, slab);
    hip_check(hipGetLastError(), "slab");
}

void launch_make_slab_q9(int64_t n, int k, int nc, const uint32_t* idx, const float* w,
                         float* slab, hipStream_t st) {
    if (n == 0) return;
    const int64_t tot = n * q9_units(k, nc) * 4;
    k_make_slab_q9<<<(tot + 255) / 256, 256, 0, st>>>(n, k, nc, idx, w,
                                                      reinterpret_cast<uint32_t*>(slab));
    hip_check(hipGetLastError(), "slab");
}

void launch_pack_div_records(int64_t n, int k, const float* src, float* dst, hipStream_t st) {
    require(k % 8 == 0 && k <= 64, "packed divergence records need k a multiple of 8");
    if (n == 0) return;
    const int64_t tot = n * packed_div_units(k) * 4;
    k_pack_div_records<<<(tot + 255) / 256, 256, 0, st>>>(n, k, src,
                                                          reinterpret_cast<uint32_t*>(dst));
    hip_check(hipGetLastError(), "pack divergence records");
}

void launch_pack_filter_records(int64_t n, int k, const float* src, float* dst,
                                hipStream_t st) {
    require(k % 8 == 0 && k <= 64, "packed filter records need k a multiple of 8");
    if (n == 0) return;
    const int64_t tot = n * packed_filter_units(k) * 4;
    k_pack_filter_records<<<(tot + 255) / 256, 256, 0, st>>>(n, k, src,
                                                             reinterpret_cast<uint32_t*>(dst));
    hip_check(hipGetLastError(), "pack filter records");
}

void launch_ragged_records(int64_t n, int T, int KP, int upg, const int32_t* ng,
                           const int64_t* off, const float* src, float* dst, hipStream_t st) {
    if (n == 0) return;
    const int64_t tot = n * KP;
    k_ragged_records<<<(tot + 255) / 256, 256, 0, st>>>(n, T, KP, upg, ng, off,
                                                        reinterpret_cast<const float4*>(src),
                                                        reinterpret_cast<float4*>(dst));
    hip_check(hipGetLastError(), "ragged records");
}

bool stencils_self_first(int64_t n, int k, const uint32_t* idx, hipStream_t st) {
    if (n == 0) return true;
    DeviceBuffer<int> flag(1);
    const int one = 1;
    flag.upload(&one, 1, st);
    k_self_first<<<(n + 255) / 256, 256, 0, st>>>(n, k, idx, flag.get());
    hip_check(hipGetLastError(), "stencil check");
    int out = 0;
    flag.download(&out, 1, st);
    NAGA_HIP(hipStreamSynchronize(st));
    return out == 1;
}

void launch_self_past_k(int64_t n, int k, const uint8_t* kvar, uint32_t* idx, hipStream_t st) {
    if (n == 0) return;
    const int64_t tot = n * k;
    k_self_past_k<<<(tot + 255) / 256, 256, 0, st>>>(n, k, kvar, idx);
    hip_check(hipGetLastError(), "stencil padding");
}

void launch_tile_unions(int64_t nfluid, int k, int tile_nodes, const uint32_t* idx, int cap,
                        int32_t* counts, int32_t* usplit, const int64_t* uoff, uint32_t* ulist,
                        float* slab_a, int ncomp_a, float* slab_b, int ncomp_b, hipStream_t st) {
    require(tile_nodes > 0 && tile_nodes % 2 == 0 && k * tile_nodes <= kUnionMax,
            "stencil too wide for tile unions");
    const int64_t ntiles = (nfluid + tile_nodes - 1) / tile_nodes;
    if (ntiles == 0) return;
    k_tile_union<<<ntiles, 256, 0, st>>>(nfluid, k, tile_nodes, idx, cap, counts, usplit, uoff,
                                          ulist, slab_a, ncomp_a, slab_b, ncomp_b);
    hip_check(hipGetLastError(), "tile unions");
}

void launch_layer_only(int64_t n, const uint32_t* idx, uint32_t lo, uint32_t hi,
                       uint32_t zero_row, uint32_t* out, hipStream_t st) {
    if (n == 0) return;
    k_layer_only<<<(n + 255) / 256, 256, 0, st>>>(n, idx, lo, hi, zero_row, out);
    hip_check(hipGetLastError(), "layer-only stencil");
}

void launch_flag_neighbours(int64_t n, int k, const uint32_t* idx, int64_t lo,
                            int64_t hi, uint8_t* flag, hipStream_t st) {
    if (n == 0) return;
    k_flag<<<(n + 255) / 256, 256, 0, st>>>(n, k, idx, lo, hi, flag);
    hip_check(hipGetLastError(), "flag");
}

void launch_divergence_apply(int D, int64_t n, int k, const uint32_t* idx,
                             const float* W, const float* F, float off, float* out,
                             hipStream_t st) {
    if (n == 0) return;
    k_div_apply<<<(n + 255) / 256, 256, 0, st>>>(D, n, k, idx, W, F, off, out);
    hip_check(hipGetLastError(), "divergence apply");
}

}  // namespace naga_amd
