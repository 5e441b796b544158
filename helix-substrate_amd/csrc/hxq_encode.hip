// CDNAv3 encoder on the GPU: 1-D k-means codebook, nearest-codebook
// assignment and percentile outliers (the sidecar), and the pair-codebook
// (vector_dim 2) k-means steps, with the reference's CPU results reproduced
// bit for bit.
//
// Reference (helix_substrate/hxq_encoder.py:107-177 _simple_kmeans,
// hxq_writer_v3.py:427-470 _build_kmeans_codebook / _chunked_assign,
// generate_sidecars_v3.py:18-40 find_outliers_percentile) computes with
// numpy; the arithmetic restated here is numpy's:
//   * assignment: argmin_j |fl(x - c_j)| in fp32, first index on ties, NaN
//     distances win (numpy argmin returns the first NaN);
//   * cluster mean: np.mean of the members in index order = fp32 sum over
//     consecutive 8192-element blocks, each block summed pairwise (blocks of
//     <= 128 with eight running sums, larger ones split at n/2 rounded down
//     to a multiple of 8), divided by the count in fp32;
//   * percentiles: numpy's 'linear' method on the sorted data (virtual index
//     (n-1) q, lerp a + (b-a) t for t < 1/2 else b - (b-a)(1-t)); fp64 for
//     the k-means initialisation (an array of percentiles), fp32 for the
//     sidecar thresholds (a scalar percentile of fp32 data);
//   * convergence: max |new - old| (fp32) < rtol * (c_last - c_first).
// Every reduction is integer or follows that fixed order: results are
// deterministic and independent of the launch shape.
#include <cfloat>
#include <cmath>

#include "hxq_common.h"

namespace hxq {
namespace enc {

constexpr int kThreads = 256;
constexpr int kMaxK = 256;     // scalar codebooks with uint8 indices
constexpr int kMaxKW = 4096;   // wide scalar codebooks (uint16 indices)

// fp32 -> uint32 whose unsigned order is numpy's sort order (NaN last).
__device__ __forceinline__ uint32_t sort_key(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;  // NaN
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_float(uint32_t k) {
    if (k == 0xffffffffu) return __uint_as_float(0x7fc00000u);
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// ---------------------------------------------------------------------------
// nearest codebook entry
// ---------------------------------------------------------------------------
__device__ __forceinline__ float absdiff(float x, float c) {
#pragma clang fp contract(off)
    return fabsf(x - c);
}

// General scan: first index of the minimum; a NaN distance is a minimum.
__device__ __forceinline__ int nearest_scan(float x, const float *cb, int k) {
    int best = 0;
    float bd = absdiff(x, cb[0]);
    if (bd != bd) return 0;
    for (int j = 1; j < k; ++j) {
        const float d = absdiff(x, cb[j]);
        if (d != d) return j;
        if (d < bd) { bd = d; best = j; }
    }
    return best;
}

// Sorted, finite codebook staged in LDS for searching: the distances
// fall then rise with j, so the minimum is at the last entry <= x or the
// first entry > x; when the entry before is as near, the first index holding
// the minimum is found by a second binary search over the falling part.
//   tree: the search tree in level order (node e's children 2e and 2e + 1;
//     entries past k are +inf), `levels` deep.  The nodes of a level are
//     neighbours, so the lanes of a wave, each on its own path, read distinct
//     banks in the upper levels; a binary search of the sorted array reads
//     strides of 64 words there, one bank.
//   lin: -inf, -inf, the k entries, +inf: the entries around a position
//     without bounds checks.
template <int KM>
struct Book {
    float tree[2 * KM];
    float lin[KM + 3];
    int flag;
};

__device__ __forceinline__ int tree_levels(int k) { return 32 - __builtin_clz(k); }  // 2^levels - 1 >= k

// Fills the book; false (uniform): not sorted and finite, lin + 2 alone is valid.
template <int KM>
__device__ __forceinline__ bool stage_codebook(const float *cb, int k, Book<KM> &s) {
    if (threadIdx.x == 0) s.flag = 1;
    __syncthreads();
    for (int j = threadIdx.x; j < k; j += blockDim.x) {
        const float v = cb[j];
        s.lin[j + 2] = v;
        // finite and non-decreasing: the search applies
        if (!isfinite(v) || (j + 1 < k && !(v <= cb[j + 1]))) s.flag = 0;
    }
    if (threadIdx.x < 2) s.lin[threadIdx.x] = -INFINITY;
    if (threadIdx.x == 2) s.lin[k + 2] = INFINITY;
    const int m = tree_levels(k);
    for (int e = 1 + threadIdx.x; e < (1 << m); e += blockDim.x) {
        const int lv = 31 - __builtin_clz(e);
        const int j = ((2 * (e - (1 << lv)) + 1) << (m - 1 - lv)) - 1;
        s.tree[e] = j < k ? cb[j] : INFINITY;
    }
    __syncthreads();
    return s.flag != 0;
}

// V values at once: the levels are LDS round trips, and V independent chains
// of them run side by side.
template <int V, int KM>
__device__ __forceinline__ void nearest_sorted(const float (&x)[V], const Book<KM> &s, int k, int (&out)[V]) {
    const int m = tree_levels(k);
    uint32_t e[V];
#pragma unroll
    for (int v = 0; v < V; ++v) e[v] = 1;
    for (int l = 0; l < m; ++l) {
#pragma unroll
        for (int v = 0; v < V; ++v) e[v] = 2 * e[v] + (s.tree[e[v]] <= x[v] ? 1u : 0u);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        // number of entries <= x (x = +inf passes the padding too)
        const int pos = min(static_cast<int>(e[v]) - (1 << m), k);
        const float dp = absdiff(x[v], s.lin[pos]), dl = absdiff(x[v], s.lin[pos + 1]),
                    dr = absdiff(x[v], s.lin[pos + 2]);
        int r = max(pos - 1, 0);                       // (every entry > x, or x NaN: 0)
        if (dr < dl) {
            r = pos;
        } else if (pos > 0 && !(dp > dl)) {
            // first j < pos with |x - cb[j]| == dl (distances non-increasing on [0, pos))
            int a = 0, b = pos - 1;
            while (a < b) {
                const int mid = (a + b) >> 1;
                if (absdiff(x[v], s.lin[mid + 2]) <= dl) b = mid; else a = mid + 1;
            }
            r = a;
        }
        out[v] = r;
    }
}

// kAssignV consecutive weights per thread and round: 16-byte loads (x is
// 16-byte aligned or vec is false), one 8- or 16-byte store of their indices.
// Bound by the searches' LDS reads (nine levels and three entries a weight):
// 22.5M weights, 256 entries, 39 us (2.9 TB/s); 70 us with a binary search of
// the sorted array, 97 us one weight per thread and two such searches.
constexpr int kAssignV = 8;
template <typename IT, int KM>
__global__ __launch_bounds__(kThreads) void assign_kernel(const float *x, int64_t n, const float *cb,
                                                          int k, IT *idx, int vec) {
    __shared__ Book<KM> s;
    const bool sorted = stage_codebook(cb, k, s);
    for (int64_t i0 = (blockIdx.x * (int64_t)kThreads + threadIdx.x) * kAssignV; i0 < n;
         i0 += (int64_t)gridDim.x * kThreads * kAssignV) {
        float v[kAssignV];
        int c[kAssignV];
        const bool whole = vec && i0 + kAssignV <= n;
        if (whole) {
            const float4 a = *reinterpret_cast<const float4 *>(x + i0);
            const float4 b = *reinterpret_cast<const float4 *>(x + i0 + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
            v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int q = 0; q < kAssignV; ++q) v[q] = i0 + q < n ? x[i0 + q] : 0.f;
        }
        if (sorted) {
            nearest_sorted(v, s, k, c);
        } else {
#pragma unroll
            for (int q = 0; q < kAssignV; ++q) c[q] = nearest_scan(v[q], s.lin + 2, k);
        }
        if (whole) {
            uint32_t o[kAssignV * sizeof(IT) / 4];
#pragma unroll
            for (int q = 0; q < static_cast<int>(sizeof(o) / 4); ++q) {
                if constexpr (sizeof(IT) == 1)
                    o[q] = c[4 * q] | c[4 * q + 1] << 8 | c[4 * q + 2] << 16 | static_cast<uint32_t>(c[4 * q + 3]) << 24;
                else
                    o[q] = c[2 * q] | static_cast<uint32_t>(c[2 * q + 1]) << 16;
            }
            if constexpr (sizeof(IT) == 1) *reinterpret_cast<uint2 *>(idx + i0) = make_uint2(o[0], o[1]);
            else *reinterpret_cast<uint4 *>(idx + i0) = make_uint4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int q = 0; q < kAssignV; ++q)
                if (i0 + q < n) idx[i0 + q] = static_cast<IT>(c[q]);
        }
    }
}

// ---------------------------------------------------------------------------
// stable counting scatter: the passes of the radix sort and of Lloyd's update
// ---------------------------------------------------------------------------
// A pass splits n elements among k buckets, keeping index order within each:
// count per block of kPer consecutive elements (blk[bucket * nblk + block]),
// scan the blocks of each bucket (one wave per bucket), scatter.  Every
// element's place is fixed by the counts, so results do not depend on timing.
constexpr int kPer = 2048;                  // elements per block
constexpr int kWaves = kThreads / kWave;
constexpr int kRounds = kPer / kThreads;    // elements per lane
constexpr int kDigits = 256;

// Waits until this wave's stores and atomics are done.  Where they are
// device-scope atomics (performed past the XCD's own L2) and are read back by
// device-scope atomic loads, this orders them before a counter that another
// block looks at; a device-scope fence would also write the L2 back, for every
// wave that meets it (the select passes: 150 us with it, 30 without).
__device__ __forceinline__ void wait_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Radix digit of the sort keys; the first pass makes the keys from x.
struct DigitSrc {
    const float *x;        // first pass, else null
    const uint32_t *keys;
    int shift;
    __device__ uint32_t value(int64_t i) const { return x ? sort_key(x[i]) : keys[i]; }
    __device__ int bucket(int64_t, uint32_t v) const { return (v >> shift) & (kDigits - 1); }
};

// Cluster ids and values of Lloyd's update.
template <typename IT>
struct ClusterSrc {
    const float *x;
    const IT *idx;
    __device__ uint32_t value(int64_t i) const { return __float_as_uint(x[i]); }
    __device__ int bucket(int64_t i, uint32_t) const { return idx[i]; }
};

__global__ __launch_bounds__(kThreads) void digit_count_kernel(DigitSrc src, int64_t n, int64_t nblk,
                                                               int32_t *blk) {
    __shared__ int32_t cnt[kDigits];
    for (int j = threadIdx.x; j < kDigits; j += kThreads) cnt[j] = 0;
    __syncthreads();
    const int64_t lo = blockIdx.x * (int64_t)kPer + threadIdx.x;
    uint32_t v[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) v[r] = lo + r * kThreads < n ? src.value(lo + r * kThreads) : 0u;
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (lo + r * kThreads < n) atomicAdd(&cnt[src.bucket(0, v[r])], 1);
    __syncthreads();
    for (int j = threadIdx.x; j < kDigits; j += kThreads) blk[j * nblk + blockIdx.x] = cnt[j];
}

// blk[j][b] -> elements of bucket j in blocks before b; counts[j] = all of them
__global__ __launch_bounds__(kThreads) void bucket_scan_kernel(int32_t *blk, int64_t nblk, int k, int32_t *counts,
                                                               const int32_t *done) {
    if (done && *done) return;
    const int lane = threadIdx.x & 63;
    const int j = blockIdx.x * kWaves + threadIdx.x / kWave;
    if (j >= k) return;
    int32_t *row = blk + j * nblk;
    int base = 0;
    for (int64_t b0 = 0; b0 < nblk; b0 += kWave) {
        const int64_t b = b0 + lane;
        const int c = b < nblk ? row[b] : 0;
        const int inc = wave_scan(c);
        if (b < nblk) row[b] = base + inc - c;
        base += __builtin_amdgcn_readlane(inc, 63);
    }
    if (lane == 0) counts[j] = base;
}

// Exclusive scan of counts[0, k) over the block: thread t owns PT consecutive
// buckets from t * PT; returns the start of its first one.
template <int PT>
__device__ __forceinline__ int block_start(const int32_t *counts, int k, int (&c)[PT], int *s_w) {
    int sum = 0;
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const int j = threadIdx.x * PT + q;
        c[q] = j < k ? counts[j] : 0;
        sum += c[q];
    }
    const int inc = wave_scan(sum);
    if ((threadIdx.x & 63) == 63) s_w[threadIdx.x / kWave] = inc;
    __syncthreads();
    int base = inc - sum;
    for (int w = 0; w < static_cast<int>(threadIdx.x / kWave); ++w) base += s_w[w];
    return base;
}

// Wave w of a block owns kPer / 4 consecutive elements, 64 per round.  The
// lanes of a round that share a bucket find each other by one ballot per
// bucket bit; a running count per (wave, bucket) in LDS carries over rounds.
template <typename SRC, int KM>
__global__ __launch_bounds__(kThreads) void bucket_scatter_kernel(SRC src, int64_t n, int64_t nblk, int k,
                                                                  const int32_t *blk, const int32_t *counts,
                                                                  uint32_t *out, const int32_t *done) {
    if (done && *done) return;
    constexpr int PT = KM / kThreads;
    __shared__ int32_t cnt[kWaves][KM];
    __shared__ int s_w[kWaves];
    for (int j = threadIdx.x; j < kWaves * KM; j += kThreads) (&cnt[0][0])[j] = 0;
    const int lane = threadIdx.x & 63, w = threadIdx.x / kWave;
    const int64_t lo = blockIdx.x * (int64_t)kPer + w * (kPer / kWaves) + lane;
    uint32_t val[kRounds];
    int bkt[kRounds], rank[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int64_t i = lo + r * kWave;
        val[r] = i < n ? src.value(i) : 0u;
        bkt[r] = i < n ? src.bucket(i, val[r]) : 0;
    }
    int c[PT];
    int start = block_start(counts, k, c, s_w);   // (its barrier also covers cnt = 0)
    volatile int32_t *mine = cnt[w];
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const bool ok = lo + r * kWave < n;
        unsigned long long same = __ballot(ok);
#pragma unroll
        for (int bit = 1; bit < KM; bit <<= 1) {
            const unsigned long long m = __ballot((bkt[r] & bit) != 0);
            same &= (bkt[r] & bit) ? m : ~m;
        }
        const int before = mine[bkt[r]];          // a wave's LDS accesses keep their order
        rank[r] = before + __popcll(same & below);
        if (ok && (same >> lane) == 1ull) mine[bkt[r]] = rank[r] + 1;   // the last of them
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PT; ++q) {
        const int j = threadIdx.x * PT + q;
        if (j < k) {
            int s = start + blk[j * nblk + blockIdx.x];
            for (int ww = 0; ww < kWaves; ++ww) {
                const int t = cnt[ww][j];
                cnt[ww][j] = s;
                s += t;
            }
        }
        start += c[q];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (lo + r * kWave < n) out[cnt[w][bkt[r]] + rank[r]] = val[r];
}

// ---------------------------------------------------------------------------
// k-means initialisation and bookkeeping
// ---------------------------------------------------------------------------
// distinct values of the sorted keys (NaNs count once, as np.unique)
__global__ void zero_i32_kernel(int32_t *p) { *p = 0; }

__global__ __launch_bounds__(kThreads) void count_unique_kernel(const uint32_t *keys, int64_t n,
                                                                int32_t *count) {
    int32_t c = 0;
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kThreads) {
        if (i == 0) { ++c; continue; }
        const uint32_t a = keys[i - 1], b = keys[i];
        // +0.0 and -0.0 are equal values
        const bool same = a == b || (key_float(a) == key_float(b));
        c += !same;
    }
    // one atomic per block, 128 of them: they queue on the one address (13 ns
    // each: 27 us with 2000)
    __shared__ int32_t s[kWaves];
    c = __builtin_amdgcn_readlane(wave_scan(c), 63);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x / kWave] = c;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(count, s[0] + s[1] + s[2] + s[3]);
}

// centroid j = percentile(data, q_j) with numpy's fp64 'linear' lerp, as fp32
__global__ __launch_bounds__(kMaxK) void kmeans_init_kernel(const uint32_t *keys, int64_t n, const double *q, int k,
                                   float *cb, double rtol, double *abs_tol, int32_t *done,
                                   int32_t *iters, int32_t *arrived) {
#pragma clang fp contract(off)
    // numpy's percentile is NaN for every q once the data holds a NaN
    // (sorted last)
    const bool has_nan = keys[n - 1] == 0xffffffffu;
    for (int j = threadIdx.x; j < k; j += blockDim.x) {
        const double v = static_cast<double>(n - 1) * q[j];
        double r;
        if (has_nan) {
            r = static_cast<double>(key_float(0xffffffffu));
        } else if (v >= static_cast<double>(n - 1)) {
            r = static_cast<double>(key_float(keys[n - 1]));
        } else {
            const int64_t i = static_cast<int64_t>(floor(v));
            const double t = v - static_cast<double>(i);
            const float a = key_float(keys[i]), b = key_float(keys[i + 1]);
            const double d = static_cast<double>(b - a);  // fp32 difference
            r = t >= 0.5 ? static_cast<double>(b) - d * (1.0 - t) : static_cast<double>(a) + d * t;
        }
        cb[j] = static_cast<float>(r);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double range = static_cast<double>(cb[k - 1] - cb[0]);
        if (range < 1e-30) range = 1.0;
        *abs_tol = rtol * range;
        *done = 0;
        *iters = 0;
        *arrived = 0;
    }
}

// Lloyd step 1: assignment + per-block cluster counts (block b: elements
// [b * kPer, (b + 1) * kPer), each thread's kRounds values searched together).
template <typename IT, int KM>
__global__ __launch_bounds__(kThreads) void km_assign_kernel(const float *x, int64_t n, int64_t nblk,
                                                             const float *cb, int k, IT *idx,
                                                             int32_t *blk, const int32_t *done) {
    if (*done) return;
    __shared__ Book<KM> s;
    __shared__ int32_t s_cnt[KM];
    const int64_t lo = blockIdx.x * (int64_t)kPer + threadIdx.x;
    float v[kRounds];
    int c[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) v[r] = lo + r * kThreads < n ? x[lo + r * kThreads] : 0.f;
    for (int j = threadIdx.x; j < KM; j += kThreads) s_cnt[j] = 0;
    const bool sorted = stage_codebook(cb, k, s);
    if (sorted) {
        nearest_sorted(v, s, k, c);
    } else {
#pragma unroll
        for (int r = 0; r < kRounds; ++r) c[r] = nearest_scan(v[r], s.lin + 2, k);
    }
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        if (lo + r * kThreads < n) {
            idx[lo + r * kThreads] = static_cast<IT>(c[r]);
            atomicAdd(&s_cnt[c[r]], 1);
        }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < k; j += kThreads) blk[j * nblk + blockIdx.x] = s_cnt[j];
}

// Lloyd steps 2 and 3 are bucket_scan_kernel and bucket_scatter_kernel: the
// values in cluster order, index order within a cluster.

// numpy's pairwise tree over m <= 8192 elements: nodes above 128 split at
// m / 2 rounded down to a multiple of 8, so leaves hold 64..128 elements (or
// all m <= 128) and lie at depth 7 at most.  The leaf that the 7-bit path t
// (from the root, first step in the top bit) reaches: its range, and its
// depth, if t is the leftmost path through it.
constexpr int kDepth = 7;
constexpr int kLeaves = 1 << kDepth;
__device__ __forceinline__ bool pairwise_path(int m, int t, int &off, int &len, int &depth) {
    off = 0;
    len = m;
    depth = 0;
    while (len > 128) {
        int m2 = len / 2;
        m2 -= m2 % 8;
        if (t >> (kDepth - 1 - depth) & 1) {
            off += m2;
            len -= m2;
        } else {
            len = m2;
        }
        ++depth;
    }
    return (t & ((1 << (kDepth - depth)) - 1)) == 0;
}

// Lloyd step 4: the mean of cluster blockIdx.x as np.mean gives it, bit for
// bit, and after the last cluster the movement and convergence test.
// Per 8192-element block of the cluster's members, staged in LDS: eight lanes
// per leaf of the pairwise tree, one for each of numpy's eight running sums
// (DPP adds in its order, then the up to seven last elements), then the tree
// level by level; block sums are added in order and divided by the count.
// Empty clusters keep their centroid.  (One thread per leaf, reading memory,
// and one listing the leaves and combining them: 93 us per step at 500K
// values, 256 clusters.)
template <int KM>
__global__ __launch_bounds__(kThreads) void km_sum_kernel(const float *sorted_vals, const int32_t *counts, int k,
                                                          float *cb, float *means, const double *abs_tol,
                                                          int32_t *done, int32_t *iters, int32_t *arrived) {
#pragma clang fp contract(off)
    if (*done) return;
    __shared__ __attribute__((aligned(16))) float s_v[8192];
    __shared__ float s_leaf[kLeaves];
    __shared__ int s_w[kWaves];
    __shared__ int s_flag;
    const int j = blockIdx.x;
    const int32_t c = counts[j];
    int before = 0;
    for (int q = threadIdx.x; q < j; q += kThreads) before += counts[q];
    before = __builtin_amdgcn_readlane(wave_scan(before), 63);
    if ((threadIdx.x & 63) == 0) s_w[threadIdx.x / kWave] = before;
    __syncthreads();
    int start = 0;
    for (int w = 0; w < kWaves; ++w) start += s_w[w];
    const float *a = sorted_vals + start;
    float sum = 0.f;
    for (int32_t s = 0; s < c; s += 8192) {
        const int m = min(8192, c - s);
        for (int i = threadIdx.x; i < m; i += kThreads) s_v[i] = a[s + i];
        __syncthreads();
        const int q = threadIdx.x & 7;
        for (int t = threadIdx.x >> 3; t < kLeaves; t += kThreads / 8) {
            int off, len, depth;
            if (!pairwise_path(m, t, off, len, depth)) continue;  // the same for a leaf's eight lanes
            const float *e = s_v + off;
            float r = 0.f;
            if (len < 8) {
                for (int i = 0; i < len; ++i) r += e[i];
            } else {
                const int whole = len - len % 8;
                r = e[q];
                for (int i = 8; i < whole; i += 8) r += e[i + q];
                r = dpp_add<0xb1, 0xf>(r);     // r0 + r1, r2 + r3, ...
                r = dpp_add<0x4e, 0xf>(r);     // (r0 + r1) + (r2 + r3), ...
                r = dpp_add<0x141, 0xf>(r);    // row_half_mirror: the other quad's sum
                for (int i = whole; i < len; ++i) r += e[i];
            }
            if (q == 0) s_leaf[t] = r;
        }
        __syncthreads();
        // node p of depth d sits at its leftmost path p << (7 - d); it is
        // inner when that path's leaf lies deeper
        if (threadIdx.x < kWave) {
            for (int d = kDepth - 1; d >= 0; --d) {
                const int p = threadIdx.x;
                const int at = p << (kDepth - d);
                if (p < (1 << d)) {
                    int off, len, depth;
                    // (a path that leaves the tree early is no node: its depth stays below d)
                    const bool node = pairwise_path(m, at, off, len, depth);
                    if (node && depth > d) s_leaf[at] = s_leaf[at] + s_leaf[at + (1 << (kDepth - 1 - d))];
                }
                wave_lds_order();
            }
        }
        __syncthreads();
        const float p = s_leaf[0];
        sum = s == 0 ? p : sum + p;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const float mean = c == 0 ? cb[j] : sum / static_cast<float>(c);
        __hip_atomic_store(&means[j], mean, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        wait_vmem();
        s_flag = atomicAdd(arrived, 1) == k - 1;
    }
    __syncthreads();
    if (!s_flag) return;
    // the last cluster's block: movement, convergence, the new codebook
    float mx = 0.f;
    int nan = 0;
    for (int q = threadIdx.x; q < k; q += kThreads) {
        const float d = fabsf(__hip_atomic_load(&means[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - cb[q]);
        nan |= d != d;
        mx = fmaxf(mx, d);
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    nan = __ballot(nan) != 0;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
        s_leaf[threadIdx.x / kWave] = mx;
        s_w[threadIdx.x / kWave] = nan;
    }
    __syncthreads();
    for (int w = 0; w < kWaves; ++w) {
        mx = fmaxf(mx, s_leaf[w]);
        nan |= s_w[w];
    }
    // numpy's max propagates NaN; NaN < tol is false: no convergence
    const bool conv = !nan && static_cast<double>(mx) < *abs_tol;
    if (!conv)
        for (int q = threadIdx.x; q < k; q += kThreads)
            cb[q] = __hip_atomic_load(&means[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (threadIdx.x == 0) {
        *iters += 1;
        *arrived = 0;
        if (conv) *done = 1;
    }
}

// ---------------------------------------------------------------------------
// radix select (exact order statistics of up to 4 ranks) and outliers
// ---------------------------------------------------------------------------
constexpr int kSelMax = 4;

// Digits of 11, 11 and 10 bits of the sort key, from the top.
constexpr int kSelBins = 2048;
__host__ __device__ constexpr int sel_shift(int pass) { return pass == 0 ? 21 : pass == 1 ? 10 : 0; }

struct SelState {
    uint32_t prefix[kSelMax];  // key bits fixed so far
    uint32_t rank[kSelMax];    // rank within the keys matching prefix
    uint32_t hist[kSelMax][kSelBins];
    int32_t nan_count;
    int32_t arrived;
};

constexpr int kSelThreads = 1024;
// One pass: a histogram of the digit over the keys that match a rank's
// prefix, and in the last block to finish, the digit each rank falls into.
// Ranks with one prefix share a histogram (all of them in the first pass,
// neighbours usually to the end).  Bound by reading x (16 bytes a lane;
// 22.5M values: 31 us for the first pass, 25 us for the others, whose matches
// are few; blocks of 4 waves, which keep half as many loads in flight, 47;
// four 8-bit passes that counted every rank for itself 69 us each, and 15 us
// for one thread a rank picking the digit).
__global__ __launch_bounds__(kSelThreads) void select_pass_kernel(const float *x, int64_t n, int m, int pass,
                                                               int vec, SelState *st, float *out) {
    __shared__ uint32_t h[kSelMax][kSelBins];
    __shared__ int s_last;
    __shared__ int s_w[kSelThreads / kWave];
    const int shift = sel_shift(pass);
    const uint32_t hi_mask = pass == 0 ? 0u : pass == 1 ? 0xffffffffu << 21 : 0xffffffffu << 10;
    uint32_t pre[kSelMax];
    int slot[kSelMax];   // the first rank with this prefix
#pragma unroll
    for (int r = 0; r < kSelMax; ++r) {
        pre[r] = st->prefix[min(r, m - 1)];
        slot[r] = r;
#pragma unroll
        for (int q = kSelMax - 1; q >= 0; --q)
            if (q < r && pre[q] == pre[r]) slot[r] = q;
    }
    for (int i = threadIdx.x; i < kSelMax * kSelBins; i += kSelThreads) (&h[0][0])[i] = 0;
    __syncthreads();
    int32_t nans = 0;
    auto count = [&](float v) {
        const uint32_t key = sort_key(v);
        if (pass == 0 && key == 0xffffffffu) ++nans;
        const uint32_t d = (key >> shift) & (pass == 2 ? 1023u : 2047u);
#pragma unroll
        for (int r = 0; r < kSelMax; ++r)
            if (r < m && slot[r] == r && ((key ^ pre[r]) & hi_mask) == 0) atomicAdd(&h[r][d], 1u);
    };
    // 8 consecutive values a thread and round
    for (int64_t i0 = (blockIdx.x * (int64_t)kSelThreads + threadIdx.x) * 8; i0 < n;
         i0 += (int64_t)gridDim.x * kSelThreads * 8) {
        if (vec && i0 + 8 <= n) {
            const float4 a = *reinterpret_cast<const float4 *>(x + i0);
            const float4 b = *reinterpret_cast<const float4 *>(x + i0 + 4);
            count(a.x); count(a.y); count(a.z); count(a.w);
            count(b.x); count(b.y); count(b.z); count(b.w);
        } else {
            for (int q = 0; q < 8; ++q)
                if (i0 + q < n) count(x[i0 + q]);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < m * kSelBins; i += kSelThreads) {
        const uint32_t v = (&h[0][0])[i];
        if (v) atomicAdd(&st->hist[i / kSelBins][i % kSelBins], v);
    }
    if (pass == 0 && nans) atomicAdd(&st->nan_count, nans);
    wait_vmem();
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(&st->arrived, 1) == static_cast<int>(gridDim.x) - 1;
    __syncthreads();
    if (!s_last) return;
    // the last block: rank r falls into the first bin whose running count
    // passes it; each thread holds PT consecutive bins
    constexpr int PT = kSelBins / kSelThreads;
    for (int r = 0; r < m; ++r) {
        uint32_t c[PT];
        uint32_t sum = 0;
#pragma unroll
        for (int q = 0; q < PT; ++q) {
            c[q] = __hip_atomic_load(&st->hist[slot[r]][threadIdx.x * PT + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sum += c[q];
        }
        const uint32_t inc = static_cast<uint32_t>(wave_scan(static_cast<int>(sum)));
        if ((threadIdx.x & 63) == 63) s_w[threadIdx.x / kWave] = static_cast<int>(inc);
        __syncthreads();
        uint32_t base = inc - sum;
        for (int w = 0; w < static_cast<int>(threadIdx.x / kWave); ++w) base += static_cast<uint32_t>(s_w[w]);
        const uint32_t rank = st->rank[r];
        if (rank >= base && rank - base < sum) {   // one thread
            uint32_t left = rank - base;
            int d = 0;
#pragma unroll
            for (int q = 0; q < PT; ++q) {
                if (d == q && left >= c[q]) {
                    left -= c[q];
                    ++d;
                }
            }
            const uint32_t p = pre[r] | static_cast<uint32_t>(threadIdx.x * PT + d) << shift;
            st->prefix[r] = p;
            h[0][r] = left;      // (st->rank[r] is still being read)
            if (pass == 2) out[r] = key_float(p);
        }
        __syncthreads();
    }
    if (threadIdx.x < m) st->rank[threadIdx.x] = h[0][threadIdx.x];
    for (int i = threadIdx.x; i < m * kSelBins; i += kSelThreads) st->hist[i / kSelBins][i % kSelBins] = 0;
    if (threadIdx.x == 0) st->arrived = 0;
}

__global__ void select_init_kernel(const int64_t *ranks, int m, SelState *st) {
    for (int i = threadIdx.x; i < kSelMax * kSelBins; i += blockDim.x) (&st->hist[0][0])[i] = 0;
    if (threadIdx.x < kSelMax) {
        st->prefix[threadIdx.x] = 0;
        st->rank[threadIdx.x] = threadIdx.x < m ? static_cast<uint32_t>(ranks[threadIdx.x]) : 0;
    }
    if (threadIdx.x == 0) {
        st->nan_count = 0;
        st->arrived = 0;
    }
}

// Outliers: x < lo or x > hi, positions ascending, in two passes over x.  A
// wave owns kChunk consecutive values, 256 a round (four consecutive ones a
// lane); the chunks' counts are scanned in between, so that no wave waits for
// another.  Bound by reading x: 22.5M values 16 us a pass (65536-value blocks
// with a block-wide scan per 256 values: 80 and 127 us, 38 us for one thread
// scanning the blocks).
constexpr int kChunk = 4096;

__device__ __forceinline__ float4 load4(const float *x, int64_t i, int64_t n, int vec) {
    if (vec && i + 4 <= n) return *reinterpret_cast<const float4 *>(x + i);
    const float none = __uint_as_float(0x7fc00000u);   // NaN: never an outlier
    return make_float4(i < n ? x[i] : none, i + 1 < n ? x[i + 1] : none, i + 2 < n ? x[i + 2] : none,
                       i + 3 < n ? x[i + 3] : none);
}

__global__ __launch_bounds__(kThreads) void outlier_count_kernel(const float *x, int64_t n, int64_t chunks, int vec,
                                                                 const float *lohi, int64_t *cnt) {
    const int lane = threadIdx.x & 63;
    const int64_t ch = blockIdx.x * (int64_t)kWaves + threadIdx.x / kWave;
    if (ch >= chunks) return;
    const float lo = lohi[0], hi = lohi[1];
    int c = 0;
#pragma unroll 8
    for (int r = 0; r < kChunk / 256; ++r) {
        const float4 v = load4(x, ch * kChunk + r * 256 + lane * 4, n, vec);
        c += (v.x < lo) | (v.x > hi);
        c += (v.y < lo) | (v.y > hi);
        c += (v.z < lo) | (v.z > hi);
        c += (v.w < lo) | (v.w > hi);
    }
    c = __builtin_amdgcn_readlane(wave_scan(c), 63);
    if (lane == 0) cnt[ch] = c;
}

// cnt[c] -> outliers in chunks before c; *total = all of them
__global__ __launch_bounds__(1024) void outlier_scan_kernel(int64_t *cnt, int64_t chunks, int64_t *total) {
    __shared__ int s_w[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int64_t base = 0;
    for (int64_t c0 = 0; c0 < chunks; c0 += 4096) {
        int v[4], sum = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t c = c0 + threadIdx.x * 4 + q;
            v[q] = c < chunks ? static_cast<int>(cnt[c]) : 0;
            sum += v[q];
        }
        const int inc = wave_scan(sum);
        if (lane == 63) s_w[w] = inc;
        __syncthreads();
        int64_t s = base + inc - sum;
        for (int q = 0; q < 16; ++q) {
            if (q < w) s += s_w[q];
            base += s_w[q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t c = c0 + threadIdx.x * 4 + q;
            if (c < chunks) cnt[c] = s;
            s += v[q];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *total = base;
}

__global__ __launch_bounds__(kThreads) void outlier_write_kernel(const float *x, int64_t n, int64_t chunks, int vec,
                                                                 const float *lohi, const int64_t *cnt,
                                                                 int64_t cap, int64_t *pos, float *val) {
    const int lane = threadIdx.x & 63;
    const int64_t ch = blockIdx.x * (int64_t)kWaves + threadIdx.x / kWave;
    if (ch >= chunks) return;
    const float lo = lohi[0], hi = lohi[1];
    int64_t base = cnt[ch];
#pragma unroll 8
    for (int r = 0; r < kChunk / 256; ++r) {
        const int64_t i = ch * kChunk + r * 256 + lane * 4;
        const float4 v = load4(x, i, n, vec);
        const float e[4] = {v.x, v.y, v.z, v.w};
        bool hit[4];
        int c = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            hit[q] = (e[q] < lo) | (e[q] > hi);
            c += hit[q];
        }
        if (__ballot(c != 0) == 0) continue;   // wave-uniform
        const int inc = wave_scan(c);
        int64_t p = base + inc - c;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (hit[q]) {
                if (p < cap) {
                    pos[p] = i + q;
                    val[p] = e[q];
                }
                ++p;
            }
        }
        base += __builtin_amdgcn_readlane(inc, 63);
    }
}

// ---------------------------------------------------------------------------
// per-group affine fit: (s, o) = argmin sum_j (s c_j + o - w_j)^2 over the
// group's elements not in the sidecar, c_j = codebook[idx_j]; fp64 sums in a
// fixed order (lane l of the group's wave adds elements l, l+64, ... in turn,
// then a xor butterfly 32, 16, ..., 1), closed-form solution in fp64, fp32
// results.  Degenerate groups (n < 2 or a zero determinant) keep s = 1 and
// take o = mean(w - c) (0 for an empty group).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void mark_kernel(const int64_t *pos, int64_t m, uint32_t *bits) {
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < m;
         i += (int64_t)gridDim.x * kThreads) {
        const int64_t p = pos[i];
        atomicOr(&bits[p >> 5], 1u << (p & 31));
    }
}

__global__ __launch_bounds__(kThreads) void zero_u32_kernel(uint32_t *p, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kThreads)
        p[i] = 0u;
}

// v + the value of the lane the moves of its two halves name
template <int CTRL>
__device__ __forceinline__ double dpp_add_f64(double v) {
#pragma clang fp contract(off)
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, false);
    return v + __longlong_as_double(static_cast<long long>(hi) << 32 | static_cast<unsigned int>(lo));
}

__device__ __forceinline__ double swap_add_f64(double p, double q, bool by32) {
#pragma clang fp contract(off)
    const long long a = __double_as_longlong(p), b = __double_as_longlong(q);
    const unsigned int al = static_cast<unsigned int>(a), ah = static_cast<unsigned int>(a >> 32);
    const unsigned int bl = static_cast<unsigned int>(b), bh = static_cast<unsigned int>(b >> 32);
    const auto lo = by32 ? __builtin_amdgcn_permlane32_swap(al, bl, false, false)
                         : __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto hi = by32 ? __builtin_amdgcn_permlane32_swap(ah, bh, false, false)
                         : __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    return __longlong_as_double(static_cast<long long>(hi[0]) << 32 | lo[0]) +
           __longlong_as_double(static_cast<long long>(hi[1]) << 32 | lo[1]);
}

// Wave sums of four values, each in the order of an xor butterfly 32, 16, ...,
// 1 and without LDS: a lane swap halves two values against each other (the
// lower lanes go on with the first, the upper ones with the second), so after
// the steps 32 and 16 one register holds all four, a row of 16 lanes each:
// v[0], v[2], v[1], v[3].  Within a row a rotation by 8, 4, 2 and 1 stands for
// the xor: after each step the values repeat with that period.
__device__ __forceinline__ double wave_sum4_f64(const double (&v)[4]) {
    const double p = swap_add_f64(v[0], v[1], true), q = swap_add_f64(v[2], v[3], true);
    double r = swap_add_f64(p, q, false);
    r = dpp_add_f64<0x128>(r);  // row_ror:8
    r = dpp_add_f64<0x124>(r);
    r = dpp_add_f64<0x122>(r);
    return dpp_add_f64<0x121>(r);
}

// A wave fits kFitUnits consecutive groups, their loads all requested first.
// 11008 x 2048 weights in groups of 128: 69 us, bound by the fp64 additions
// (each sum by itself over the wave 90; by LDS permutes, one group per wave,
// 120).
constexpr int kFitUnits = 4;
template <typename IT, int KM>
__global__ __launch_bounds__(kThreads) void affine_fit_kernel(const float *w, const IT *idx,
                                                              const float *cb, int k, int64_t rows,
                                                              int64_t cols, int group,
                                                              const uint32_t *bits, float *scale,
                                                              float *offset) {
#pragma clang fp contract(off)
    __shared__ float s_cb[KM];
    for (int j = threadIdx.x; j < KM; j += kThreads) s_cb[j] = j < k ? cb[j] : 0.f;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t ngroups = cols / group, units = rows * ngroups;
    const int64_t u0 = (blockIdx.x * (int64_t)kWaves + threadIdx.x / kWave) * kFitUnits;
    double sc[kFitUnits], sw[kFitUnits], scc[kFitUnits], scw[kFitUnits], sn[kFitUnits];
#pragma unroll
    for (int u = 0; u < kFitUnits; ++u) sc[u] = sw[u] = scc[u] = scw[u] = sn[u] = 0.0;
    for (int t = lane; t - lane < group; t += kWave) {
        float x[kFitUnits];
        int id[kFitUnits];
        bool use[kFitUnits];
#pragma unroll
        for (int u = 0; u < kFitUnits; ++u) {
            // the groups of a row, and the rows, follow each other in memory
            const int64_t e = (u0 + u) * group + t;
            use[u] = u0 + u < units && t < group;
            x[u] = use[u] ? w[e] : 0.f;
            id[u] = use[u] ? idx[e] : 0;
            if (bits && use[u]) use[u] = !((bits[e >> 5] >> (e & 31)) & 1u);
        }
#pragma unroll
        for (int u = 0; u < kFitUnits; ++u) {
            if (use[u]) {
                // an index past the table (a caller error) reads a zero entry, in bounds
                const double c = static_cast<double>(s_cb[min(id[u], KM - 1)]);
                const double v = static_cast<double>(x[u]);
                sc[u] = sc[u] + c;
                sw[u] = sw[u] + v;
                scc[u] = scc[u] + c * c;
                scw[u] = scw[u] + c * v;
            }
            sn[u] += static_cast<double>(__popcll(__ballot(use[u])));  // (exact in any order)
        }
    }
    // row r of 16 lanes holds group {0, 2, 1, 3}[r]; its first lane solves it
    const double a = wave_sum4_f64(sc), b = wave_sum4_f64(sw), aa = wave_sum4_f64(scc), ab = wave_sum4_f64(scw);
    const int row = lane >> 4;
    const int u = (row >> 1) | ((row & 1) << 1);
    const double n = u == 0 ? sn[0] : u == 1 ? sn[1] : u == 2 ? sn[2] : sn[3];
    if ((lane & 15) == 0 && u0 + u < units) {
        double s = 1.0, o = 0.0;
        const double det = n * aa - a * a;
        if (n >= 2.0 && det > 0.0) {
            s = (n * ab - a * b) / det;
            o = (b - s * a) / n;
        } else if (n > 0.0) {
            o = (b - a) / n;
        }
        scale[u0 + u] = static_cast<float>(s);
        offset[u0 + u] = static_cast<float>(o);
    }
}

static int grid_for(int64_t n) {
    const int64_t g = (n + kThreads - 1) / kThreads;
    return static_cast<int>(std::min<int64_t>(std::max<int64_t>(g, 1), 8192));
}

// ---------------------------------------------------------------------------
// pair (vector_dim 2) codebook: nearest centroid and centroid update
// ---------------------------------------------------------------------------
// The reference's numpy arithmetic (hxq_encoder.py:280-300):
//   d_j = fl(fl(|x|^2 + |c_j|^2) - 2 x.c_j), |v|^2 = fl(fl(v0*v0) + fl(v1*v1)),
//   x.c = fma(x1, c1, fl(x0*c0)) (what numpy's sgemm gives a K = 2 product),
//   first index of the minimum;  new c_j = fp32(fp64 sum / fp32 count).
// 2 x.c is exact, so fl(t - fl(2 x.c)) is the single rounding fma(-2, x.c, t).
constexpr int kPairMaxK = 4096;
constexpr int kPairThreads = 512;
constexpr int kUpdThreads = 1024;     // one owner thread per cluster id mod 1024
constexpr int kUpdChunk = 1024;       // ids staged in LDS per pass
constexpr int kUpdMaxBlocks = 512;
constexpr int kUpdSlots = kPairMaxK / kUpdThreads;

// {c0, c1, |c|^2, 0} per centroid.
__global__ __launch_bounds__(256) void pair_table_kernel(const float *__restrict__ cb, int k,
                                                         float4 *__restrict__ tab) {
#pragma clang fp contract(off)
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < k) {
        const float c0 = cb[2 * j], c1 = cb[2 * j + 1];
        tab[j] = make_float4(c0, c1, c0 * c0 + c1 * c1, 0.0f);
    }
}

// V pairs per thread (pair i = block base + threadIdx.x + v * kPairThreads);
// the table is staged once per block in LDS and read as a broadcast.
// MIN: writes dmin[i] = max(min_j d_j, 0) instead of the index (the k-means++
// seeding distance, np.maximum(d, 0).min(axis=1)), for the rows rows[i] of x
// when rows is given (an out-of-range row gives NaN).
template <int V, bool MIN>
__global__ __launch_bounds__(kPairThreads) void pair_assign_kernel(
    const float2 *__restrict__ x, int64_t n, const int64_t *__restrict__ rows, int64_t m,
    const float4 *__restrict__ tab, int k, uint16_t *__restrict__ idx, float *__restrict__ dmin) {
#pragma clang fp contract(off)
    extern __shared__ float4 stab[];
    for (int j = threadIdx.x; j < k; j += kPairThreads) stab[j] = tab[j];
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * (kPairThreads * V) + threadIdx.x;
    float x0[V], x1[V], xsq[V], best[V];
    int bj[V];
    const float4 c = stab[0];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int64_t i = base + static_cast<int64_t>(v) * kPairThreads;
        int64_t r = i;
        if (MIN && rows != nullptr && i < m) r = rows[i];
        float2 p = make_float2(0.0f, 0.0f);
        if (i < m) p = (r >= 0 && r < n) ? x[r] : make_float2(NAN, NAN);
        x0[v] = p.x;
        x1[v] = p.y;
        xsq[v] = p.x * p.x + p.y * p.y;
        best[v] = fmaf(-2.0f, fmaf(x1[v], c.y, x0[v] * c.x), xsq[v] + c.z);
        bj[v] = 0;
    }
    if constexpr (MIN) {
        for (int j = 1; j < k; ++j) {
            const float4 cj = stab[j];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const float d = fmaf(-2.0f, fmaf(x1[v], cj.y, x0[v] * cj.x), xsq[v] + cj.z);
                if (d < best[v]) best[v] = d;
            }
        }
    } else {
        // Entries in groups of 8: the group's minimum (fminf skips NaN, as the
        // strict compare does) replaces the best only if strictly smaller, and
        // only then is its first index looked up -- the same (value, first
        // index) as a strict-compare scan, with the index work done on the
        // few groups that improve.  Entries past k read entry k - 1 again; it
        // sits earlier in the same group, so a tie never picks the copy.
        for (int j0 = 1; j0 < k; j0 += 8) {
            float4 cg[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) cg[t] = stab[min(j0 + t, k - 1)];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                float d[8];
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    d[t] = fmaf(-2.0f, fmaf(x1[v], cg[t].y, x0[v] * cg[t].x), xsq[v] + cg[t].z);
                const float g = fminf(fminf(fminf(d[0], d[1]), fminf(d[2], d[3])),
                                      fminf(fminf(d[4], d[5]), fminf(d[6], d[7])));
                if (g < best[v]) {
                    int at = j0 + 7;
#pragma unroll
                    for (int t = 6; t >= 0; --t) at = d[t] == g ? j0 + t : at;
                    best[v] = g;
                    bj[v] = at;
                }
            }
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int64_t i = base + static_cast<int64_t>(v) * kPairThreads;
        if (i < m) {
            if (MIN)
                dmin[i] = best[v] >= 0.0f || best[v] != best[v] ? best[v] : 0.0f;
            else
                idx[i] = static_cast<uint16_t>(bj[v]);
        }
    }
}

// fp64 sums and counts per cluster over one block's range of pairs.  Thread
// t = 64 * wave + lane owns the ids with id % 1024 == t and adds their pairs
// in index order, so the partials do not depend on timing.  The ids are
// wave-uniform (read from LDS, made scalar), so the owner test is a scalar
// branch and only the owning lane does vector work.  Block 0 clears
// *max_delta for the finish kernel that follows on the stream.
__global__ __launch_bounds__(kUpdThreads) void pair_partial_kernel(
    const float2 *__restrict__ x, int64_t n, const uint16_t *__restrict__ idx, int k,
    int64_t per_block, double *__restrict__ psum, uint32_t *__restrict__ pcnt,
    float *__restrict__ max_delta) {
    __shared__ uint16_t sidx[kUpdChunk];
    __shared__ float2 sx[kUpdChunk];
    const int t = threadIdx.x;
    const int wave = t >> 6, lane = t & 63;
    if (blockIdx.x == 0 && t == 0) *max_delta = 0.0f;
    double s0[kUpdSlots], s1[kUpdSlots];
    uint32_t cnt[kUpdSlots];
#pragma unroll
    for (int s = 0; s < kUpdSlots; ++s) {
        s0[s] = 0.0;
        s1[s] = 0.0;
        cnt[s] = 0;
    }
    const int64_t lo = static_cast<int64_t>(blockIdx.x) * per_block;
    const int64_t hi = lo + per_block < n ? lo + per_block : n;
    for (int64_t b = lo; b < hi; b += kUpdChunk) {
        const int m = static_cast<int>(hi - b < kUpdChunk ? hi - b : kUpdChunk);
        __syncthreads();
        if (t < m) {
            sidx[t] = idx[b + t];
            sx[t] = x[b + t];
        }
        __syncthreads();
        for (int i = 0; i < m; ++i) {
            const int id = __builtin_amdgcn_readfirstlane(static_cast<int>(sidx[i]));
            if (((id >> 6) & 15) != wave) continue;
            if (lane != (id & 63)) continue;
            const float2 v = sx[i];
            const int slot = id >> 10;
#pragma unroll
            for (int s = 0; s < kUpdSlots; ++s) {
                if (slot == s) {
                    s0[s] += static_cast<double>(v.x);
                    s1[s] += static_cast<double>(v.y);
                    cnt[s] += 1;
                }
            }
        }
    }
#pragma unroll
    for (int s = 0; s < kUpdSlots; ++s) {
        const int j = s * kUpdThreads + t;
        if (j < k) {
            psum[(2 * static_cast<int64_t>(blockIdx.x)) * k + j] = s0[s];
            psum[(2 * static_cast<int64_t>(blockIdx.x) + 1) * k + j] = s1[s];
            pcnt[static_cast<int64_t>(blockIdx.x) * k + j] = cnt[s];
        }
    }
}

// Adds the block partials in a fixed order (wave w of 16 takes blocks w,
// w + 16, ... in turn; the 16 wave totals are then added in wave order),
// writes the new centroids (empty clusters keep the old one) and raises
// *max_delta to max |new - old| (non-negative floats order as their bits).
__global__ __launch_bounds__(1024) void pair_finish_kernel(
    const double *__restrict__ psum, const uint32_t *__restrict__ pcnt, int nparts, int k,
    const float *__restrict__ old, float *__restrict__ out, float *__restrict__ max_delta) {
    __shared__ double l0[16][64], l1[16][64];
    __shared__ uint32_t lc[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + lane;
    double a0 = 0.0, a1 = 0.0;
    uint32_t c = 0;
    if (j < k) {
        for (int p = w; p < nparts; p += 16) {
            a0 += psum[(2 * static_cast<int64_t>(p)) * k + j];
            a1 += psum[(2 * static_cast<int64_t>(p) + 1) * k + j];
            c += pcnt[static_cast<int64_t>(p) * k + j];
        }
    }
    l0[w][lane] = a0;
    l1[w][lane] = a1;
    lc[w][lane] = c;
    __syncthreads();
    if (w != 0) return;
    float dmax = 0.0f;
    if (j < k) {
        double t0 = 0.0, t1 = 0.0;
        uint32_t tc = 0;
        for (int q = 0; q < 16; ++q) {
            t0 += l0[q][lane];
            t1 += l1[q][lane];
            tc += lc[q][lane];
        }
        const float o0 = old[2 * j], o1 = old[2 * j + 1];
        float n0 = o0, n1 = o1;
        if (tc > 0) {
            const double fc = static_cast<double>(static_cast<float>(tc));
            n0 = static_cast<float>(t0 / fc);
            n1 = static_cast<float>(t1 / fc);
        }
        out[2 * j] = n0;
        out[2 * j + 1] = n1;
        dmax = fmaxf(fabsf(n0 - o0), fabsf(n1 - o1));
    }
    for (int off = 32; off > 0; off >>= 1) dmax = fmaxf(dmax, __shfl_xor(dmax, off));
    if (lane == 0 && dmax > 0.0f)
        atomicMax(reinterpret_cast<unsigned int *>(max_delta), __float_as_uint(dmax));
}

struct PairPlan {
    int64_t per_block;
    int64_t nparts;
};

static PairPlan pair_plan(int64_t n) {
    PairPlan p;
    int64_t per = (n + kUpdMaxBlocks - 1) / kUpdMaxBlocks;
    per = (per + kUpdChunk - 1) / kUpdChunk * kUpdChunk;
    p.per_block = per < kUpdChunk ? kUpdChunk : per;
    p.nparts = n <= 0 ? 1 : (n + p.per_block - 1) / p.per_block;
    return p;
}


}  // namespace enc
}  // namespace hxq

using namespace hxq;
using namespace hxq::enc;

template <typename IT, int KM>
static int assign_nearest_impl(const float *x, int64_t n, const float *codebook, int32_t k,
                               IT *indices, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && codebook && indices, "x, codebook and indices are required");
    HXQ_REQUIRE(n >= 0 && k >= 1 && k <= KM, KM == kMaxK ? "k must be 1..256" : "k must be 1..4096");
    if (n == 0) return HXQ_OK;
    // eight blocks per CU: one staging of the codebook for many weights
    const int64_t blocks = (n + kThreads * kAssignV - 1) / (kThreads * kAssignV);
    const int vec = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(indices)) & 15u) == 0;
    hipLaunchKernelGGL((assign_kernel<IT, KM>), dim3(static_cast<uint32_t>(std::min<int64_t>(blocks, 8 * device_cu_count()))),
                       dim3(kThreads), 0, stream, x, n, codebook, k, indices, vec);
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

extern "C" int hxq_assign_nearest(const float *x, int64_t n, const float *codebook, int32_t k,
                                  uint8_t *indices, hipStream_t stream) {
    return assign_nearest_impl<uint8_t, kMaxK>(x, n, codebook, k, indices, stream);
}

extern "C" int hxq_assign_nearest_wide(const float *x, int64_t n, const float *codebook, int32_t k,
                                       uint16_t *indices, hipStream_t stream) {
    return assign_nearest_impl<uint16_t, kMaxKW>(x, n, codebook, k, indices, stream);
}

extern "C" int64_t hxq_sort_workspace_bytes(int64_t n) {
    if (n <= 0) return 0;
    int64_t p = 2048;
    while (p < n) p <<= 1;
    return 4 * p;
}

// Four 8-bit passes between keys and tmp (n keys each), ending in keys.
static int sort_keys(const float *x, int64_t n, uint32_t *keys, uint32_t *tmp, int32_t *blk, int32_t *counts,
                     hipStream_t stream) {
    const int64_t nblk = (n + kPer - 1) / kPer;
    const dim3 grid(static_cast<uint32_t>(nblk));
    for (int pass = 0; pass < 4; ++pass) {
        const DigitSrc src{pass == 0 ? x : nullptr, pass & 1 ? tmp : keys, 8 * pass};
        hipLaunchKernelGGL(digit_count_kernel, grid, dim3(kThreads), 0, stream, src, n, nblk, blk);
        HXQ_LAUNCH_CHECK();
        hipLaunchKernelGGL(bucket_scan_kernel, dim3(kDigits / kWaves), dim3(kThreads), 0, stream, blk, nblk,
                           kDigits, counts, nullptr);
        HXQ_LAUNCH_CHECK();
        hipLaunchKernelGGL((bucket_scatter_kernel<DigitSrc, kDigits>), grid, dim3(kThreads), 0, stream, src, n,
                           nblk, kDigits, blk, counts, pass & 1 ? keys : tmp, nullptr);
        HXQ_LAUNCH_CHECK();
    }
    return HXQ_OK;
}

static int64_t align256(int64_t b) { return (b + 255) & ~int64_t{255}; }

// k-means workspace regions, each 256-byte aligned: sort keys, cluster-ordered
// values (the sort's second buffer), per-block counts / offsets, then counts,
// means, the fp64 tolerance, the done flag and the arrival counter
struct KmLayout {
    int64_t vals, blk, counts, means, tol, done, total;
    explicit KmLayout(int64_t n) {
        const int64_t nblk = (n + kPer - 1) / kPer;
        vals = align256(4 * n);
        blk = vals + align256(4 * n);
        counts = blk + align256(4 * nblk * kMaxKW);
        means = counts + 4 * kMaxKW;
        tol = means + 4 * kMaxKW;
        done = tol + 8;
        total = align256(done + 8);
    }
};

extern "C" int64_t hxq_kmeans_workspace_bytes(int64_t n) {
    return n <= 0 ? 0 : KmLayout(n).total;
}

extern "C" int hxq_kmeans_init(const float *x, int64_t n, void *workspace, int64_t workspace_bytes,
                               int32_t *n_unique, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && workspace && n_unique && n >= 1, "bad arguments");
    HXQ_REQUIRE(n < (int64_t{1} << 31), "n too large");
    HXQ_REQUIRE(workspace_bytes >= hxq_kmeans_workspace_bytes(n), "workspace too small");
    char *ws = static_cast<char *>(workspace);
    const KmLayout lay(n);
    uint32_t *keys = reinterpret_cast<uint32_t *>(ws);
    if (int rc = sort_keys(x, n, keys, reinterpret_cast<uint32_t *>(ws + lay.vals),
                           reinterpret_cast<int32_t *>(ws + lay.blk),
                           reinterpret_cast<int32_t *>(ws + lay.counts), stream))
        return rc;
    hipLaunchKernelGGL(zero_i32_kernel, dim3(1), dim3(1), 0, stream, n_unique);
    HXQ_LAUNCH_CHECK();
    hipLaunchKernelGGL(count_unique_kernel, dim3(std::min(grid_for(n), 128)), dim3(kThreads), 0, stream, keys,
                       n, n_unique);
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

template <typename IT, int KM>
static int kmeans_run_impl(const float *x, int64_t n, const double *percentiles01, int32_t k,
                           int32_t max_iters, double rtol, void *workspace, int64_t workspace_bytes,
                           float *codebook, IT *assignments, int32_t *iters, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && percentiles01 && workspace && codebook && assignments && iters, "bad arguments");
    // max_iters == 0 leaves the reference's assignments unbound (an error there)
    HXQ_REQUIRE(n >= 1 && n < (int64_t{1} << 31) && k >= 1 && k <= KM && max_iters >= 1,
                KM == kMaxK ? "bad sizes (n 1..2^31-1, k 1..256, max_iters >= 1)"
                            : "bad sizes (n 1..2^31-1, k 1..4096, max_iters >= 1)");
    HXQ_REQUIRE(workspace_bytes >= hxq_kmeans_workspace_bytes(n), "workspace too small");
    char *ws = static_cast<char *>(workspace);
    const int64_t nblk = (n + kPer - 1) / kPer;
    const KmLayout lay(n);
    uint32_t *keys = reinterpret_cast<uint32_t *>(ws);              // sorted by hxq_kmeans_init
    float *vals = reinterpret_cast<float *>(ws + lay.vals);
    int32_t *blk = reinterpret_cast<int32_t *>(ws + lay.blk);
    int32_t *counts = reinterpret_cast<int32_t *>(ws + lay.counts);
    float *means = reinterpret_cast<float *>(ws + lay.means);
    double *abs_tol = reinterpret_cast<double *>(ws + lay.tol);
    int32_t *done = reinterpret_cast<int32_t *>(ws + lay.done);
    int32_t *arrived = done + 1;
    hipLaunchKernelGGL(kmeans_init_kernel, dim3(1), dim3(kMaxK), 0, stream, keys, n, percentiles01,
                       k, codebook, rtol, abs_tol, done, iters, arrived);
    HXQ_LAUNCH_CHECK();
    const dim3 grid(static_cast<uint32_t>(nblk));
    const ClusterSrc<IT> src{x, assignments};
    // four launches a step: 34 us at 500K values and 256 clusters (190 us with
    // one thread scanning the blocks of a cluster, 64 shuffles per element's
    // rank, one thread per leaf of the means)
    for (int it = 0; it < max_iters; ++it) {
        hipLaunchKernelGGL((km_assign_kernel<IT, KM>), grid, dim3(kThreads), 0, stream, x, n, nblk, codebook, k,
                           assignments, blk, done);
        HXQ_LAUNCH_CHECK();
        hipLaunchKernelGGL(bucket_scan_kernel, dim3((k + kWaves - 1) / kWaves), dim3(kThreads), 0, stream, blk,
                           nblk, k, counts, done);
        HXQ_LAUNCH_CHECK();
        hipLaunchKernelGGL((bucket_scatter_kernel<ClusterSrc<IT>, KM>), grid, dim3(kThreads), 0, stream, src, n,
                           nblk, k, blk, counts, reinterpret_cast<uint32_t *>(vals), done);
        HXQ_LAUNCH_CHECK();
        hipLaunchKernelGGL(km_sum_kernel<KM>, dim3(k), dim3(kThreads), 0, stream, vals, counts, k, codebook,
                           means, abs_tol, done, iters, arrived);
        HXQ_LAUNCH_CHECK();
    }
    return HXQ_OK;
}

extern "C" int hxq_kmeans_run(const float *x, int64_t n, const double *percentiles01, int32_t k,
                              int32_t max_iters, double rtol, void *workspace,
                              int64_t workspace_bytes, float *codebook, uint8_t *assignments,
                              int32_t *iters, hipStream_t stream) {
    return kmeans_run_impl<uint8_t, kMaxK>(x, n, percentiles01, k, max_iters, rtol, workspace,
                                           workspace_bytes, codebook, assignments, iters, stream);
}

extern "C" int hxq_kmeans_run_wide(const float *x, int64_t n, const double *percentiles01, int32_t k,
                                   int32_t max_iters, double rtol, void *workspace,
                                   int64_t workspace_bytes, float *codebook, uint16_t *assignments,
                                   int32_t *iters, hipStream_t stream) {
    return kmeans_run_impl<uint16_t, kMaxKW>(x, n, percentiles01, k, max_iters, rtol, workspace,
                                             workspace_bytes, codebook, assignments, iters, stream);
}

extern "C" int64_t hxq_select_workspace_bytes(void) { return sizeof(SelState); }

extern "C" int hxq_select_f32(const float *x, int64_t n, const int64_t *ranks, int32_t m,
                              float *values, int32_t *nan_count, void *workspace,
                              int64_t workspace_bytes, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && ranks && values && workspace, "bad arguments");
    HXQ_REQUIRE(m >= 1 && m <= kSelMax && n >= 1 && n < (int64_t{1} << 32), "bad sizes");
    HXQ_REQUIRE(workspace_bytes >= static_cast<int64_t>(sizeof(SelState)), "workspace too small");
    SelState *st = static_cast<SelState *>(workspace);
    hipLaunchKernelGGL(select_init_kernel, dim3(1), dim3(256), 0, stream, ranks, m, st);
    HXQ_LAUNCH_CHECK();
    // two blocks of 16 waves per CU: the histograms (32 KB of LDS) are added up
    // once per block
    const int64_t blocks = (n + kSelThreads * 8 - 1) / (kSelThreads * 8);
    const dim3 grid(static_cast<uint32_t>(std::min<int64_t>(blocks, 2 * device_cu_count())));
    const int vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    for (int pass = 0; pass < 3; ++pass) {
        hipLaunchKernelGGL(select_pass_kernel, grid, dim3(kSelThreads), 0, stream, x, n, m, pass, vec, st, values);
        HXQ_LAUNCH_CHECK();
    }
    if (nan_count)
        HXQ_HIP_TRY(hipMemcpyAsync(nan_count, &st->nan_count, 4, hipMemcpyDeviceToDevice, stream));
    return HXQ_OK;
}

extern "C" int64_t hxq_outliers_workspace_bytes(int64_t n) {
    return 8 * std::max<int64_t>((n + kChunk - 1) / kChunk, 1) + 64;  // 64: alignment
}

extern "C" int hxq_outliers_f32(const float *x, int64_t n, const float *lohi, int64_t capacity,
                                int64_t *positions, float *values, int64_t *count, void *workspace,
                                int64_t workspace_bytes, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && lohi && count && workspace && (capacity == 0 || (positions && values)),
                "bad arguments");
    HXQ_REQUIRE(n >= 1 && capacity >= 0, "bad sizes");
    HXQ_REQUIRE(workspace_bytes >= hxq_outliers_workspace_bytes(n), "workspace too small");
    const int64_t chunks = (n + kChunk - 1) / kChunk;
    const dim3 grid(static_cast<uint32_t>((chunks + kWaves - 1) / kWaves));
    HXQ_REQUIRE((chunks + kWaves - 1) / kWaves < (int64_t{1} << 31), "n too large");
    const int vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    // (any alignment: the counts start at the next multiple of 8, in the spare bytes)
    int64_t *cnt = reinterpret_cast<int64_t *>((reinterpret_cast<uintptr_t>(workspace) + 7u) & ~uintptr_t{7});
    hipLaunchKernelGGL(outlier_count_kernel, grid, dim3(kThreads), 0, stream, x, n, chunks, vec, lohi, cnt);
    HXQ_LAUNCH_CHECK();
    hipLaunchKernelGGL(outlier_scan_kernel, dim3(1), dim3(1024), 0, stream, cnt, chunks, count);
    HXQ_LAUNCH_CHECK();
    if (capacity > 0) {
        hipLaunchKernelGGL(outlier_write_kernel, grid, dim3(kThreads), 0, stream, x, n, chunks, vec, lohi, cnt,
                           capacity, positions, values);
        HXQ_LAUNCH_CHECK();
    }
    return HXQ_OK;
}

extern "C" int64_t hxq_affine_fit_workspace_bytes(int64_t rows, int64_t cols) {
    return rows <= 0 || cols <= 0 ? 0 : 4 * ((rows * cols + 31) / 32);
}

template <typename IT, int KM>
static int affine_fit_impl(const float *w, const IT *indices, const float *codebook, int32_t k,
                           int64_t rows, int64_t cols, int32_t group_size,
                           const int64_t *exclude_positions, int64_t n_exclude, void *workspace,
                           int64_t workspace_bytes, float *scale, float *offset, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(w && indices && codebook && scale && offset, "bad arguments");
    HXQ_REQUIRE(k >= 1 && k <= KM && rows >= 1 && cols >= 1,
                KM == kMaxK ? "bad sizes (k 1..256)" : "bad sizes (k 1..4096)");
    HXQ_REQUIRE(group_size >= 1 && cols % group_size == 0, "cols must be a multiple of group_size");
    HXQ_REQUIRE(n_exclude >= 0 && (n_exclude == 0 || exclude_positions), "bad exclusion list");
    uint32_t *bits = nullptr;
    if (n_exclude > 0) {
        HXQ_REQUIRE(workspace && workspace_bytes >= hxq_affine_fit_workspace_bytes(rows, cols),
                    "workspace too small");
        bits = static_cast<uint32_t *>(workspace);
        const int64_t words = (rows * cols + 31) / 32;
        hipLaunchKernelGGL(zero_u32_kernel, dim3(grid_for(words)), dim3(kThreads), 0, stream, bits,
                           words);
        HXQ_LAUNCH_CHECK();
        hipLaunchKernelGGL(mark_kernel, dim3(grid_for(n_exclude)), dim3(kThreads), 0, stream,
                           exclude_positions, n_exclude, bits);
        HXQ_LAUNCH_CHECK();
    }
    const int64_t units = rows * (cols / group_size);
    const int64_t per_block = kWaves * kFitUnits;
    const int64_t blocks = (units + per_block - 1) / per_block;
    HXQ_REQUIRE(blocks < (int64_t{1} << 31), "too many groups");
    hipLaunchKernelGGL((affine_fit_kernel<IT, KM>), dim3(static_cast<uint32_t>(blocks)), dim3(kThreads),
                       0, stream, w, indices, codebook, k, rows, cols, group_size, bits, scale, offset);
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

extern "C" int hxq_affine_fit(const float *w, const uint8_t *indices, const float *codebook,
                              int32_t k, int64_t rows, int64_t cols, int32_t group_size,
                              const int64_t *exclude_positions, int64_t n_exclude, void *workspace,
                              int64_t workspace_bytes, float *scale, float *offset,
                              hipStream_t stream) {
    return affine_fit_impl<uint8_t, kMaxK>(w, indices, codebook, k, rows, cols, group_size,
                                           exclude_positions, n_exclude, workspace, workspace_bytes,
                                           scale, offset, stream);
}

extern "C" int hxq_affine_fit_wide(const float *w, const uint16_t *indices, const float *codebook,
                                   int32_t k, int64_t rows, int64_t cols, int32_t group_size,
                                   const int64_t *exclude_positions, int64_t n_exclude,
                                   void *workspace, int64_t workspace_bytes, float *scale,
                                   float *offset, hipStream_t stream) {
    return affine_fit_impl<uint16_t, kMaxKW>(w, indices, codebook, k, rows, cols, group_size,
                                             exclude_positions, n_exclude, workspace,
                                             workspace_bytes, scale, offset, stream);
}

extern "C" int64_t hxq_vq2_workspace_bytes(int64_t n, int32_t k) {
    if (n < 0 || k < 1 || k > kPairMaxK) return -1;
    const PairPlan p = pair_plan(n);
    return align256(int64_t{16} * k) + align256(p.nparts * 16 * k) + align256(p.nparts * 4 * k);
}

static int pair_table(const float *codebook, int32_t k, float4 *tab, hipStream_t stream) {
    hipLaunchKernelGGL(pair_table_kernel, dim3((k + 255) / 256), dim3(256), 0, stream, codebook, k,
                       tab);
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

template <bool MIN>
static int pair_launch(const float2 *x, int64_t n, const int64_t *rows, int64_t m,
                       const float4 *tab, int32_t k, uint16_t *indices, float *dmin,
                       hipStream_t stream) {
    const size_t lds = static_cast<size_t>(k) * sizeof(float4);
    const int64_t big = (m + kPairThreads * 8 - 1) / (kPairThreads * 8);
    if (big >= 1024) {
        HXQ_REQUIRE(big < (int64_t{1} << 31), "too many pairs");
        hipLaunchKernelGGL((pair_assign_kernel<8, MIN>), dim3(static_cast<uint32_t>(big)),
                           dim3(kPairThreads), lds, stream, x, n, rows, m, tab, k, indices, dmin);
    } else {
        const int64_t g = (m + kPairThreads * 2 - 1) / (kPairThreads * 2);
        hipLaunchKernelGGL((pair_assign_kernel<2, MIN>), dim3(static_cast<uint32_t>(g)),
                           dim3(kPairThreads), lds, stream, x, n, rows, m, tab, k, indices, dmin);
    }
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}

extern "C" int hxq_vq2_assign(const float *x, int64_t n, const float *codebook, int32_t k,
                              uint16_t *indices, void *workspace, int64_t workspace_bytes,
                              hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && codebook && indices && workspace, "x, codebook, indices and workspace are required");
    HXQ_REQUIRE(n >= 0 && k >= 1 && k <= kPairMaxK, "k must be 1..4096");
    HXQ_REQUIRE(workspace_bytes >= int64_t{16} * k, "workspace too small");
    if (n == 0) return HXQ_OK;
    float4 *tab = static_cast<float4 *>(workspace);
    const int rc = pair_table(codebook, k, tab, stream);
    if (rc != HXQ_OK) return rc;
    return pair_launch<false>(reinterpret_cast<const float2 *>(x), n, nullptr, n, tab, k, indices,
                              nullptr, stream);
}

extern "C" int hxq_vq2_min_dist(const float *x, int64_t n, const int64_t *rows, int64_t m,
                                const float *codebook, int32_t k, float *dmin, void *workspace,
                                int64_t workspace_bytes, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && codebook && dmin && workspace, "x, codebook, dmin and workspace are required");
    HXQ_REQUIRE(n >= 0 && m >= 0 && k >= 1 && k <= kPairMaxK, "k must be 1..4096");
    HXQ_REQUIRE(rows != nullptr || m <= n, "without rows, m must be <= n");
    HXQ_REQUIRE(workspace_bytes >= int64_t{16} * k, "workspace too small");
    if (m == 0) return HXQ_OK;
    float4 *tab = static_cast<float4 *>(workspace);
    const int rc = pair_table(codebook, k, tab, stream);
    if (rc != HXQ_OK) return rc;
    return pair_launch<true>(reinterpret_cast<const float2 *>(x), n, rows, m, tab, k, nullptr, dmin,
                             stream);
}

extern "C" int hxq_vq2_update(const float *x, int64_t n, const uint16_t *indices, int32_t k,
                              const float *centroids, float *new_centroids, float *max_delta,
                              void *workspace, int64_t workspace_bytes, hipStream_t stream) {
    clear_error();
    HXQ_REQUIRE(x && indices && centroids && new_centroids && max_delta && workspace,
                "x, indices, centroids, new_centroids, max_delta and workspace are required");
    HXQ_REQUIRE(n >= 0 && k >= 1 && k <= kPairMaxK, "k must be 1..4096");
    HXQ_REQUIRE(workspace_bytes >= hxq_vq2_workspace_bytes(n, k), "workspace too small");
    HXQ_REQUIRE(new_centroids != centroids, "new_centroids must not alias centroids");
    const PairPlan p = pair_plan(n);
    char *ws = static_cast<char *>(workspace) + align256(int64_t{16} * k);
    double *psum = reinterpret_cast<double *>(ws);
    uint32_t *pcnt = reinterpret_cast<uint32_t *>(ws + align256(p.nparts * 16 * k));
    hipLaunchKernelGGL(pair_partial_kernel, dim3(static_cast<uint32_t>(p.nparts)),
                       dim3(kUpdThreads), 0, stream, reinterpret_cast<const float2 *>(x), n,
                       indices, k, p.per_block, psum, pcnt, max_delta);
    HXQ_LAUNCH_CHECK();
    hipLaunchKernelGGL(pair_finish_kernel, dim3((k + 63) / 64), dim3(1024), 0, stream, psum, pcnt,
                       static_cast<int>(p.nparts), k, centroids, new_centroids, max_delta);
    HXQ_LAUNCH_CHECK();
    return HXQ_OK;
}
