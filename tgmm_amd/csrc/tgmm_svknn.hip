// tgmm_svknn.hip -- supervoxel nearest neighbours (knnCUDA_,
// temporalLogicalRules/knnCUDA/knnCuda.cu:142-232 with its kernel :56-140):
// for each query centroid, the K <= 11 nearest reference centroids under the
// scaled squared distance, in the reference's slot layout. The tracker calls
// it three times per frame (supervoxels against themselves, the previous and
// the next frame; mainTrackingGaussianMixtureModel.cpp:874-888,
// lineageHyperTree.cpp:2526-2775) and reads the slots in order.
//
// The slot layout is the outcome of a scan of the references in index
// order: a reference whose distance is not above the current threshold (the
// largest slot distance) replaces the first slot holding it. The kernel
// replays that scan exactly, but a wave looks only at the references that
// can matter to its queries:
//   - the queries are sorted along a Morton curve of cells, so that a wave's
//     queries lie close together (their order changes no result: each query
//     is its own scan);
//   - a reference farther from the box around the wave's queries than the
//     largest of their thresholds is dropped. Per axis the gap between the
//     reference and the box is no larger than |q - r| of any query in it, and
//     the bound is formed with the distance's own float operations in the
//     same order, so by monotonicity of rounding it never exceeds a member's
//     computed distance: the scan would not insert the reference. Blocks of
//     64 consecutive references are tested by their box first, 64 blocks at
//     once;
//   - the references left, still in index order, are collected in LDS 64 at
//     a time. Each lane marks, branch-free, those not above its threshold at
//     the start (a superset of the ones the scan inserts, since the threshold
//     only falls) and walks its marks in order with the exact test.
// Thresholds only fall, so a stale one only keeps more.
// With a coordinate that is not finite (or beyond 1e18) a distance can be NaN,
// and a NaN threshold takes any next reference: a wave with such a query, and
// every wave if a reference is such, walks the references with the
// reference's own test and slot update (scan_all). It leaves out a block of
// 64 that is farther from each of its queries than the query's threshold; a
// block that holds such a reference has an unbounded box and is always taken,
// as every block is for such a query.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <mutex>
#include <vector>

#include "../../include/tgmm_em.h"
#include "tgmm_runtime_internal.h"

namespace {

constexpr int kKB = 64;  // references per bounding box
constexpr int kKM = TGMM_SV_KNN_MAX;

constexpr int kCellBits = 5;    // Morton cells per axis: 32
constexpr int kCells = 1 << (3 * kCellBits);
constexpr int kKU = 4;          // blocks of references loaded together
constexpr int kMaxPacked = 1 << 27;  // reference indices that fit beside a slot number

// Written by the preparation kernels, cleared before: the largest ordered
// image of the query coordinates (hi) and of their complements (lo) per axis,
// and whether a reference's coordinate is not regular.
struct KnnPrep {
  unsigned hi[3], lo[3];
  unsigned irregular;
  unsigned pad;
};

// order-preserving image of a float
__device__ inline unsigned ordered(float v) {
  const unsigned u = __float_as_uint(v);
  return (u >> 31) ? ~u : (u | 0x80000000u);
}
__device__ inline float unordered(unsigned u) {
  return __uint_as_float((u >> 31) ? (u & 0x7fffffffu) : ~u);
}
__device__ inline bool regular(float v) { return fabsf(v) <= 1e18f; }

// Bounding box of each block of 64 references (box[a][b] = min, box[3+a][b]
// = max of coordinate a; unbounded with an irregular coordinate), and, in the
// blocks after, the queries' extent.
__global__ __launch_bounds__(kKB) void k_svknn_boxes(const float* __restrict__ ref, int R,
                                                     int Rp, int nblk, float* __restrict__ box,
                                                     const float* __restrict__ query, long long Q,
                                                     KnnPrep* prep) {
  const int b = blockIdx.x;
  float lo[3], hi[3];
  bool bad = false;
  if (b < nblk) {
    const int r = b * kKB + threadIdx.x;
    for (int a = 0; a < 3; a++) {
      const float v = r < R ? ref[r + (long long)a * Rp] : 0.0f;
      lo[a] = r < R ? v : INFINITY;
      hi[a] = r < R ? v : -INFINITY;
      bad |= !regular(v);
    }
  } else {
    for (int a = 0; a < 3; a++) {
      lo[a] = INFINITY;
      hi[a] = -INFINITY;
    }
    const long long step = (long long)(gridDim.x - nblk) * kKB;
    for (long long q = (long long)(b - nblk) * kKB + threadIdx.x; q < Q; q += step)
      for (int a = 0; a < 3; a++) {
        const float v = query[q + a * Q];
        if (regular(v)) {
          lo[a] = fminf(lo[a], v);
          hi[a] = fmaxf(hi[a], v);
        }
      }
  }
  for (int m = 32; m >= 1; m >>= 1)
    for (int a = 0; a < 3; a++) {
      lo[a] = fminf(lo[a], __shfl_xor(lo[a], m, 64));
      hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], m, 64));
    }
  bad = __any(bad);
  if (threadIdx.x != 0) return;
  if (bad) atomicOr(&prep->irregular, 1u);
  for (int a = 0; a < 3; a++) {
    if (b < nblk) {
      box[(long long)a * nblk + b] = bad ? -INFINITY : lo[a];
      box[(long long)(3 + a) * nblk + b] = bad ? INFINITY : hi[a];
    } else if (lo[a] <= hi[a]) {
      atomicMax(&prep->hi[a], ordered(hi[a]));
      atomicMax(&prep->lo[a], ~ordered(lo[a]));
    }
  }
}

// Morton cell of a query: cubic cells in scaled coordinates, 32 along the
// longest extent.
__device__ inline int query_cell(const KnnPrep* prep, float x, float y, float z, float s0,
                                 float s1, float s2) {
  const float v[3] = {x, y, z}, s[3] = {fabsf(s0), fabsf(s1), fabsf(s2)};
  float ext = 0.0f, lo[3];
  for (int a = 0; a < 3; a++) {
    lo[a] = unordered(~prep->lo[a]);
    const float e = (unordered(prep->hi[a]) - lo[a]) * s[a];
    ext = e > ext ? e : ext;
  }
  int c = 0;
  for (int a = 0; a < 3; a++) {
    const float t = (v[a] - lo[a]) * s[a] * (float)(1 << kCellBits) / ext;
    int i = t > 0.0f ? (t < 31.0f ? (int)t : 31) : 0;  // NaN: 0
    for (int bit = 0; bit < kCellBits; bit++) c |= ((i >> bit) & 1) << (3 * bit + a);
  }
  return c;
}

// (the n queries of one piece; axes Q apart)
__global__ __launch_bounds__(256) void k_svknn_count(const float* __restrict__ query, long long n,
                                                     long long Q, float s0, float s1, float s2,
                                                     const KnnPrep* __restrict__ prep,
                                                     int* __restrict__ cell,
                                                     int* __restrict__ cnt) {
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  const int c = query_cell(prep, query[q], query[q + Q], query[q + 2 * Q], s0, s1, s2);
  cell[q] = c;
  atomicAdd(cnt + c, 1);
}

// exclusive scan of the kCells counts in place, one block
__global__ __launch_bounds__(1024) void k_svknn_scan(int* __restrict__ cnt) {
  constexpr int PT = kCells / 1024;  // entries per thread
  __shared__ int wsum[16];
  int4* p = reinterpret_cast<int4*>(cnt) + threadIdx.x * (PT / 4);
  int4 v[PT / 4];
  int sum = 0;
#pragma unroll
  for (int i = 0; i < PT / 4; i++) {
    v[i] = p[i];
    sum += v[i].x + v[i].y + v[i].z + v[i].w;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = sum;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  int at = x - sum;
  for (int i = 0; i < w; i++) at += wsum[i];
#pragma unroll
  for (int i = 0; i < PT / 4; i++) {
    int4 r;
    r.x = at;
    r.y = r.x + v[i].x;
    r.z = r.y + v[i].y;
    r.w = r.z + v[i].z;
    at = r.w + v[i].w;
    p[i] = r;
  }
}

__global__ __launch_bounds__(256) void k_svknn_scatter(const float* __restrict__ query,
                                                       long long n, long long Q,
                                                       const int* __restrict__ cell,
                                                       int* __restrict__ start,
                                                       float4* __restrict__ q4) {
  const long long q = (long long)blockIdx.x * 256 + threadIdx.x;
  if (q >= n) return;
  q4[atomicAdd(start + cell[q], 1)] =
      make_float4(query[q], query[q + Q], query[q + 2 * Q], __int_as_float((int)q));
}

// the reference's scaled squared distance, float, x then y then z, no contraction
__device__ inline float svdist(float q0, float q1, float q2, float4 r, float s0, float s1,
                               float s2) {
#pragma clang fp contract(off)
  float a = (q0 - r.x) * s0;
  float d = a * a;
  a = (q1 - r.y) * s1;
  d += a * a;
  a = (q2 - r.z) * s2;
  d += a * a;
  return d;
}

// The reference's insertion test (knnCuda.cu:103-113): it leaves a reference
// as soon as the x term, or the x + y partial sum, is above the threshold,
// and takes it when the full sum is not. For finite coordinates the partial
// sums are non-decreasing and only the full sum decides; a NaN makes the sums
// after it NaN (never above the threshold), so the partial sums before it
// still decide. Returns true with d = the full sum when the reference is
// taken.
__device__ inline bool svtake(float q0, float q1, float q2, float4 r, float s0, float s1,
                              float s2, float thr, float& d) {
#pragma clang fp contract(off)
  float a = (q0 - r.x) * s0;
  const float p1 = a * a;
  a = (q1 - r.y) * s1;
  const float p2 = p1 + a * a;
  a = (q2 - r.z) * s2;
  d = p2 + a * a;
  return !(p1 > thr) && !(p2 > thr) && !(d > thr);
}

// Lower bound of the computed distance from a reference to any query of the
// wave's box [lo, hi], from the per-axis gaps (each no larger than |q - r| of
// any of them), in the distance's operations.
__device__ inline float box_bound(float x, float y, float z, const float (&lo)[3],
                                  const float (&hi)[3], float s0, float s1, float s2) {
#pragma clang fp contract(off)
  float a = (x - __builtin_amdgcn_fmed3f(x, lo[0], hi[0])) * s0;
  float d = a * a;
  a = (y - __builtin_amdgcn_fmed3f(y, lo[1], hi[1])) * s1;
  d += a * a;
  a = (z - __builtin_amdgcn_fmed3f(z, lo[2], hi[2])) * s2;
  d += a * a;
  return d;
}
// the same from a box of references to the wave's box
__device__ inline float gap_bound(float g0, float g1, float g2, float s0, float s1, float s2) {
#pragma clang fp contract(off)
  float a = fmaxf(g0, 0.0f) * s0;
  float d = a * a;
  a = fmaxf(g1, 0.0f) * s1;
  d += a * a;
  a = fmaxf(g2, 0.0f) * s2;
  d += a * a;
  return d;
}

// Orders of the LDS accesses of one wave's lanes.
__device__ inline void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane exchanges within the four lanes of a query, as DPP moves.
constexpr int QL = 4;
__device__ inline int dpp_last(int v) {  // the group's last lane's value
  return __builtin_amdgcn_mov_dpp(v, 0xFF, 0xf, 0xf, true);
}
__device__ inline float dpp_last(float v) { return __int_as_float(dpp_last(__float_as_int(v))); }
__device__ inline int dpp_prev(int v) {  // the previous lane's (first lane: unused)
  return __builtin_amdgcn_mov_dpp(v, 0x111, 0xf, 0xf, true);
}
__device__ inline unsigned dpp_or(unsigned v) {  // OR over the group
  v |= (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true);
  v |= (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xf, 0xf, true);
  return v;
}

// The reference's scan (any coordinates) for query q4[i] of a group of L lanes,
// which split the marking of each 64.
template <int L>
__device__ __noinline__ void scan_all(const float4* __restrict__ q4, long long i, long long n,
                                      long long Q, const float* __restrict__ ref, int R, int Rp,
                                      int K,
                                      float s0, float s1, float s2,
                                      const float* __restrict__ box, int nblk,
                                      int* __restrict__ ind, float* __restrict__ dist) {
  const int sub = threadIdx.x % L;
  const bool live = i < n;
  const float4 qq = live ? q4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  const float q0 = qq.x, q1 = qq.y, q2 = qq.z;
  const long long q = __float_as_int(qq.w);
  // only a regular query's distances to a block's regular references are
  // bounded by its box
  const bool all = !(regular(q0) && regular(q1) && regular(q2) && regular(s0) && regular(s1) &&
                     regular(s2));
  float md[kKM];
  int mi[kKM];
#pragma unroll
  for (int j = 0; j < kKM; j++) {
    md[j] = 1e32f;
    mi[j] = -1;
  }
  float thr = live ? 1e32f : -INFINITY;  // a lane past the end inserts nothing
  int pos = 0;
  for (int b = 0; b < nblk; b++) {
    const float lb = gap_bound(fmaxf(box[b] - q0, q0 - box[3 * nblk + b]),
                               fmaxf(box[nblk + b] - q1, q1 - box[4 * nblk + b]),
                               fmaxf(box[2 * nblk + b] - q2, q2 - box[5 * nblk + b]), s0, s1, s2);
    if (!__any(all || !(lb > thr))) continue;  // no query of the wave takes any of it
    const int rb = b * kKB;
    const float t0 = thr;
    unsigned cl = 0u, ch = 0u;
#pragma unroll
    for (int v = 0; v < 64 / L; v++) {
      const int r = rb + v * L + sub;  // below Rp
      const float d =
          svdist(q0, q1, q2, make_float4(ref[r], ref[r + Rp], ref[r + 2 * Rp], 0.0f), s0, s1, s2);
      const unsigned bit = (d > t0) ? 0u : 1u << ((v * L + sub) & 31);
      if (v * L < 32)
        cl |= bit;
      else
        ch |= bit;
    }
    if constexpr (L > 1) {
      static_assert(L == QL, "one group size for the lane exchanges");
      cl = dpp_or(cl);
      ch = dpp_or(ch);
    }
    const unsigned long long nmask = R - rb < 64 ? (1ull << (R - rb)) - 1ull : ~0ull;
    unsigned long long cand = (((unsigned long long)ch << 32) | cl) & nmask;
    while (cand) {
      const int u = __builtin_ctzll(cand), r = rb + u;
      cand &= cand - 1ull;
      float d;
      if (!svtake(q0, q1, q2, make_float4(ref[r], ref[r + Rp], ref[r + 2 * Rp], 0.0f), s0, s1, s2,
                  thr, d))
        continue;
#pragma unroll
      for (int j = 0; j < kKM; j++)
        if (j == pos) {
          md[j] = d;
          mi[j] = r;
        }
      thr = md[0];
      pos = 0;
#pragma unroll
      for (int j = 1; j < kKM; j++)
        if (j < K && thr < md[j]) {
          thr = md[j];
          pos = j;
        }
      // a NaN in slot 0 makes the threshold NaN (findMaxPosition's `<` never
      // moves off it): the scan then takes the next reference, whatever its
      // distance, so the rest is walked
      if (thr != thr && u + 1 < 64) cand |= (~0ull << (u + 1)) & nmask;
    }
  }
  if (!live) return;
#pragma unroll
  for (int j = 0; j < kKM; j++)
    if (j < K && j % L == sub) {
      ind[q + j * Q] = mi[j];
      if (dist) dist[q + j * Q] = md[j];
    }
}

// Whether a distance to some reference may not be bounded by the boxes, or the
// references are too many to be packed: then every query is scanned for by
// scan_all, from kScanAlone queries on in a kernel of its own with a lane a
// query. Four lanes shorten the marking, one does more queries a wave of the
// walk over the marks, which is most of it, where there are 64-query waves for
// every SIMD: K = 10, one reference NaN / 1% of them, four lanes and one,
// 5,000 queries and references 0.76 / 1.03 and 0.86 / 1.15 ms a call, 100,000
// 7.7 / 26.9 and 6.95 / 15.9 (4.2 where all are regular). Beside the other
// form in one kernel its registers (64 references' loads together) cost that a
// tenth.
constexpr long long kScanAlone = 65536;
__device__ inline bool scans_all(const KnnPrep* prep, int R, float s0, float s1, float s2) {
  return prep->irregular != 0 || !regular(s0) || !regular(s1) || !regular(s2) || R >= kMaxPacked;
}

__global__ __launch_bounds__(64) void k_svknn_all(
    const float4* __restrict__ q4, long long n, long long Q, const float* __restrict__ ref, int R,
    int Rp, int K, float s0, float s1, float s2, const float* __restrict__ box, int nblk,
    const KnnPrep* __restrict__ prep, int* __restrict__ ind, float* __restrict__ dist) {
  if (scans_all(prep, R, s0, s1, s2))
    scan_all<1>(q4, (long long)blockIdx.x * 64 + threadIdx.x, n, Q, ref, R, Rp, K, s0, s1, s2, box,
                nblk, ind, dist);
}

// QL lanes share a query. ref is SoA with axis stride Rp = nblk * 64 (padded
// with zeros past R), q4 the sorted queries with their indices.
// The slots are kept sorted by distance over the group's lanes (E places a
// lane), each with its slot number beside its index: an insertion evicts the
// last and takes its slot, a median and three selects per place, with no
// search for the largest. Among equal largest distances the scan replaces the
// first slot, so a tie at the end first moves the lowest of their slots there
// (rare). The marking is split among the lanes too.
// What bounds it: VALU issue. In raster order the references come nearer
// slice by slice and a query inserts about 1,000 of 100,000, one after
// another; per wave and 64 references the box test is about 26 instructions,
// per reference kept the marking 12 / QL, per mark walked about 50, and a wave
// pays for its busiest query. More lanes a query shorten a wave's chain and
// split its insertions; fewer share the box test: 2, 4 lanes took 3.1, 2.2 ms
// (102,083 queries and references, K = 11), against 7.3 ms for one lane a
// query over blocks of 64 references skipped by their boxes alone; 5,208
// queries, 0.23 ms against 0.91.
__global__ __launch_bounds__(64) void k_svknn(
    const float4* __restrict__ q4, long long n, long long Q, const float* __restrict__ ref, int R,
    int Rp, int K, float s0, float s1, float s2, const float* __restrict__ box, int nblk,
    const KnnPrep* __restrict__ prep, int* __restrict__ ind, float* __restrict__ dist) {
#pragma clang fp contract(off)
  constexpr int E = 12 / QL;  // places per lane
  static_assert(kKM <= 12, "places");
  __shared__ float4 buf[64 + 64 * kKU];
  const int lane = threadIdx.x, sub = lane % QL;
  const long long i = (long long)blockIdx.x * (64 / QL) + lane / QL;
  const bool live = i < n;
  const float4 qq = live ? q4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  const float q0 = qq.x, q1 = qq.y, q2 = qq.z;
  const long long q = __float_as_int(qq.w);
  const bool every = scans_all(prep, R, s0, s1, s2);
  if (every && n >= kScanAlone) return;
  if (every || __any(!regular(q0) || !regular(q1) || !regular(q2))) {
    scan_all<QL>(q4, i, n, Q, ref, R, Rp, K, s0, s1, s2, box, nblk, ind, dist);
    return;
  }
  // the box around the wave's queries
  float lo[3] = {live ? q0 : INFINITY, live ? q1 : INFINITY, live ? q2 : INFINITY};
  float hi[3] = {live ? q0 : -INFINITY, live ? q1 : -INFINITY, live ? q2 : -INFINITY};
  for (int m = 32; m >= QL; m >>= 1)
    for (int a = 0; a < 3; a++) {
      lo[a] = fminf(lo[a], __shfl_xor(lo[a], m, 64));
      hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], m, 64));
    }
  // place p = sub * E + e: distances in increasing order in the last K places
  // (the others hold -inf for good), and index * 16 + slot (index -1: never
  // filled); a lane past the end inserts nothing
  float md[E];
  int pay[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    const int j = sub * E + e - (12 - K);
    md[e] = j >= 0 && live ? 1e32f : -INFINITY;
    pay[e] = -16 + (j & 15);
  }
  float thr = live ? 1e32f : -INFINITY;  // the last place
  float second = K > 1 ? thr : -INFINITY;  // the place before
  int tail = dpp_last(pay[E - 1]);
  // cnt collected references at buf[base ..] through the scan
  auto process = [&](int base, int cnt) {
    unsigned cl = 0u, ch = 0u;
    const float t0 = thr;
#pragma unroll
    for (int v = 0; v < 64 / QL; v++) {
      const int u = v * QL + sub;
      const float d = svdist(q0, q1, q2, buf[base + u], s0, s1, s2);
      const unsigned bit = 1u << (u & 31);
      if (v * QL < 32)
        cl |= (d > t0) ? 0u : bit;
      else
        ch |= (d > t0) ? 0u : bit;
    }
    cl = dpp_or(cl);
    ch = dpp_or(ch);
    unsigned long long cand = ((unsigned long long)ch << 32) | cl;
    cand &= cnt < 64 ? (1ull << cnt) - 1ull : ~0ull;
    while (cand) {  // the same in the group's lanes
      const int u = __builtin_ctzll(cand);
      cand &= cand - 1ull;
      const float4 r = buf[base + u];
      const float d = svdist(q0, q1, q2, r, s0, s1, s2);
      if (d > thr) continue;
      if (second == thr) {  // the first slot among equal largest distances
        int best = 16;
#pragma unroll
        for (int e = 0; e < E; e++)
          best = md[e] == thr && (pay[e] & 15) < best ? pay[e] & 15 : best;
#pragma unroll
        for (int m = QL / 2; m >= 1; m >>= 1) best = min(best, __shfl_xor(best, m, QL));
        int p = INT_MIN;
#pragma unroll
        for (int e = 0; e < E; e++) {
          const bool at = md[e] == thr && (pay[e] & 15) == best;
          p = at ? pay[e] : p;
          pay[e] = at ? tail : pay[e];
        }
#pragma unroll
        for (int m = QL / 2; m >= 1; m >>= 1) p = max(p, __shfl_xor(p, m, QL));
        if (sub == QL - 1) pay[E - 1] = p;
        tail = p;
      }
      const int np = __float_as_int(r.w) * 16 + (tail & 15);
      const int pp = dpp_prev(pay[E - 1]);
      float pm = __int_as_float(dpp_prev(__float_as_int(md[E - 1])));
      pm = sub == 0 ? -INFINITY : pm;
      // c: the new entry goes at or before place e; the last place is evicted
      bool c = sub == QL - 1 || d < md[E - 1];
#pragma unroll
      for (int e = E - 1; e >= 0; e--) {
        const float left = e > 0 ? md[e - 1] : pm;
        const int lp = e > 0 ? pay[e - 1] : pp;
        const bool b = d < left;
        pay[e] = b ? lp : (c ? np : pay[e]);
        md[e] = __builtin_amdgcn_fmed3f(left, d, md[e]);
        c = b;
      }
      thr = dpp_last(md[E - 1]);
      second = dpp_last(md[E - 2]);
      tail = dpp_last(pay[E - 1]);
    }
  };
  float top = 1e32f;  // largest threshold of the wave's queries
  int nbuf = 0;
  for (int b0 = 0; b0 < nblk; b0 += 64) {
    const int bl = b0 + lane;
    bool keep = bl < nblk;
    if (keep) {
      const float lb =
          gap_bound(fmaxf(box[bl] - hi[0], lo[0] - box[3 * nblk + bl]),
                    fmaxf(box[nblk + bl] - hi[1], lo[1] - box[4 * nblk + bl]),
                    fmaxf(box[2 * nblk + bl] - hi[2], lo[2] - box[5 * nblk + bl]), s0, s1, s2);
      keep = !(lb > top);
    }
    unsigned long long blocks = __ballot(keep);
    while (blocks) {
      int r[kKU];
      float x[kKU], y[kKU], z[kKU];
#pragma unroll
      for (int t = 0; t < kKU; t++) {
        r[t] = R;
        if (blocks) {
          r[t] = (b0 + __builtin_ctzll(blocks)) * kKB + lane;
          blocks &= blocks - 1ull;
        }
        const int p = r[t] < R ? r[t] : 0;
        x[t] = ref[p];
        y[t] = ref[p + Rp];
        z[t] = ref[p + 2 * Rp];
      }
#pragma unroll
      for (int t = 0; t < kKU; t++) {
        const bool in = r[t] < R && !(box_bound(x[t], y[t], z[t], lo, hi, s0, s1, s2) > top);
        const unsigned long long m = __ballot(in);
        if (in)
          buf[nbuf + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
              make_float4(x[t], y[t], z[t], __int_as_float(r[t]));
        nbuf += __popcll(m);
      }
      if (nbuf < 64) continue;
      lds_sync();
      int base = 0;
      for (; base + 64 <= nbuf; base += 64) process(base, 64);
      top = thr;
#pragma unroll
      for (int m = 32; m >= QL; m >>= 1) top = fmaxf(top, __shfl_xor(top, m, 64));
      nbuf -= base;
      const float4 rest = buf[base + (lane < nbuf ? lane : 0)];
      lds_sync();  // the references left move to the front
      if (lane < nbuf) buf[lane] = rest;
    }
  }
  lds_sync();
  if (nbuf > 0) process(0, nbuf);
  if (!live) return;
#pragma unroll
  for (int e = 0; e < E; e++)
    if (sub * E + e >= 12 - K) {
      const long long o = q + (pay[e] & 15) * Q;
      ind[o] = pay[e] >> 4;
      if (dist) dist[o] = md[e];
    }
}

// Queries sorted and searched for together: four lanes each and a 32-bit index
// within the piece, for any number of queries (2^30 at once would be a grid of
// 2^32 threads, which no launch takes), and 20 bytes of scratch for no more
// than a piece of them.
constexpr long long kPiece = 1LL << 22;

inline size_t up256(size_t n) { return (n + 255) & ~size_t(255); }

struct KnnWs {
  void* dev = nullptr;
  size_t cap = 0;
};
std::mutex g_mu;
std::vector<KnnWs> g_ws;

int hip_fail(hipError_t e, const char* what) {
  tgmm_set_error("knnCUDA_: %s failed: %s", what, hipGetErrorString(e));
  return e == hipErrorOutOfMemory ? TGMM_ERR_OOM : TGMM_ERR_DEVICE;
}

}  // namespace

extern "C" int tgmm_knnCUDA_(int* ind, float* dist, const float* query, const float* ref,
                             long long query_nb, int ref_nb, int KNN, const float* scale,
                             int devCUDA) {
  if (KNN < 1 || KNN > kKM) {
    tgmm_set_error("knnCUDA_: KNN = %d outside 1..%d (maxKNN)", KNN, kKM);
    return TGMM_ERR_LIMIT;
  }
  if (query_nb < 0 || !scale) {
    tgmm_set_error("knnCUDA_: negative query_nb or NULL scale");
    return TGMM_ERR_ARG;
  }
  if (ref_nb <= 0) {  // no possible assignments (knnCuda.cu:165-171)
    if (dist)
      for (long long i = 0; i < query_nb * KNN; i++) dist[i] = 1e32f;
    return TGMM_OK;
  }
  if (query_nb == 0) return TGMM_OK;
  if (!ind || !query || !ref) {
    tgmm_set_error("knnCUDA_: NULL argument");
    return TGMM_ERR_ARG;
  }
  hipError_t e = hipSetDevice(devCUDA);
  if (e != hipSuccess) return hip_fail(e, "hipSetDevice");
  const long long Q = query_nb, R = ref_nb;
  const int nblk = (int)((R + kKB - 1) / kKB);
  const long long Rp = (long long)nblk * kKB;
  const long long piece = std::min(Q, kPiece);
  const size_t o_q = 0;
  const size_t o_r = o_q + up256((size_t)Q * 12);
  const size_t o_box = o_r + up256((size_t)Rp * 12);
  const size_t o_prep = o_box + up256((size_t)nblk * 24);
  const size_t o_cnt = o_prep + 256;
  const size_t o_cell = o_cnt + up256((size_t)kCells * 4);
  const size_t o_q4 = o_cell + up256((size_t)piece * 4);
  const size_t o_ind = o_q4 + up256((size_t)piece * 16);
  const size_t o_dist = o_ind + up256((size_t)Q * KNN * 4);
  const size_t total = o_dist + up256((size_t)Q * KNN * 4);
  std::lock_guard<std::mutex> lk(g_mu);
  if ((int)g_ws.size() <= devCUDA) g_ws.resize(devCUDA + 1);
  KnnWs& ws = g_ws[devCUDA];
  if (total > ws.cap) {
    if (ws.dev) (void)hipFree(ws.dev);
    ws.dev = nullptr;
    ws.cap = 0;
    if ((e = hipMalloc(&ws.dev, total)) != hipSuccess) return hip_fail(e, "hipMalloc");
    ws.cap = total;
  }
  char* base = (char*)ws.dev;
  auto* dq = (float*)(base + o_q);
  auto* dr = (float*)(base + o_r);
  auto* dbox = (float*)(base + o_box);
  auto* dprep = (KnnPrep*)(base + o_prep);
  auto* dcnt = (int*)(base + o_cnt);
  auto* dcell = (int*)(base + o_cell);
  auto* dq4 = (float4*)(base + o_q4);
  auto* dind = (int*)(base + o_ind);
  auto* ddist = (float*)(base + o_dist);
  if ((e = hipMemcpyAsync(dq, query, (size_t)Q * 12, hipMemcpyHostToDevice, 0)) != hipSuccess)
    return hip_fail(e, "upload of the queries");
  for (int a = 0; a < 3; a++)
    if ((e = hipMemcpyAsync(dr + a * Rp, ref + a * R, (size_t)R * 4, hipMemcpyHostToDevice, 0)) !=
            hipSuccess ||
        (Rp > R && (e = hipMemsetAsync(dr + a * Rp + R, 0, (size_t)(Rp - R) * 4, 0)) !=
                       hipSuccess))
      return hip_fail(e, "upload of the references");
  // bounds, flag and counts start from zero
  if ((e = hipMemsetAsync(dprep, 0, o_cell - o_prep, 0)) != hipSuccess)
    return hip_fail(e, "clearing the counts");
  const float s0 = scale[0], s1 = scale[1], s2 = scale[2];
  k_svknn_boxes<<<nblk + (unsigned)std::min<long long>(256, (Q + kKB - 1) / kKB), kKB, 0, 0>>>(
      dr, (int)R, (int)Rp, nblk, dbox, dq, Q, dprep);
  for (long long p = 0; p < Q; p += piece) {
    const long long n = std::min(piece, Q - p);
    const unsigned qb = (unsigned)((n + 255) / 256);
    int* pind = dind + p;
    float* pdist = dist ? ddist + p : nullptr;
    if (p > 0 && (e = hipMemsetAsync(dcnt, 0, (size_t)kCells * 4, 0)) != hipSuccess)
      return hip_fail(e, "clearing the counts");
    k_svknn_count<<<qb, 256, 0, 0>>>(dq + p, n, Q, s0, s1, s2, dprep, dcell, dcnt);
    k_svknn_scan<<<1, 1024, 0, 0>>>(dcnt);
    k_svknn_scatter<<<qb, 256, 0, 0>>>(dq + p, n, Q, dcell, dcnt, dq4);
    k_svknn<<<(unsigned)((n * QL + 63) / 64), 64, 0, 0>>>(dq4, n, Q, dr, (int)R, (int)Rp, KNN, s0,
                                                          s1, s2, dbox, nblk, dprep, pind, pdist);
    if (n >= kScanAlone)  // returns at once unless it has to
      k_svknn_all<<<(unsigned)((n + 63) / 64), 64, 0, 0>>>(dq4, n, Q, dr, (int)R, (int)Rp, KNN, s0,
                                                           s1, s2, dbox, nblk, dprep, pind, pdist);
  }
  if ((e = hipGetLastError()) != hipSuccess) return hip_fail(e, "kernel launch");
  if ((e = hipMemcpy(ind, dind, (size_t)Q * KNN * 4, hipMemcpyDeviceToHost)) != hipSuccess ||
      (dist && (e = hipMemcpy(dist, ddist, (size_t)Q * KNN * 4, hipMemcpyDeviceToHost)) !=
                   hipSuccess))
    return hip_fail(e, "download of the neighbours");
  return TGMM_OK;
}
