// Two-tree Barnes–Hut on the device (gfx950).
//
// Reference: src/compute_link.cpp:294-934 (trees, moments, far field, node-pair
// traversal) and src/linking_number_certificate.cpp:102-229 (adaptive beta).
//
// Trees.  Each curve's segments are sorted by the 30-bit Morton code of their
// midpoint in the curve's box: short curves by a block each, the others by one
// segmented radix sort.  A curve's tree is the balanced median split of its
// Morton-ordered segments (left half floor(n/2)), down to leaf buckets of at
// most leaf_size segments; a subtree is a contiguous range of the sorted order
// (the reference's ModifiedKdBVH.h:128-131 property).  Every node's range and
// children follow from the segment counts alone and come from one launch.
//
// Moments (reference compute_link.cpp:333-389) are built bottom-up in FP64
// about each node's box centre: nodes of at most 8 segments sum their
// segments' closed forms (FP32 terms, FP64 centring), larger nodes shift their
// children's moments in FP64 (Eqs. 21-23), and the records are stored in FP32.  The centre keeps an FP32 hi/lo split so node
// separations are exact to FP32 precision of the separation itself.
//
// Traversal.  Work items are (pair, node1, node2).  A pass goes level by level, one
// kernel a level, or, with few segments a pair, depth first in a few rounds of
// bh_walk; either classifies every item: leaf-bucket pairs go to a leaf list
// evaluated exactly by a second kernel, pairs with |r|^2 > beta^2 (r1+r2)^2
// are evaluated with the second-order far field (reference
// compute_link.cpp:410-524, Supplemental Eqs. 29-30) and the Eq. 14 error
// estimate, the rest split the larger node (a leaf is never split).  A pass whose
// buffers overflow is run again from the host, in chunks of a level with a LIFO
// stack, so memory is bounded by depth x chunk whatever the frontier width.  Per-pair sums and
// error estimates are FP64; a block of 1024 items reduces its sums and queue
// slots in LDS before one global atomic each.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "bh_types.h"
#include "mlp_infer.h"
#include "flk_internal.h"

namespace flk {

// ---------------------------------------------------------------- records
struct BhRange {    // node range during construction
  int32_t lo, hi;
};
// Nodes of at most this many segments take their moments from their segments
// (no FP64 record round trip; a node reads at most 2 x 8 segments).
constexpr int32_t kDirectSegments = 8;

struct Mom64 {      // FP64 moments during construction
  double box[6];
  double c[3];
  double D[9];
  double Q[18];
};


namespace {

constexpr float kInv2PiF = 0.15915494309189533577f;
constexpr float kInv4PiF = 0.07957747154594766788f;

__device__ __forceinline__ uint32_t spread10(uint32_t v) {  // bits of v to every third place
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  return (v | (v << 2)) & 0x09249249u;
}

// Sort keys of the Barnes–Hut segments, one block per tile of the segmented
// sort (a tile lies within one curve, tcurve[b]): the Morton code of the
// segment midpoint in the curve's box, 10 bits per axis; the value is the
// segment's first vertex.  cbox holds per curve the box corner (3 doubles)
// and 1024 / extent per axis (0 for a flat axis).  The segmented sort keeps
// every curve's segments in its own range, and segments sharing a cell keep
// their order along the curve (the sort is stable).  The vertices are read as
// VP: the FP64 coordinates (double4), or, when every stored coordinate is
// exact in FP32, their FP32 copies (float4, half the bytes, the same values).
template <typename VP>
__device__ __forceinline__ uint32_t segment_key(const VP &p, const VP &q, const double *__restrict__ cb) {
  const double m[3] = {0.5 * ((double)p.x + (double)q.x), 0.5 * ((double)p.y + (double)q.y),
                       0.5 * ((double)p.z + (double)q.z)};
  uint32_t code = 0;
  for (int d = 0; d < 3; ++d) {
    const double u = (m[d] - cb[d]) * cb[3 + d];
    code |= spread10((uint32_t)fmin(fmax(u, 0.0), 1023.0)) << (2 - d);
  }
  return code;
}

template <typename VP>
__global__ __launch_bounds__(256) void bh_keys(const VP *__restrict__ pts, const int64_t *__restrict__ seg_off,
                                               const int64_t *__restrict__ vtx_off, const double *__restrict__ cbox,
                                               const RadixTile *__restrict__ tiles,
                                               const int32_t *__restrict__ tcurve, uint32_t *__restrict__ keys,
                                               uint32_t *__restrict__ vals) {
  const RadixTile tl = tiles[blockIdx.x];
  const int c = tcurve[blockIdx.x];
  const int64_t v0 = vtx_off[c] - seg_off[c];
  for (int o = threadIdx.x; o < tl.count; o += 256) {
    const int64_t g = (int64_t)tl.start + o;
    const int64_t v = v0 + g;
    keys[g] = segment_key(pts[v], pts[v + 1], cbox + 6 * c);
    vals[g] = (uint32_t)v;
  }
}

// Exclusive scan of one value per thread over a block of WAVES waves; *total
// receives the sum.  sw: WAVES ints of LDS.  Contains block barriers.
template <int WAVES> __device__ __forceinline__ int block_scan(int v, int *total, int *sw) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(inc, d, 64);
    if (lane >= d) inc += u;
  }
  if (lane == 63) sw[w] = inc;
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) {
    off += k < w ? sw[k] : 0;
    tot += sw[k];
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

// The trees' shape follows from the segment counts alone.  A node of s segments
// splits into floor(s / 2) and the rest while s > leaf, so a curve of n segments
// has 2^l nodes on every level l up to its first that does not split whole,
// l = full, with m or m + 1 segments each, m = n >> full <= leaf.  Below that, if
// m == leaf, the big nodes alone have children.  The nodes of a level lie in the
// order of curves and then of segments, as a level-by-level construction numbers
// them, and a node's segments are those of the bits of its place (with j nodes
// of the level before it, j m segments and one for every big node of them, so
// the split nodes' ranks need no scan).
struct BhShape {
  int32_t n, full, m;
  __device__ __forceinline__ BhShape(int32_t n_, int32_t leaf) : n(n_), full(max(0, __clz(leaf) - __clz(n_))) {
    full += (n >> full) > leaf;  // as many bits as leaf, so at most one level more
    m = n >> full;
  }
  __device__ __forceinline__ int32_t big() const { return n - (m << full); }
  __device__ __forceinline__ int32_t nodes(int32_t lev, int32_t leaf) const {
    return lev <= full ? 1 << lev : lev == full + 1 && m == leaf ? 2 * big() : 0;
  }
};

// Each curve's first node on each level, counted from the level's: block l scans
// the curves' nodes of level l.
__global__ __launch_bounds__(256) void bh_level_offsets(const int64_t *__restrict__ seg_off, int32_t nc, int32_t leaf,
                                                        int32_t *__restrict__ loff) {
  __shared__ int sw[4];
  const int lev = blockIdx.x;
  int carry = 0;
  for (int32_t c0 = 0; c0 < nc; c0 += 256) {
    const int32_t k = c0 + threadIdx.x;
    const int v = k < nc ? BhShape((int32_t)(seg_off[k + 1] - seg_off[k]), leaf).nodes(lev, leaf) : 0;
    int tot;
    const int pos = carry + block_scan<4>(v, &tot, sw);
    if (k < nc) loff[(int64_t)lev * nc + k] = pos;
    carry += tot;
  }
}

struct BhLevels {
  int32_t depth, base[33];  // levels, each one's first node, and the nodes' number
};

// Segment range and children of every node, a thread for each two siblings (or
// root).  Bound by the 16 bytes a node it writes and by latency.  Level by level
// (a launch each, and three more for a scan of the split flags where not all
// nodes split) these took, as launches: 2 x 8M segments 326 us, 1,000 curves of
// 31M 1,010, 400 of 4e5 195, ten of 24,000 150, of which the launches' own time
// is 5-7 us each.
__global__ __launch_bounds__(256) void bh_topology(const int64_t *__restrict__ seg_off, int32_t nc, int32_t leaf,
                                                   BhLevels L, const int32_t *__restrict__ loff,
                                                   BhRange *__restrict__ range, int2 *__restrict__ child) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  // unit -> level and place: a root, or the pair of siblings at 2 i of its level
  int lev = 0;
  int64_t first = 0, count = nc;
  while (u >= first + count) {
    first += count;
    if (++lev >= L.depth) return;
    count = (L.base[lev + 1] - L.base[lev]) / 2;
  }
  const int32_t at = (int32_t)(u - first) * (lev ? 2 : 1);
  const int32_t *row = loff + (int64_t)lev * nc;
  int32_t k = 0, hi = nc;  // the last curve whose nodes start at or before `at`
  while (hi - k > 1) {
    const int32_t mid = k + (hi - k) / 2;
    if (row[mid] <= at) k = mid;
    else hi = mid;
  }
  const int32_t seg0 = (int32_t)seg_off[k];
  const BhShape C((int32_t)seg_off[k + 1] - seg0, leaf);
  // the parent's segments (a root's own): down the bits of its place, or, below
  // the last whole level, to the r-th big node
  int32_t lo = 0, size = C.n, j = at - row[k];
  if (lev <= C.full) {
    for (int b = lev - 2; b >= 0; --b) {
      const int32_t half = size / 2;
      const bool right = (j >> (b + 1)) & 1;
      lo += right ? half : 0;
      size = right ? size - half : half;
    }
  } else {
    int32_t r = j / 2;
    for (int b = C.full - 1; b >= 0; --b) {
      const int32_t half = size / 2, left = half - (C.m << b);
      const bool right = r >= left;
      r -= right ? left : 0;
      lo += right ? half : 0;
      size = right ? size - half : half;
    }
  }
  const int32_t mid = size / 2;
  const int32_t below = lev < C.full + 1 && lev + 1 < L.depth ? L.base[lev + 1] + row[nc + k] : 0;
  for (int c = 0; c < (lev ? 2 : 1); ++c, ++j) {
    const int32_t l = lev && c ? lo + mid : lo, s = !lev ? size : c ? size - mid : mid;
    const int64_t id = (int64_t)L.base[lev] + at + c;
    range[id] = BhRange{seg0 + l, seg0 + l + s};
    const int32_t to = below + 2 * (lev < C.full ? j : l - j * C.m);
    child[id] = s > leaf ? make_int2(to, to + 1) : make_int2(-1, -1);
  }
}

__host__ __device__ __forceinline__ int qidx(int i, int j) { return sym_idx(i, j); }

// Endpoints of every segment in sorted order, gathered once after the sort
// (six values per segment, copied unchanged from the vertex array), so the
// moment kernels read each node's segments as one contiguous run.  SP is
// double2 (48 bytes per segment), or float2 (24 bytes) when every stored
// coordinate is exact in FP32 (the curve set has no FP32 lo parts): the FP64
// values read back are then the same bits, at half the traffic, and they are
// gathered from the FP32 copies of the vertices (VP float4, 16 bytes a
// vertex instead of 32).
__device__ __forceinline__ double2 mk2(double2, double x, double y) { return make_double2(x, y); }
__device__ __forceinline__ float2 mk2(float2, double x, double y) { return make_float2((float)x, (float)y); }

template <typename SP, typename VP>
__device__ __forceinline__ void stage_segment(const VP &a, const VP &b, SP *__restrict__ sp) {
  sp[0] = mk2(SP{}, a.x, a.y);
  sp[1] = mk2(SP{}, a.z, b.x);
  sp[2] = mk2(SP{}, b.y, b.z);
}

template <typename SP, typename VP>
__global__ __launch_bounds__(256) void bh_stage_segments(const uint32_t *__restrict__ order,
                                                         const VP *__restrict__ pts, int64_t nseg,
                                                         SP *__restrict__ sp) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseg) return;
  const uint32_t v = order[s];
  stage_segment(pts[v], pts[v + 1], sp + 3 * s);
}

// Keys, sort and (sp not null) staged end points of a curve of at most CAP
// segments in one block, list[b] its rank: the same order as the segmented
// sort's.  Each wave sorts runs of 64 across its lanes, key and place as one
// number, and runs are merged by each element finding its place in the other run
// by its key alone (a left run's places are all below the right one's: an element
// of the right follows the left's equal keys), a thread's E elements side by side
// in 6 bytes of LDS each.  Bound by latency,
// as the segmented sort's 14-18 launches are, which took 110 us for ten curves of
// 24,000 segments and 165 for 400 of 4e5: 37 and 36 here (43 and 42 with a branch
// for each of a thread's elements).  8,192 takes 48 KB, two blocks a CU.
constexpr int kSmallSorts = 3;
constexpr int kSmallSort[kSmallSorts] = {1024, 4096, 8192}, kSmallThreads[kSmallSorts] = {256, 1024, 1024};
template <typename SP, typename VP, int THREADS, int CAP>
__global__ __launch_bounds__(THREADS) void bh_sort_small(const VP *__restrict__ pts,
                                                         const int64_t *__restrict__ seg_off,
                                                         const int64_t *__restrict__ vtx_off,
                                                         const double *__restrict__ cbox,
                                                         const int32_t *__restrict__ list,
                                                         uint32_t *__restrict__ order, SP *__restrict__ sp) {
  constexpr int E = CAP / THREADS;
  constexpr int kPlaceBits = 13;
  static_assert(CAP <= 1 << kPlaceBits && THREADS % 64 == 0, "places fit, whole waves");
  __shared__ uint32_t keys[CAP];
  __shared__ uint16_t places[CAP];
  const int c = list[blockIdx.x], lane = threadIdx.x & 63;
  const int64_t g0 = seg_off[c], v0 = vtx_off[c];
  const int n = (int)(seg_off[c + 1] - g0), padded = (n + 63) / 64 * 64;
  // sets of 64 segments, this wave's
  const int sets = __builtin_amdgcn_readfirstlane(max(0, (n - ((int)threadIdx.x - lane) + THREADS - 1) / THREADS));
  // a wave with one set takes the code for one, any other that for E: without a
  // branch for each set the sets' exchanges and searches overlap
  auto sort_runs = [&](auto count) {
    constexpr int N = decltype(count)::value;
    uint64_t x[N];
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const int i = e * THREADS + (int)threadIdx.x;
      x[e] = 1ull << (30 + kPlaceBits) | (uint64_t)i;  // behind every segment
      if (i < n) x[e] = (uint64_t)segment_key(pts[v0 + i], pts[v0 + i + 1], cbox + 6 * c) << kPlaceBits | (uint64_t)i;
    }
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1)
#pragma unroll
      for (int d = k / 2; d > 0; d >>= 1) {
        const bool low = ((lane & d) == 0) == ((lane & k) == 0);  // keeps the smaller
        uint64_t y[N];
#pragma unroll
        for (int e = 0; e < N; ++e) y[e] = __shfl_xor(x[e], d, 64);
#pragma unroll
        for (int e = 0; e < N; ++e) x[e] = (x[e] < y[e]) == low ? x[e] : y[e];
      }
#pragma unroll
    for (int e = 0; e < N; ++e)
      if (e < sets) {
        keys[e * THREADS + (int)threadIdx.x] = (uint32_t)(x[e] >> kPlaceBits);
        places[e * THREADS + (int)threadIdx.x] = (uint16_t)(x[e] & ((1u << kPlaceBits) - 1));
      }
  };
  uint32_t key[E];
  uint16_t place[E];
  int to[E];  // the element's place in the merged run
  auto find = [&](auto count, int run) {
    constexpr int N = decltype(count)::value;
    int start[N], len[N], before[N];  // the other run, and how many of it go before
    uint32_t below[N];
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const int i = min(e * THREADS + (int)threadIdx.x, padded - 1);
      start[e] = min((i & ~(run - 1)) ^ run, padded);
      len[e] = min(padded - start[e], run);
      before[e] = 0;
      key[e] = keys[i];
      place[e] = places[i];
      below[e] = key[e] + ((i & run) ? 1u : 0u);
      to[e] = (i & ~(2 * run - 1)) + (i & (run - 1));
    }
    for (int h = run; h > 0; h >>= 1) {
      uint32_t k[N];
#pragma unroll
      for (int e = 0; e < N; ++e) k[e] = keys[min(start[e] + before[e] + h, padded) - 1];
#pragma unroll
      for (int e = 0; e < N; ++e) before[e] += before[e] + h <= len[e] && k[e] < below[e] ? h : 0;
    }
#pragma unroll
    for (int e = 0; e < N; ++e) to[e] += before[e];
  };
  using One = std::integral_constant<int, 1>;
  using All = std::integral_constant<int, E>;
  if (sets == 1) sort_runs(One{});
  else if (sets) sort_runs(All{});
  for (int run = 64; run < n; run *= 2) {
    __syncthreads();
    if (sets == 1) find(One{}, run);
    else if (sets) find(All{}, run);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (e < sets) {
        keys[to[e]] = key[e];
        places[to[e]] = place[e];
      }
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = e * THREADS + (int)threadIdx.x;
    if (i >= n) continue;
    const int64_t v = v0 + places[i];
    order[g0 + i] = (uint32_t)v;
    if (sp) stage_segment(pts[v], pts[v + 1], sp + 3 * (g0 + i));
  }
}

template <typename SP>
__device__ __forceinline__ void seg_ends(const SP *__restrict__ sp, int s, double (&pa)[3], double (&pb)[3]) {
  const SP u = sp[3 * (int64_t)s], v = sp[3 * (int64_t)s + 1], w = sp[3 * (int64_t)s + 2];
  pa[0] = u.x; pa[1] = u.y; pa[2] = v.x;
  pb[0] = v.y; pb[1] = w.x; pb[2] = w.y;
}

// f(pa, pb) for the segments [lo, lo + cnt) in order, their end points read
// kSegChunk segments at a time with every load of a chunk issued before the
// first is used (one round trip per chunk, not per segment).
constexpr int kSegChunk = 4;
template <typename SP, class F>
__device__ __forceinline__ void each_seg(const SP *__restrict__ sp, int lo, int cnt, F &&f) {
  for (int q0 = 0; q0 < cnt; q0 += kSegChunk) {
    const SP *p = sp + 3 * ((int64_t)lo + q0);
    SP v[3 * kSegChunk];
#pragma unroll
    for (int q = 0; q < kSegChunk; ++q)
      if (q0 + q < cnt) {
        v[3 * q] = p[3 * q];
        v[3 * q + 1] = p[3 * q + 1];
        v[3 * q + 2] = p[3 * q + 2];
      }
#pragma unroll
    for (int q = 0; q < kSegChunk; ++q)
      if (q0 + q < cnt) {
        double pa[3] = {(double)v[3 * q].x, (double)v[3 * q].y, (double)v[3 * q + 1].x};
        double pb[3] = {(double)v[3 * q + 1].y, (double)v[3 * q + 2].x, (double)v[3 * q + 2].y};
        f(pa, pb);
      }
  }
}

// Bounding box of the segments [r.lo, r.hi) of a small node.
template <typename SP>
__device__ void leaf_box(BhRange r, const SP *__restrict__ sp, double (&box)[6]) {
  for (int t = 0; t < 3; ++t) {
    box[t] = DBL_MAX;
    box[3 + t] = -DBL_MAX;
  }
  each_seg(sp, r.lo, r.hi - r.lo, [&](const double (&pa)[3], const double (&pb)[3]) {
    for (int d = 0; d < 3; ++d) {
      box[d] = fmin(box[d], fmin(pa[d], pb[d]));
      box[3 + d] = fmax(box[3 + d], fmax(pa[d], pb[d]));
    }
  });
}

// FP64 moments -> FP32 node records (centre hi/lo, radius, children, segment
// range, moment norms for the error estimate; c, D, Q).
__device__ __forceinline__ void node_records(const Mom64 &M, int2 ch, BhRange r, BhGeo &g, BhMom &m) {
  double ctr[3], dsq = 0;
  for (int d = 0; d < 3; ++d) {
    ctr[d] = 0.5 * (M.box[3 + d] + M.box[d]);
    const double e = M.box[3 + d] - M.box[d];
    dsq += e * e;
  }
  const float hx = (float)ctr[0], hy = (float)ctr[1], hz = (float)ctr[2];
  g.cx = hx; g.cy = hy; g.cz = hz;
  g.lx = (float)(ctr[0] - hx); g.ly = (float)(ctr[1] - hy); g.lz = (float)(ctr[2] - hz);
  g.rsq = (float)(0.25 * dsq);
  g.radius = (float)sqrt(0.25 * dsq);
  g.c0 = ch.x;
  g.c1 = ch.y;
  g.seg0 = r.lo;
  g.nseg = r.hi - r.lo;
  double dn = 0, qn = 0;
  for (int t = 0; t < 9; ++t) dn += M.D[t] * M.D[t];
  for (int kk = 0; kk < 3; ++kk)
    for (int t = 0; t < 6; ++t) {
      const double v = M.Q[6 * kk + t];
      qn += ((t == 1 || t == 2 || t == 4) ? 2.0 : 1.0) * v * v;
    }
  g.cn = (float)sqrt(M.c[0] * M.c[0] + M.c[1] * M.c[1] + M.c[2] * M.c[2]);
  g.dn = (float)(sqrt(dn) * 0.57735026918962576451);
  g.qn = (float)((1.0 / 3.0) * sqrt(qn));
  g.pad = 0.f;
  for (int t = 0; t < 3; ++t) m.c[t] = (float)M.c[t];
  for (int t = 0; t < 9; ++t) m.D[t] = (float)M.D[t];
  for (int t = 0; t < 18; ++t) m.Q[t] = (float)M.Q[t];
  m.pad[0] = m.pad[1] = 0.f;
}

// Moments and records of a node of at most `direct` segments, from its
// segments: the box and centre in FP64, each segment's tangent and centred
// midpoint rounded to FP32 from FP64, and the closed forms (reference
// compute_link.cpp:333-356: c += t, D += t (m - ctr)^T,
// Q_k += t_k (t t^T / 12 + (m - ctr)(m - ctr)^T)) accumulated in FP32
// (at most `direct` terms, the precision of the FP32 records they end in).
// Both moment kernels use it, so a node's records depend only on its own
// segments, never on which launch computed them.
template <typename SP>
__device__ __forceinline__ void direct_records(BhRange rr, int2 ch, const SP *__restrict__ sp, BhGeo &gr,
                                               BhMom &m) {
  double box[6];
  leaf_box(rr, sp, box);
  double ctr[3], dsq = 0;
  for (int d = 0; d < 3; ++d) {
    ctr[d] = 0.5 * (box[3 + d] + box[d]);
    const double e = box[3 + d] - box[d];
    dsq += e * e;
  }
  for (int t = 0; t < 3; ++t) m.c[t] = 0.f;
  for (int t = 0; t < 9; ++t) m.D[t] = 0.f;
  for (int t = 0; t < 18; ++t) m.Q[t] = 0.f;
  each_seg(sp, rr.lo, rr.hi - rr.lo, [&](const double (&pa)[3], const double (&pb)[3]) {
    float t[3], w[3];
    for (int d = 0; d < 3; ++d) {
      t[d] = (float)(pb[d] - pa[d]);
      w[d] = (float)(0.5 * (pa[d] + pb[d]) - ctr[d]);
    }
    for (int i = 0; i < 3; ++i) {
      m.c[i] += t[i];
      for (int j = 0; j < 3; ++j) m.D[3 * i + j] = fmaf(t[i], w[j], m.D[3 * i + j]);
    }
    for (int kk = 0; kk < 3; ++kk)
      for (int i = 0; i < 3; ++i)
        for (int j = i; j < 3; ++j)
          m.Q[6 * kk + qidx(i, j)] =
              fmaf(t[kk], fmaf((1.0f / 12.0f) * t[i], t[j], w[i] * w[j]), m.Q[6 * kk + qidx(i, j)]);
  });
  m.pad[0] = m.pad[1] = 0.f;
  const float hx = (float)ctr[0], hy = (float)ctr[1], hz = (float)ctr[2];
  gr.cx = hx; gr.cy = hy; gr.cz = hz;
  gr.lx = (float)(ctr[0] - hx); gr.ly = (float)(ctr[1] - hy); gr.lz = (float)(ctr[2] - hz);
  gr.rsq = (float)(0.25 * dsq);
  gr.radius = sqrtf(gr.rsq);
  gr.c0 = ch.x;
  gr.c1 = ch.y;
  gr.seg0 = rr.lo;
  gr.nseg = rr.hi - rr.lo;
  float dn = 0.f, qn = 0.f;
  for (int t = 0; t < 9; ++t) dn = fmaf(m.D[t], m.D[t], dn);
  for (int kk = 0; kk < 3; ++kk)
    for (int t = 0; t < 6; ++t) {
      const float v = m.Q[6 * kk + t];
      qn = fmaf((t == 1 || t == 2 || t == 4) ? 2.f * v : v, v, qn);
    }
  gr.cn = sqrtf(fmaf(m.c[0], m.c[0], fmaf(m.c[1], m.c[1], m.c[2] * m.c[2])));
  gr.dn = sqrtf(dn) * 0.57735026918962576451f;
  gr.qn = (1.0f / 3.0f) * sqrtf(qn);
  gr.pad = 0.f;
  if (gr.nseg == 1) {  // a one-segment leaf: its tangent instead of a BhMom record
    gr.c0 = kLeafSegment;
    gr.c1 = __builtin_bit_cast(int32_t, m.c[0]);
    gr.pad = m.c[1];
    gr.dn = m.c[2];
  }
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// Stores the FP32 records of a wave's nw consecutive nodes (lane l holds
// node l's; geo and mom point at the wave's first node) through the wave's
// LDS buffer sw (at least 256 float4), so each store instruction writes 1 KB
// of contiguous memory.  One-segment leaves write no BhMom record.
__device__ __forceinline__ void wave_store_records(const BhGeo &gr, const BhMom &m, BhGeo *__restrict__ geo,
                                                   BhMom *__restrict__ mom, int nw, float4 *sw) {
  const int lane = threadIdx.x & 63;
  const float4 *g4 = reinterpret_cast<const float4 *>(&gr);
#pragma unroll
  for (int i = 0; i < 4; ++i) sw[4 * lane + i] = g4[i];
  wave_lds_sync();
  float4 *gdst = reinterpret_cast<float4 *>(geo);
  for (int c = lane; c < 4 * nw; c += 64) gdst[c] = sw[c];
  wave_lds_sync();
  const unsigned long long keep = __ballot(lane < nw && !is_leaf_segment(gr));
  const float4 *m4 = reinterpret_cast<const float4 *>(&m);
  float4 *mdst = reinterpret_cast<float4 *>(mom);
#pragma unroll
  for (int h = 0; h < 2; ++h) {  // records of lanes 32h .. 32h + 31
    if (((keep >> (32 * h)) & 0xffffffffull) == 0) continue;  // wave-uniform
    if ((lane >> 5) == h)
#pragma unroll
      for (int i = 0; i < 8; ++i) sw[8 * (lane & 31) + i] = m4[i];
    wave_lds_sync();
    const int lim = 8 * min(32, nw - 32 * h);
    for (int c = lane; c < lim; c += 64)
      if ((keep >> (32 * h + c / 8)) & 1ull) mdst[256 * h + c] = sw[c];
    wave_lds_sync();
  }
}

// The same for FP64 records, kept only by the lanes in `has` (others skip
// theirs): 16 lanes' records (288 float4) per pass through sw.
__device__ __forceinline__ void wave_store_m64(const Mom64 &M, unsigned long long has, Mom64 *__restrict__ dst,
                                               int nw, float4 *sw) {
  constexpr int kChunks = (int)(sizeof(Mom64) / 16);  // 18
  static_assert(sizeof(Mom64) % 16 == 0, "whole 16-byte chunks");
  const int lane = threadIdx.x & 63;
  const float4 *src = reinterpret_cast<const float4 *>(&M);
  float4 *d = reinterpret_cast<float4 *>(dst);
#pragma unroll
  for (int h = 0; h < 4; ++h) {  // lanes 16h .. 16h + 15
    if ((has >> (16 * h)) & 0xffffull) {
      if ((lane >> 4) == h && ((has >> lane) & 1ull))
#pragma unroll
        for (int i = 0; i < kChunks; ++i) sw[kChunks * (lane & 15) + i] = src[i];
      wave_lds_sync();
      for (int c = lane; c < kChunks * 16; c += 64) {
        const int owner = 16 * h + c / kChunks;
        if (owner < nw && ((has >> owner) & 1ull)) d[kChunks * 16 * h + c] = sw[c];
      }
      wave_lds_sync();
    }
  }
}

// The bottom levels, where every node has at most `direct` segments, in one
// launch over all of them; registers stay low enough for full occupancy.
// A wave's 64 consecutive records leave through a 4 KB LDS buffer, so every
// store instruction writes 1 KB of contiguous memory instead of one 16-byte
// piece of each lane's own record.
template <typename SP>
__global__ __launch_bounds__(256) void bh_moments_direct(const BhRange *__restrict__ range, int32_t base,
                                                         int32_t n, const int2 *__restrict__ child,
                                                         const SP *__restrict__ sp, BhGeo *__restrict__ geo,
                                                         BhMom *__restrict__ mom) {
  __shared__ float4 stage[4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int k0 = blockIdx.x * blockDim.x + w * 64;  // this wave's first node past base
  if (k0 >= n) return;                                // whole wave: no LDS exchange to join
  const int k = k0 + lane, nw = min(64, n - k0);
  BhGeo gr;
  BhMom m;
  if (k < n) direct_records(range[base + k], child[base + k], sp, gr, m);
  wave_store_records(gr, m, geo + base + k0, mom + base + k0, nw, stage[w]);
}

// FP64 moments of a node above `direct` segments from its two children.
template <typename SP>
__device__ void node_moments(BhRange rr, int2 ch, int32_t direct, const BhRange *__restrict__ range,
                             const SP *__restrict__ sp, const Mom64 *m64, const BhMom *mom, Mom64 &M) {
  for (int t = 0; t < 3; ++t) M.c[t] = 0;
  for (int t = 0; t < 9; ++t) M.D[t] = 0;
  for (int t = 0; t < 18; ++t) M.Q[t] = 0;
  {
    const BhRange rc[2] = {range[ch.x], range[ch.y]};
    const int cid[2] = {ch.x, ch.y};
    double cb[2][6];
    for (int side = 0; side < 2; ++side) {
      if (rc[side].hi - rc[side].lo <= direct) leaf_box(rc[side], sp, cb[side]);
      else
        for (int t = 0; t < 6; ++t) cb[side][t] = m64[cid[side]].box[t];
    }
    for (int d = 0; d < 3; ++d) {
      M.box[d] = fmin(cb[0][d], cb[1][d]);
      M.box[3 + d] = fmax(cb[0][3 + d], cb[1][3 + d]);
    }
    double ctr[3];
    for (int d = 0; d < 3; ++d) ctr[d] = 0.5 * (M.box[3 + d] + M.box[d]);
    // a child's moments about its own box centre (an FP64 record, or the FP32
    // record of a child of at most `direct` segments, written by an earlier
    // launch) shifted to this node's centre
    auto shift_add = [&](const auto &C, const double (&cbox)[6]) {
      double r[3];
      for (int d = 0; d < 3; ++d) r[d] = 0.5 * (cbox[3 + d] + cbox[d]) - ctr[d];
      double cc[3];
      for (int i = 0; i < 3; ++i) cc[i] = C.c[i];
      for (int kk = 0; kk < 3; ++kk) {
        double dk[3];
        for (int j = 0; j < 3; ++j) dk[j] = C.D[3 * kk + j];
        for (int i = 0; i < 3; ++i)
          for (int j = i; j < 3; ++j)
            M.Q[6 * kk + qidx(i, j)] += (double)C.Q[6 * kk + qidx(i, j)] + r[j] * dk[i] + r[i] * dk[j] +
                                        cc[kk] * (r[i] * r[j]);
        for (int j = 0; j < 3; ++j) M.D[3 * kk + j] += dk[j] + cc[kk] * r[j];
        M.c[kk] += cc[kk];
      }
    };
    for (int side = 0; side < 2; ++side) {
      if (rc[side].hi - rc[side].lo <= direct) shift_add(mom[cid[side]], cb[side]);
      else shift_add(m64[cid[side]], cb[side]);
    }
  }
}

// Bottom-up moments of one level (children already done) and the node's FP32
// records.  A node of at most `direct` segments (leaf buckets and the small
// subtrees above them, which are most of the nodes) gets direct_records and
// keeps no FP64 record; a larger node shifts each child's moments to its own
// centre with the shift formulas of the reference (compute_link.cpp:358-389,
// Eqs. 21-23): a larger child's FP64 record, or a small child's FP32 record.  Only nodes above
// `direct` segments write FP64 records, so the bottom levels never round-trip
// them through memory.  Children are read one at a time.
template <typename SP>
__device__ __forceinline__ void moments_wave(const BhRange *__restrict__ range, int32_t k0, int32_t n, int32_t base,
                                             int32_t direct, const int2 *__restrict__ child,
                                             const SP *__restrict__ sp, Mom64 *m64, BhGeo *geo, BhMom *mom,
                                             float4 *stage) {
  const int k = k0 + (threadIdx.x & 63), nw = min(64, n - k0);
  BhGeo gr;
  BhMom m;
  Mom64 M;
  bool fp64 = false;
  if (k < n) {
    const int id = base + k;
    const int2 ch = child[id];
    const BhRange rr = range[id];
    if (ch.x < 0 || rr.hi - rr.lo <= direct) {
      direct_records(rr, ch, sp, gr, m);
    } else {
      fp64 = true;
      node_moments(rr, ch, direct, range, sp, m64, mom, M);
      node_records(M, ch, rr, gr, m);
    }
  }
  wave_store_m64(M, __ballot(fp64), m64 + base + k0, nw, stage);
  wave_store_records(gr, m, geo + base + k0, mom + base + k0, nw, stage);
}

template <typename SP>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(3))) void bh_moments(
    const BhRange *__restrict__ range, int32_t n, int32_t base, int32_t direct, const int2 *__restrict__ child,
    const SP *__restrict__ sp, Mom64 *__restrict__ m64, BhGeo *__restrict__ geo, BhMom *__restrict__ mom) {
  __shared__ float4 stage[2][18 * 16];
  const int w = threadIdx.x >> 6;
  const int k0 = blockIdx.x * blockDim.x + w * 64;  // this wave's first node past base
  if (k0 >= n) return;                                // whole wave: no LDS exchange to join
  moments_wave(range, k0, n, base, direct, child, sp, m64, geo, mom, stage[w]);
}

// The top levels, `top` to 0, in one launch: a block takes a curve's levels of at
// most 128 nodes one after the other, its own stores read back after a barrier.
// A launch each they took 5-17 us a level, most of it latency and the launch:
// 400 curves of 4e5 segments 115 -> 63 us, 1,000 of 3.1e7 141 -> 114.
constexpr int kTopLevels = 8;
template <typename SP>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(3))) void bh_moments_top(
    const BhRange *__restrict__ range, int32_t nc, BhLevels L, const int32_t *__restrict__ loff, int32_t top,
    int32_t direct, const int2 *__restrict__ child, const SP *__restrict__ sp, Mom64 *m64, BhGeo *geo, BhMom *mom) {
  static_assert(1 << (kTopLevels - 1) <= 128, "a level's nodes fit the block");
  __shared__ float4 stage[2][18 * 16];
  const int w = threadIdx.x >> 6, c = blockIdx.x;
  for (int lev = top; lev >= 0; --lev) {
    const int32_t *row = loff + (int64_t)lev * nc;
    const int32_t first = row[c], n = (c + 1 < nc ? row[c + 1] : L.base[lev + 1] - L.base[lev]) - first;
    if (64 * w < n)
      moments_wave(range, 64 * w, n, L.base[lev] + first, direct, child, sp, m64, geo, mom, stage[w]);
    __syncthreads();
  }
}

// ---------------------------------------------------------------- far field
struct F3 {
  float x, y, z;
};
__device__ __forceinline__ F3 f3(float a, float b, float c) { return F3{a, b, c}; }
__device__ __forceinline__ float dot3(F3 a, F3 b) { return fmaf(a.x, b.x, fmaf(a.y, b.y, a.z * b.z)); }
__device__ __forceinline__ F3 cross3(F3 a, F3 b) {
  return f3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ F3 add3(F3 a, F3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ F3 sub3(F3 a, F3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ F3 Dv(const float *D, F3 v) {  // D v
  return f3(fmaf(D[0], v.x, fmaf(D[1], v.y, D[2] * v.z)), fmaf(D[3], v.x, fmaf(D[4], v.y, D[5] * v.z)),
            fmaf(D[6], v.x, fmaf(D[7], v.y, D[8] * v.z)));
}
__device__ __forceinline__ F3 DTv(const float *D, F3 v) {  // D^T v
  return f3(fmaf(D[0], v.x, fmaf(D[3], v.y, D[6] * v.z)), fmaf(D[1], v.x, fmaf(D[4], v.y, D[7] * v.z)),
            fmaf(D[2], v.x, fmaf(D[5], v.y, D[8] * v.z)));
}
// Q_k v  (row i: sum_j Q_k,ij v_j) from the symmetric packing
__device__ __forceinline__ F3 Qv(const float *Q, int k, F3 v) {
  const float *q = Q + 6 * k;
  return f3(fmaf(q[0], v.x, fmaf(q[1], v.y, q[2] * v.z)), fmaf(q[1], v.x, fmaf(q[3], v.y, q[4] * v.z)),
            fmaf(q[2], v.x, fmaf(q[4], v.y, q[5] * v.z)));
}
__device__ __forceinline__ float Qel(const float *Q, int k, int i, int j) { return Q[6 * k + qidx(i, j)]; }

// Second-order far field between node A (curve 1) and node B (curve 2) with
// r = ctr_B - ctr_A: returns the linking-number contribution and writes the
// Eq. 14 error estimate (both already multiplied by 1/(4 pi |r|^3)).
__device__ float far_field(const BhMom &A, const BhMom &B, const BhGeo &GA, const BhGeo &GB, F3 r,
                           float dsq, float &err) {
  const F3 ca = f3(A.c[0], A.c[1], A.c[2]), cb = f3(B.c[0], B.c[1], B.c[2]);
  const F3 wa = f3(A.D[5] - A.D[7], A.D[6] - A.D[2], A.D[1] - A.D[3]);
  const F3 wb = f3(B.D[5] - B.D[7], B.D[6] - B.D[2], B.D[1] - B.D[3]);
  const float ir2 = 1.0f / dsq;
  float acc = dot3(r, cross3(cb, ca));  // monopole
  // dipole (Eq. 29)
  acc -= dot3(ca, wb) + dot3(wa, cb);
  acc -= 3.0f * ir2 * (dot3(cross3(Dv(B.D, r), ca), r) + dot3(cross3(Dv(A.D, r), cb), r));
  // quadrupole (Eq. 30)
  const F3 ta = f3(Qel(A.Q, 0, 0, 0) + Qel(A.Q, 0, 1, 1) + Qel(A.Q, 0, 2, 2),
                   Qel(A.Q, 1, 0, 0) + Qel(A.Q, 1, 1, 1) + Qel(A.Q, 1, 2, 2),
                   Qel(A.Q, 2, 0, 0) + Qel(A.Q, 2, 1, 1) + Qel(A.Q, 2, 2, 2));
  const F3 tb = f3(Qel(B.Q, 0, 0, 0) + Qel(B.Q, 0, 1, 1) + Qel(B.Q, 0, 2, 2),
                   Qel(B.Q, 1, 0, 0) + Qel(B.Q, 1, 1, 1) + Qel(B.Q, 1, 2, 2),
                   Qel(B.Q, 2, 0, 0) + Qel(B.Q, 2, 1, 1) + Qel(B.Q, 2, 2, 2));
  const float s2a = -dot3(r, add3(cross3(ta, cb), cross3(ca, tb)));
  auto rd = [](const float *X, int a, const float *Y, int b) {
    return fmaf(X[3 * a], Y[3 * b], fmaf(X[3 * a + 1], Y[3 * b + 1], X[3 * a + 2] * Y[3 * b + 2]));
  };
  const float s2b = 2.0f * (r.x * (rd(A.D, 1, B.D, 2) - rd(A.D, 2, B.D, 1)) +
                            r.y * (rd(A.D, 2, B.D, 0) - rd(A.D, 0, B.D, 2)) +
                            r.z * (rd(A.D, 0, B.D, 1) - rd(A.D, 1, B.D, 0)));
  // u_i = eps_ijk (Q_j r)_k ... as (Q1 r)_2 - (Q2 r)_1 etc.
  const F3 a0 = Qv(A.Q, 0, r), a1 = Qv(A.Q, 1, r), a2 = Qv(A.Q, 2, r);
  const F3 b0 = Qv(B.Q, 0, r), b1 = Qv(B.Q, 1, r), b2 = Qv(B.Q, 2, r);
  const F3 ua = f3(a1.z - a2.y, a2.x - a0.z, a0.y - a1.x);
  const F3 ub = f3(b1.z - b2.y, b2.x - b0.z, b0.y - b1.x);
  float s3 = dot3(cb, ua) - dot3(ca, ub);
  s3 += dot3(r, sub3(DTv(A.D, wb), DTv(B.D, wa)));
  const F3 rra = f3(dot3(r, a0), dot3(r, a1), dot3(r, a2));
  const F3 rrb = f3(dot3(r, b0), dot3(r, b1), dot3(r, b2));
  const float s1 = -dot3(r, cross3(cb, rra)) + dot3(r, cross3(ca, rrb)) +
                   2.0f * dot3(Dv(A.D, r), cross3(r, Dv(B.D, r)));
  acc -= 1.5f * ir2 * ((s2a + s2b + 2.0f * s3) + 5.0f * ir2 * s1);
  const float mult = ir2 * __builtin_amdgcn_rsqf(dsq) * kInv4PiF;
  err = mult * ir2 *
        (GA.qn * (GA.radius * GB.cn + 3.0f * geo_dn(GB)) + GB.qn * (GB.radius * GA.cn + 3.0f * geo_dn(GA)));
  return mult * acc;
}

// Reference leaf term (compute_link.cpp:576-606) from relative midpoint r and
// tangents t1, t2: det == 0 handled with copysign as the reference does.
__device__ __forceinline__ float leaf_term(F3 r, F3 t1, F3 t2) {
  const float det = dot3(r, cross3(t2, t1));
  const F3 a = f3(fmaf(0.5f, t1.x - t2.x, r.x), fmaf(0.5f, t1.y - t2.y, r.y), fmaf(0.5f, t1.z - t2.z, r.z));
  const F3 b = f3(fmaf(-0.5f, t1.x + t2.x, r.x), fmaf(-0.5f, t1.y + t2.y, r.y), fmaf(-0.5f, t1.z + t2.z, r.z));
  const F3 c = f3(fmaf(0.5f, t2.x - t1.x, r.x), fmaf(0.5f, t2.y - t1.y, r.y), fmaf(0.5f, t2.z - t1.z, r.z));
  const F3 d = f3(fmaf(0.5f, t2.x + t1.x, r.x), fmaf(0.5f, t2.y + t1.y, r.y), fmaf(0.5f, t2.z + t1.z, r.z));
  const float la = sqrtf(dot3(a, a)), lb = sqrtf(dot3(b, b)), lc = sqrtf(dot3(c, c)), ld = sqrtf(dot3(d, d));
  const float ac = dot3(a, c);
  const float div1 = la * lb * lc + dot3(a, b) * lc + ac * lb + dot3(b, c) * la;
  const float div2 = la * ld * lc + dot3(a, d) * lc + ac * ld + dot3(d, c) * la;
  const float xp = fmaf(div1, div2, -det * det);
  const float s = det == 0.f ? copysignf(1.f, div1) + copysignf(1.f, div2) : div1 + div2;
  const float yp = det * s;
  const float sg = det == 0.f ? -copysignf(1.f, div1) : copysignf(1.f, det);
  return kInv2PiF * atan2f(yp, xp) + ((s < 0.f || (s == 0.f && det < 0.f)) ? sg : 0.f);
}

// Wave-aggregated append of `cnt` slots; returns this lane's first slot.
__device__ __forceinline__ int64_t wave_append(unsigned long long *counter, int cnt) {
  int incl = cnt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off, 64);
    if ((int)(threadIdx.x & 63) >= off) incl += y;
  }
  const int total = __shfl(incl, 63, 64);
  unsigned long long base = 0;
  if ((threadIdx.x & 63) == 63 && total > 0) base = atomicAdd(counter, (unsigned long long)total);
  base = __shfl(base, 63, 64);
  return (int64_t)base + incl - cnt;
}

// Traversal blocks: 256 threads, each classifying IPT items (2, 4 or 8, a
// tunable shape), so one block owns 256 * IPT consecutive items.  Queue slots,
// sums and statistics are reduced in LDS and published with one global atomic
// per block: atomics on a single address serialise across the chip (one per
// wave capped a 4M-item level at ~7 ns per atomic), and one per 1024 items
// removes that ceiling.
constexpr int kTravBlock = 256;

struct TravShared {
  double v[4], e[4];
  int pair[4];
  int scan[4];
  int nsplit, nleaf;
  unsigned long long base[2];
};

// Adds every thread's (pair, v, e) into sum/err.  When all contributions of
// the block share a pair (items of one pair cluster in the queues) this is one
// atomic per quantity per block; mixed waves fall back to one per item.
// Called by every thread of the block.
__device__ void block_pair_add(int pair, bool active, double v, double e, double *__restrict__ sum,
                               double *__restrict__ err, TravShared &sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long act = __ballot(active);
  int p0 = -1;
  bool uniform = true;
  if (act) {
    p0 = __shfl(pair, __ffsll((long long)act) - 1, 64);
    uniform = __ballot(active && pair != p0) == 0;
  }
  if (!uniform && active) {
    atomicAdd(sum + pair, v);
    if (e != 0.0) atomicAdd(err + pair, e);
  }
  double a = (active && uniform) ? v : 0.0, b = (active && uniform) ? e : 0.0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_xor(a, off, 64);
    b += __shfl_xor(b, off, 64);
  }
  __syncthreads();
  if (lane == 0) {
    sh.pair[w] = (act && uniform) ? p0 : -1;
    sh.v[w] = a;
    sh.e[w] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int p = -1;
    bool same = true;
    for (int k = 0; k < kTravBlock / 64; ++k)
      if (sh.pair[k] >= 0) {
        if (p < 0) p = sh.pair[k];
        else if (sh.pair[k] != p) same = false;
      }
    if (p >= 0 && same) {
      double sa = 0.0, sb = 0.0;
      for (int k = 0; k < kTravBlock / 64; ++k)
        if (sh.pair[k] >= 0) {
          sa += sh.v[k];
          sb += sh.e[k];
        }
      atomicAdd(sum + p, sa);
      if (sb != 0.0) atomicAdd(err + p, sb);
    } else if (p >= 0) {
      for (int k = 0; k < kTravBlock / 64; ++k)
        if (sh.pair[k] >= 0) {
          atomicAdd(sum + sh.pair[k], sh.v[k]);
          if (sh.e[k] != 0.0) atomicAdd(err + sh.pair[k], sh.e[k]);
        }
    }
  }
}

// Slot of this lane among the wave's lanes with `pred`, and the wave's
// first slot from an LDS counter (one LDS atomic per wave).
__device__ __forceinline__ int wave_lds_slot(bool pred, int *counter) {
  const unsigned long long m = __ballot(pred);
  if (m == 0) return -1;
  const int lead = __ffsll((long long)m) - 1;
  int base = 0;
  if ((int)(threadIdx.x & 63) == lead) base = atomicAdd(counter, __popcll(m));
  base = __shfl(base, lead, 64);
  const unsigned long long below = m & ((1ull << (threadIdx.x & 63)) - 1ull);
  return pred ? base + __popcll(below) : -1;
}

// Learned criterion inside the level kernel: the network's biases and input
// normalisation, and each wave's rows of features and predictions.
struct MlpShared {
  InferImage img;  // weight fragments in LDS: the level kernel has no VGPRs to spare for them
  __attribute__((aligned(16))) _Float16 xs[kTravBlock / 64][64][16];
  float ys[kTravBlock / 64][64];
  unsigned int evals;  // network evaluations of the block
};
struct NoMlpShared {};

// Predictions of the learned criterion for the wave's 64 items (one per
// lane; log10 of the far-field error, +inf where the decision does not
// depend on it): the features of the items that need the network are
// compacted into the wave's LDS rows and evaluated 16 per tile, all of the
// wave's tiles through each weight fragment read from LDS (infer_tiles), and
// each lane reads its item's prediction back.  Wave-uniform: every lane calls
// it.
__device__ __forceinline__ float wave_predict(bool need, const BhGeo &A, const BhGeo &B, float dsq, MlpShared &ms,
                                              unsigned int &wave_evals) {
  const unsigned long long m = __ballot(need);
  if (m == 0) return __builtin_inff();
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, g = l >> 4, c = l & 15;
  const int pos = __popcll(m & ((1ull << l) - 1ull));
  if (need) {
    float f[FLK_MLP_NFEAT];
    mlp_features_t<true>(A, B, dsq, f);  // log2 features, normalised with mean2 / istd2
    f16x8 v0, v1;
#pragma unroll
    for (int j = 0; j < 8; ++j) v0[j] = (_Float16)((f[j] - ms.img.L.mean2[j]) * ms.img.L.istd2[j]);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v1[j] = (_Float16)(j < FLK_MLP_NFEAT - 8 ? (f[8 + j] - ms.img.L.mean2[8 + j]) * ms.img.L.istd2[8 + j] : 0.f);
    *reinterpret_cast<f16x8 *>(&ms.xs[w][pos][0]) = v0;
    *reinterpret_cast<f16x8 *>(&ms.xs[w][pos][8]) = v1;
  }
  wave_lds_sync();
  const int cnt = __popcll(m);
  wave_evals += (unsigned int)cnt;
  // rows past cnt are zero (their predictions are not kept); four tiles when
  // more than two are needed, else two
  f16x8 bx[4];
  float yv[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int row = 16 * t + c;
    if (g < 2 && row < cnt) bx[t] = *reinterpret_cast<const f16x8 *>(&ms.xs[w][row][8 * g]);
    else
#pragma unroll
      for (int j = 0; j < 8; ++j) bx[t][j] = (_Float16)0.f;
  }
  if (cnt > 32) infer_tiles<4>(LdsWeights{(LdsW *)&ms.img.W, l}, ms.img.L, bx, yv);
  else infer_tiles<2>(LdsWeights{(LdsW *)&ms.img.W, l}, ms.img.L, bx, yv);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int row = 16 * t + c;
    if (g == 0 && row < cnt) ms.ys[w][row] = yv[t];
  }
  wave_lds_sync();
  const float p = need ? ms.ys[w][pos] : __builtin_inff();
  wave_lds_sync();  // every lane has its prediction before the rows are reused
  return p;
}

// Classification of one node pair and, where it is a far field, its value.
struct BhVisit {
  int kind;  // -1 none, 0 leaf pair, 1 far field, 2 split
  int ca, cb;  // the split node's children
  bool split_a;
  float val, err;
};

template <bool MLP, typename MS>
__device__ __forceinline__ BhVisit bh_visit(const BhItem &it, bool live, const BhGeo *__restrict__ geo,
                                            const BhMom *__restrict__ mom, const float *__restrict__ beta2, float eps,
                                            float log_tol, MS &ms, unsigned int &wave_evals) {
  BhVisit out{-1, 0, 0, false, 0.f, 0.f};
  float pv = __builtin_inff();  // learned criterion: predicted log10 far-field error
  // Learned criterion: both node records are loaded once, before the
  // prediction, and kept for the classification (a dead lane reads node 0
  // of its empty item; loading them again after the network's LDS fences
  // cost another round trip: 2x8M learned 11.75 -> 11.15 ms).  Beta loads
  // them inside the live branch (loading them before it measured 4% slower).
  BhGeo A0, B0;
  if constexpr (MLP) {
    A0 = geo[it.a];
    B0 = geo[it.b];
    const float rx = (B0.cx - A0.cx) + (B0.lx - A0.lx), ry = (B0.cy - A0.cy) + (B0.ly - A0.ly),
                rz = (B0.cz - A0.cz) + (B0.lz - A0.lz);
    const float dsq = fmaf(rx, rx, fmaf(ry, ry, rz * rz)) + eps;
    const float rs = A0.radius + B0.radius;
    pv = wave_predict(live && !(A0.c0 < 0 && B0.c0 < 0) && dsq > rs * rs + eps, A0, B0, dsq, ms, wave_evals);
  }
  if (live) {
    const BhGeo A = MLP ? A0 : geo[it.a], B = MLP ? B0 : geo[it.b];
    const F3 r = f3((B.cx - A.cx) + (B.lx - A.lx), (B.cy - A.cy) + (B.ly - A.ly),
                    (B.cz - A.cz) + (B.lz - A.lz));
    const float dsq = dot3(r, r) + eps;
    const bool la = A.c0 < 0, lb = B.c0 < 0;
    const float rs = A.radius + B.radius;
    // Learned criterion: far field when the spheres are disjoint and the
    // predicted log10 error is below the tolerance; the squared predicted
    // error is accumulated (the pair's estimate is the root of the sum, as
    // for independent signs).  Otherwise the reference's beta test.
    const bool far = MLP ? (dsq > rs * rs + eps && pv < log_tol) : (dsq > rs * rs * beta2[it.pair] + eps);
    if (la && lb) {
      out.kind = 0;
    } else if (far) {
      out.kind = 1;
      out.val = far_field(node_mom(mom, it.a, A), node_mom(mom, it.b, B), A, B, r, dsq, out.err);
      if (MLP) out.err = exp10f(2.0f * pv);
    } else {
      out.kind = 2;
      out.split_a = (!la && !lb) ? !(B.rsq > A.rsq) : lb;
      out.ca = out.split_a ? A.c0 : B.c0;
      out.cb = out.split_a ? A.c1 : B.c1;
    }
  }
  return out;
}

// The network's LDS image, every load of a thread in flight at once.  Ends
// with a barrier.
__device__ __forceinline__ void load_infer_image(const InferImage *__restrict__ mlp_img, MlpShared &ms) {
  constexpr int kWords = (int)(sizeof(InferImage) / 16);
  static_assert(kWords > 3 * kTravBlock && kWords <= 4 * kTravBlock, "four 16-byte words per thread");
  const int4 *src = reinterpret_cast<const int4 *>(mlp_img) + threadIdx.x;
  int4 *dst = reinterpret_cast<int4 *>(&ms.img) + threadIdx.x;
  const bool w3 = 3 * kTravBlock + (int)threadIdx.x < kWords;
  const int4 v0 = src[0], v1 = src[kTravBlock], v2 = src[2 * kTravBlock];
  const int4 v3 = w3 ? src[3 * kTravBlock] : int4{};
  dst[0] = v0;
  dst[kTravBlock] = v1;
  dst[2 * kTravBlock] = v2;
  if (w3) dst[3 * kTravBlock] = v3;
  if (threadIdx.x == 0) ms.evals = 0;
  __syncthreads();
}

// One traversal level over a chunk of items.  Split items are staged in LDS
// as (pair with the split side in its sign, unsplit node, child 0, child 1)
// from the front of the block's stage, leaf-bucket items from the back; after
// the block has classified its 256 * IPT items the stage is copied out
// coalesced behind one queue atomic each.  A queue past the roots holds these
// records as they are, one for the two items of a split: bound by the bytes it
// moves, a visit reads and writes 8 of the queue instead of 16.  MLP: the learned criterion, its
// network evaluated here on the node records the level already holds (the
// weight fragments in LDS, loaded once per block); *evals counts the
// evaluations.
template <int IPT, bool MLP>
__global__ __launch_bounds__(kTravBlock) __attribute__((amdgpu_waves_per_eu(4))) void bh_level(
    const int4 *__restrict__ items, int64_t n, const unsigned long long *__restrict__ n_dev, int roots,
    const BhGeo *__restrict__ geo, const BhMom *__restrict__ mom, const float *__restrict__ beta2,
    float eps, const InferImage *__restrict__ mlp_img, float log_tol, unsigned long long *__restrict__ evals,
    int4 *__restrict__ next, unsigned long long *__restrict__ next_count, int64_t next_cap,
    BhItem *__restrict__ leaves, unsigned long long *__restrict__ leaf_count, int64_t leaf_cap,
    double *__restrict__ psum, double *__restrict__ perr) {
  constexpr int kTravItems = kTravBlock * IPT;
  // A level enqueued before its count reached the host reads the count from
  // the previous level's queue counter; n is then the bound (the buffer's
  // capacity).  A block takes chunks blockIdx.x, blockIdx.x + gridDim.x, ...:
  // one chunk per block when the grid covers the bound, several on a
  // persistent grid.  The loop condition is uniform across the block.  A
  // count above the bound means the previous level overflowed its buffer
  // (its last item may be unwritten): the level is skipped, and the host,
  // seeing the count, discards the pass.
  if (n_dev) n = level_count(n_dev, n);
  __shared__ int4 stage[kTravItems];
  __shared__ TravShared sh;
  __shared__ std::conditional_t<MLP, MlpShared, NoMlpShared> ms;
  unsigned int wave_evals = 0;
  // Items per chunk: 256 * IPT, or, for a level that one round of the grid
  // covers, the count spread over every block in whole multiples of 256, so
  // a small level costs its threads one or two item iterations (each a chain
  // of dependent loads) instead of IPT.  Uniform across the grid.
  const int64_t gsz = (int64_t)gridDim.x;
  const int64_t csz =
      n <= gsz * kTravItems ? min<int64_t>(kTravItems, ((n + gsz - 1) / gsz + kTravBlock - 1) / kTravBlock * kTravBlock)
                            : kTravItems;
  if constexpr (MLP) {
    if ((int64_t)blockIdx.x * csz >= n) return;  // the whole block, before any barrier
    load_infer_image(mlp_img, ms);
  }
  for (int64_t chunk = blockIdx.x; chunk * csz < n; chunk += gridDim.x) {
  if (threadIdx.x == 0) sh.nsplit = sh.nleaf = 0;
  __syncthreads();
  const int64_t b0 = chunk * csz + threadIdx.x;
  int tp = -1;  // this thread's far-field pair and its running sums
  double tv = 0.0, te = 0.0;
#pragma unroll 1
  for (int k = 0; k < IPT && k * kTravBlock < csz; ++k) {
    const int64_t t = b0 + (int64_t)k * kTravBlock;
    const bool live = t < n;
    BhItem it{0, 0, 0, 0};
    if (live && roots) {
      const int4 r = items[t];
      it = BhItem{r.x, r.y, r.z, 0};
    } else if (live) {  // one of a split node's two children with the other side's node
      const int4 r = items[t >> 1];
      const int c = t & 1 ? r.w : r.z;
      it = r.x < 0 ? BhItem{~r.x, c, r.y, 0} : BhItem{r.x, r.y, c, 0};
    }
    const BhVisit v = bh_visit<MLP>(it, live, geo, mom, beta2, eps, log_tol, ms, wave_evals);
    if (v.kind == 1) {
      if (tp < 0 || tp == it.pair) {
        tp = it.pair;
        tv += (double)v.val;
        te += (double)v.err;
      } else {
        atomicAdd(psum + it.pair, (double)v.val);
        if (v.err != 0.f) atomicAdd(perr + it.pair, (double)v.err);
      }
    }
    const int ss = wave_lds_slot(v.kind == 2, &sh.nsplit);
    if (ss >= 0) stage[ss] = make_int4(v.split_a ? ~it.pair : it.pair, v.split_a ? it.b : it.a, v.ca, v.cb);
    const int sl = wave_lds_slot(v.kind == 0, &sh.nleaf);
    if (sl >= 0) stage[kTravItems - 1 - sl] = make_int4(it.pair, it.a, it.b, 0);
  }
  block_pair_add(tp, tp >= 0, tv, te, psum, perr, sh);
  // block_pair_add ends with every stage write visible (it synchronises)
  const int ns = sh.nsplit, nl = sh.nleaf;
  if (threadIdx.x == 0) {
    sh.base[0] = ns ? atomicAdd(next_count, 2ull * (unsigned long long)ns) : 0ull;
    sh.base[1] = nl ? atomicAdd(leaf_count, (unsigned long long)nl) : 0ull;
  }
  __syncthreads();
  const int64_t bn = (int64_t)sh.base[0], bl = (int64_t)sh.base[1];
  for (int i = threadIdx.x; i < ns; i += kTravBlock)
    if (bn + 2 * (int64_t)i + 1 < next_cap) next[bn / 2 + i] = stage[i];
  for (int i = threadIdx.x; i < nl; i += kTravBlock) {
    const int64_t s = bl + i;
    if (s < leaf_cap) {
      const int4 r = stage[kTravItems - 1 - i];
      leaves[s] = BhItem{r.x, r.y, r.z, 0};
    }
  }
  __syncthreads();  // the stage and the shared counters are reused by the next chunk
  }
  if constexpr (MLP) {
    if ((threadIdx.x & 63) == 0 && wave_evals) atomicAdd(&ms.evals, wave_evals);
    __syncthreads();
    if (threadIdx.x == 0 && ms.evals) atomicAdd(evals, (unsigned long long)ms.evals);
  }
}

// One round of a walked pass (the beta criterion's, see PassShape): every wave
// takes chunks of the round's items and walks their whole subtrees of node
// pairs depth first, from a stack of its own in LDS, 64 items a step, one a
// lane, with no barrier.  Splits push their children; leaf pairs gather in LDS
// and leave 64 or more at a time for bh_leaf_pairs.  No wave waits for another:
// once its segment's chunks are all taken and a quarter of its waves have
// ended, a wave still at work leaves its stack to the next round within
// kWalkSteps steps, so a round ends with the chip full, and the first rounds,
// whose few items widen twofold a step, take the work to every wave.  The last
// round leaves nothing.  Items beyond the queue's capacity fail the pass, and the
// host re-runs the batch.
// Level by level the 2 x depth + 1 launches cost 5-10 us each whatever they do:
// device time of certificates of ten loops of 2,000-4,000 vertices (10 pairs)
// 473 -> 336 us, 400 rings of 64-4,096 (1,038 pairs) 1,004 -> 706 us, 2,000
// rings of 64-16,384 2.73 -> 2.26 ms, two random walks of 5,000 0.68 -> 0.58 ms.
// Counters that every wave of the chip would update or read serialise it (about
// 7 ns each on one address), so the queues, the leaf list and their counters
// come in kSegs segments on lines of their own, one for every 16 blocks, each
// of one XCD; a round takes its chunks from all segments alike.
constexpr int kWalkSteps = 8;
constexpr int kSegs = 64;
constexpr int kLine = 16;  // words of a counter line (128 bytes)

// Counter words of a pass.  Walked: [4] root items, [6] set when the leaf list
// could not hold every item, and lines of
// the segments' totals (visits, splits, -, leaf items, leaf segment pairs) and,
// for each round, of its items, the chunks taken of it and the waves that have
// ended.  Level by level: [2] leaf segment pairs, [3] network evaluations, [4 +
// 2d] the items of level d, [5] leaf items.  bh_merge makes of either the
// kPassHead words that the host reads: visits, splits, leaf segment pairs,
// evaluations, root items, leaf items, overflow.
constexpr int kPassHead = 8;
constexpr int kMaxLevels = 1000;
__host__ __device__ __forceinline__ int pass_words(int rounds) { return 16 + kLine * kSegs * (2 + rounds); }
static_assert(16 + kLine * kSegs * 2 >= 4 + 2 * (kMaxLevels + 1), "a level pass's counters fit");
__host__ __device__ __forceinline__ unsigned long long *seg_totals(unsigned long long *cnt, int seg) {
  return cnt + 16 + kLine * seg;
}
__host__ __device__ __forceinline__ unsigned long long *seg_round(unsigned long long *cnt, int round, int seg) {
  return cnt + 16 + kLine * (kSegs * (1 + round) + seg);
}

constexpr int kStack = 512, kLeaves = 128;
constexpr int kDepth = 2 * 31;              // two trees of at most 2^30 segments
constexpr int kWide = kStack - 64;
static_assert(kWide + kDepth <= kStack, "a walk's stack holds what its newest item adds");
struct WalkLds {  // a wave's stack (circular) and its leaf pairs waiting to leave
  int p[kStack], a[kStack], b[kStack];
  int lp[kLeaves], la[kLeaves], lb[kLeaves];
};

__global__ __launch_bounds__(kTravBlock) __attribute__((amdgpu_waves_per_eu(4))) void bh_walk(
    const BhItem *__restrict__ items, int64_t cap, const BhGeo *__restrict__ geo, const BhMom *__restrict__ mom,
    const float *__restrict__ beta2, float eps, unsigned long long *__restrict__ cnt, int round, int last,
    BhItem *__restrict__ next, BhItem *__restrict__ leaves, double *__restrict__ psum, double *__restrict__ perr,
    int copies, int64_t copy_stride) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int seg = blockIdx.x & (kSegs - 1);
  const int64_t seg_cap = cap / kSegs;
  // the round's items: its segments' counts (round 0: the roots), lane s first
  // holding segment s's end
  int64_t end = 0;
  if (round == 0) end = (int64_t)cnt[4];
  else {
    end = level_count(seg_round(cnt, round, lane), seg_cap);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int64_t u = __shfl_up(end, d, 64);
      if (lane >= d) end += u;
    }
  }
  const int64_t n = __shfl(end, 63, 64);
  // chunks of 1 to 64 items, two for each wave of the grid when there are
  // enough; a segment's waves take every kSegs-th chunk, in turn
  const int64_t nwaves = (int64_t)gridDim.x * (kTravBlock / 64);
  const int64_t csz = max((int64_t)1, min((int64_t)64, n / (2 * nwaves)));
  const int64_t nchunks = (n + csz - 1) / csz;
  const int64_t mine = nchunks > seg ? (nchunks - seg + kSegs - 1) / kSegs : 0;
  const int64_t seg_wave = (int64_t)(blockIdx.x / kSegs) * (kTravBlock / 64);  // this block's first wave of its segment
  if (seg_wave >= mine) return;  // the whole block, before any barrier
  __shared__ WalkLds lds[kTravBlock / 64];
  __shared__ int64_t ends[kSegs];
  __shared__ TravShared sh;
  if (w == 0) ends[lane] = end;
  if (threadIdx.x < 2) sh.base[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t below = (1ull << lane) - 1ull;
  unsigned long long *totals = seg_totals(cnt, seg);
  unsigned long long *taken = seg_round(cnt, round, seg) + 1, *nextq = seg_round(cnt, round + 1, seg);
  WalkLds &L = lds[w];
  unsigned long long visits = 0, splits = 0;  // of the wave
  int tp = -1;  // this lane's far-field pair and its running sums
  double tv = 0.0, te = 0.0;
  psum += (blockIdx.x % (unsigned)copies) * copy_stride;
  perr += (blockIdx.x % (unsigned)copies) * copy_stride;
  auto wrap = [](int k) { return k < kStack ? k : k - kStack; };
  int nleaf = 0, leaf_seg = seg;
  // A segment's share of the leaf list that is full sends the rest to the next
  // one's: shares fill unevenly, by a tenth of the list and more.
  auto flush_leaves = [&]() {
    wave_lds_sync();
    for (int from = 0, full = 0; from < nleaf && full < kSegs;) {
      unsigned long long at = 0;
      if (lane == 0) at = atomicAdd(seg_totals(cnt, leaf_seg) + 3, (unsigned long long)(nleaf - from));
      at = __shfl(at, 0, 64);
      const int fits = (int)max((int64_t)0, min((int64_t)(nleaf - from), seg_cap - (int64_t)at));
      for (int i = lane; i < fits; i += 64)
        leaves[leaf_seg * seg_cap + (int64_t)at + i] = BhItem{L.lp[from + i], L.la[from + i], L.lb[from + i], 0};
      from += fits;
      if (from < nleaf) {
        leaf_seg = (leaf_seg + 1) & (kSegs - 1);
        if (++full == kSegs && lane == 0) atomicOr(cnt + 6, 1ull);
      }
    }
    wave_lds_sync();
    nleaf = 0;
  };
  NoMlpShared no_mlp;
  unsigned int no_evals = 0;
  int bot = 0, num = 0;
  int64_t chunk = seg_wave + w;  // of the segment's chunks; a wave's first is its own
  const int64_t seg_waves = (int64_t)((gridDim.x - seg + kSegs - 1) / kSegs) * (kTravBlock / 64);
  // none left to take once every chunk is some wave's first
  bool more = chunk < mine, drained = mine <= seg_waves;
  const int started = (int)min(mine, seg_waves);
  // waves of the segment that ended before the others share what is left
  const int enough = started - (int)(seg_waves * 3 / 4);
  bool starving = drained && enough <= 0;
  int steps = kWalkSteps, tick = 0;
  while (more || num > 0) {
    if (more && num < 64) {
      const int64_t c0 = (chunk * kSegs + seg) * csz;
      const int m = (int)min(csz, n - c0);
      if (lane < m) {
        int64_t at = c0 + lane;
        if (round > 0) {  // the segment that holds item `at`: ends before it
          int lo = 0;
#pragma unroll
          for (int d = kSegs / 2; d > 0; d >>= 1)
            if (ends[lo + d - 1] <= at) lo += d;
          at += lo * seg_cap - (lo ? ends[lo - 1] : 0);
        }
        const BhItem it = items[at];
        const int k = wrap(wrap(bot + num) + lane);
        L.p[k] = it.pair;
        L.a[k] = it.a;
        L.b[k] = it.b;
      }
      num += m;
      wave_lds_sync();
      if (drained) {
        more = false;
      } else {
        unsigned long long c = 0;
        if (lane == 0) c = atomicAdd(taken, 1ull);
        chunk = seg_waves + (int64_t)__shfl(c, 0, 64);
        if (chunk >= mine) more = false;
      }
      continue;
    }
    // the oldest items go to the next round when the stack could overflow, and
    // all of them kWalkSteps steps after the segment's chunks ran out
    const int out = last ? 0 : steps <= 0 ? num : num > kWide ? num / 2 : 0;
    if (out) {
      unsigned long long at = 0;
      if (lane == 0) at = atomicAdd(nextq, (unsigned long long)out);
      at = __shfl(at, 0, 64);
      for (int i = lane; i < out; i += 64) {
        const int k = wrap(bot + i);
        if ((int64_t)at + i < seg_cap) next[seg * seg_cap + (int64_t)at + i] = BhItem{L.p[k], L.a[k], L.b[k], 0};
      }
      wave_lds_sync();
      bot = wrap(bot + out);
      num -= out;
      continue;
    }
    // In the last round a filling stack narrows the steps: those of several items
    // leave it at kWide at most, and the newest item alone adds no more than the
    // splits above a leaf pair, kDepth, before it is done.
    const int take = last ? max(1, min(min(num, 64), kWide - num)) : min(num, 64);
    num -= take;
    const int base = wrap(bot + num);
    const bool live = lane < take;
    const int k0 = wrap(base + lane);
    BhItem it{0, 0, 0, 0};
    if (live) it = BhItem{L.p[k0], L.a[k0], L.b[k0], 0};
    unsigned long long poll = 0;
    const bool look = !starving && (++tick & 7) == 0;
    if (look) poll = __hip_atomic_load(taken + (drained ? 1 : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    wave_lds_sync();  // every item is in registers before its slot is reused
    const BhVisit v = bh_visit<false>(it, live, geo, mom, beta2, eps, 0.f, no_mlp, no_evals);
    if (v.kind == 1) {
      if (tp < 0 || tp == it.pair) {
        tp = it.pair;
        tv += (double)v.val;
        te += (double)v.err;
      } else {
        atomicAdd(psum + it.pair, (double)v.val);
        if (v.err != 0.f) atomicAdd(perr + it.pair, (double)v.err);
      }
    }
    const uint64_t ms2 = __ballot(v.kind == 2), ms0 = __ballot(v.kind == 0);
    if (v.kind == 2) {
      const int k = wrap(base + 2 * __popcll(ms2 & below));
      const int k1 = wrap(k + 1);
      L.p[k] = L.p[k1] = it.pair;
      L.a[k] = v.split_a ? v.ca : it.a;
      L.b[k] = v.split_a ? it.b : v.ca;
      L.a[k1] = v.split_a ? v.cb : it.a;
      L.b[k1] = v.split_a ? it.b : v.cb;
    } else if (v.kind == 0) {
      const int k = nleaf + __popcll(ms0 & below);
      L.lp[k] = it.pair;
      L.la[k] = it.a;
      L.lb[k] = it.b;
    }
    const int ns = __popcll(ms2);
    num += 2 * ns;
    nleaf += __popcll(ms0);
    visits += (unsigned long long)take;
    splits += (unsigned long long)ns;
    wave_lds_sync();
    if (nleaf > kLeaves - 64) flush_leaves();
    // `taken` runs past the end once a wave found no chunk
    const int polled = __builtin_amdgcn_readfirstlane((int)min(poll, 0x7fffffffull));
    if (starving) --steps;
    else if (!look) continue;
    else if (drained) starving = polled >= enough;
    else drained = seg_waves + (int64_t)polled > mine;
  }
  if (lane == 0 && visits) atomicAdd(taken + 1, 1ull);
  if (nleaf) flush_leaves();
  block_pair_add(tp, tp >= 0, tv, te, psum, perr, sh);
  __syncthreads();
  if (lane == 0) {
    atomicAdd(&sh.base[0], visits);
    atomicAdd(&sh.base[1], splits);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicAdd(totals, sh.base[0]);
    atomicAdd(totals + 1, sh.base[1]);
  }
}

// Exact evaluation of leaf-bucket pairs: every segment pair of the two
// buckets with the reference leaf term, from FP32 hi/lo vertices (two
// one-segment leaves: from their node records, which hold the midpoints and
// the edge vectors).  Blocks of
// 256 * IPT items as in bh_level; *counters gets the segment-pair count.
// With a device-scheduled pass's counters (cnt) n is the list's capacity and the
// count is read there: a level pass's list is one, a walked pass's comes in
// segments, block b taking segment b % kSegs, its sums going to one of the
// sums' copies.
template <int IPT>
__global__ __launch_bounds__(kTravBlock) void bh_leaf_pairs(
    const BhItem *__restrict__ items, int64_t n, unsigned long long *__restrict__ cnt, int walked,
    const BhGeo *__restrict__ geo, const uint32_t *__restrict__ order, const float4 *__restrict__ hi,
    const float4 *__restrict__ lo, const float4 *__restrict__ ed, double *__restrict__ psum,
    double *__restrict__ perr, unsigned long long *__restrict__ counters, int copies, int64_t copy_stride) {
  constexpr int kTravItems = kTravBlock * IPT;
  int64_t first = blockIdx.x, stride = gridDim.x;
  int64_t csz = kTravItems;
  if (cnt) {
    unsigned long long *count = cnt + 5;
    counters = cnt + 2;
    if (walked) {
      const int seg = blockIdx.x & (kSegs - 1);
      n /= kSegs;
      items += seg * n;
      count = seg_totals(cnt, seg) + 3;
      counters = count + 1;
      first = blockIdx.x / kSegs;
      stride = gridDim.x / kSegs;
      psum += (blockIdx.x % (unsigned)copies) * copy_stride;
      perr += (blockIdx.x % (unsigned)copies) * copy_stride;
    }
    // (a walked share may have been asked for more than it holds)
    n = walked ? min((int64_t)*count, n) : level_count(count, n);
    if (n == 0) return;
    // a short list spread over the blocks in whole multiples of 256
    csz = min<int64_t>(csz, ((n + stride - 1) / stride + kTravBlock - 1) / kTravBlock * kTravBlock);
  }
  __shared__ TravShared sh;
  int npairs = 0;
  for (int64_t chunk = first; chunk * csz < n; chunk += stride) {
  const int64_t b0 = chunk * csz + threadIdx.x;
  int tp = -1;
  double tv = 0.0;
#pragma unroll 1
  for (int k = 0; k < IPT && k * kTravBlock < csz; ++k) {
    const int64_t t = b0 + (int64_t)k * kTravBlock;
    if (t >= n) break;
    const BhItem it = items[t];
    const BhGeo A = geo[it.a], B = geo[it.b];
    float acc = 0.f;
    if (is_leaf_segment(A) && is_leaf_segment(B)) {
      // one segment each: the records already hold the midpoints (the box
      // centres, hi/lo) and the FP32 edge vectors, so no vertex is read
      const F3 r = f3((B.cx - A.cx) + (B.lx - A.lx), (B.cy - A.cy) + (B.ly - A.ly), (B.cz - A.cz) + (B.lz - A.lz));
      acc = leaf_term(r, f3(__builtin_bit_cast(float, A.c1), A.pad, A.dn),
                      f3(__builtin_bit_cast(float, B.c1), B.pad, B.dn));
      ++npairs;
    } else {
      for (int i = A.seg0; i < A.seg0 + A.nseg; ++i) {
        const uint32_t va = order[i];
        const float4 pa = hi[va], pb = hi[va + 1], qa = lo[va], qb = lo[va + 1], ea = ed[va];
        for (int j = B.seg0; j < B.seg0 + B.nseg; ++j) {
          const uint32_t vb = order[j];
          const float4 ra = hi[vb], rb = hi[vb + 1], sa = lo[vb], sb = lo[vb + 1], eb = ed[vb];
          // r = m2 - m1 = ((q0 - p0) + (q1 - p1)) / 2, each difference hi/lo exact
          const F3 r = f3(0.5f * (((ra.x - pa.x) + (sa.x - qa.x)) + ((rb.x - pb.x) + (sb.x - qb.x))),
                          0.5f * (((ra.y - pa.y) + (sa.y - qa.y)) + ((rb.y - pb.y) + (sb.y - qb.y))),
                          0.5f * (((ra.z - pa.z) + (sa.z - qa.z)) + ((rb.z - pb.z) + (sb.z - qb.z))));
          acc += leaf_term(r, f3(ea.x, ea.y, ea.z), f3(eb.x, eb.y, eb.z));
          ++npairs;
        }
      }
    }
    if (tp < 0 || tp == it.pair) {
      tp = it.pair;
      tv += (double)acc;
    } else {
      atomicAdd(psum + it.pair, (double)acc);
    }
  }
  block_pair_add(tp, tp >= 0, tv, 0.0, psum, perr, sh);
  __syncthreads();  // sh is reused by the next chunk
  }
  int tot = npairs;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off, 64);
  if ((threadIdx.x & 63) == 0) sh.scan[threadIdx.x >> 6] = tot;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long s = 0;
    for (int k = 0; k < kTravBlock / 64; ++k) s += (unsigned long long)sh.scan[k];
    if (s) atomicAdd(counters, s);
  }
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  return z ^ (z >> 31);
}

// Training-sample traversal level: every node pair with disjoint bounding
// spheres is a candidate sample (kept with probability p when the exact label
// costs at most max_pairs segment pairs); pairs are split further until they
// pass beta_stop, so samples cover 1 < |r|/(r1+r2) <= beta_stop at every depth.
__global__ __launch_bounds__(256) void bh_sample_level(
    const BhItem *__restrict__ items, int64_t n, const BhGeo *__restrict__ geo, float eps,
    float stop2, double p, uint64_t seed, int64_t max_pairs, BhItem *__restrict__ next,
    unsigned long long *__restrict__ next_count, BhItem *__restrict__ samp,
    unsigned long long *__restrict__ samp_count, int64_t samp_cap) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = t < n;
  BhItem it = live ? items[t] : BhItem{0, 0, 0, 0};
  bool split = false, keep = false;
  int ca = 0, cb = 0;
  bool split_a = false;
  if (live) {
    const BhGeo A = geo[it.a], B = geo[it.b];
    const float rx = (B.cx - A.cx) + (B.lx - A.lx), ry = (B.cy - A.cy) + (B.ly - A.ly),
                rz = (B.cz - A.cz) + (B.lz - A.lz);
    const float dsq = rx * rx + ry * ry + rz * rz + eps;
    const bool la = A.c0 < 0, lb = B.c0 < 0;
    const float rs = A.radius + B.radius;
    if (!(la && lb)) {
      if (dsq > rs * rs + eps) {
        const uint64_t h = mix64(seed ^ ((uint64_t)(uint32_t)it.a << 32 | (uint32_t)it.b));
        keep = (int64_t)A.nseg * B.nseg <= max_pairs && (double)(h >> 11) * 0x1.0p-53 < p;
      }
      split = !(dsq > rs * rs * stop2 + eps);
      if (split) {
        split_a = (!la && !lb) ? !(B.rsq > A.rsq) : lb;
        ca = split_a ? A.c0 : B.c0;
        cb = split_a ? A.c1 : B.c1;
      }
    }
  }
  const int64_t s = wave_append(next_count, split ? 2 : 0);
  if (split) {
    if (split_a) {
      next[s] = BhItem{0, ca, it.b, 0};
      next[s + 1] = BhItem{0, cb, it.b, 0};
    } else {
      next[s] = BhItem{0, it.a, ca, 0};
      next[s + 1] = BhItem{0, it.a, cb, 0};
    }
  }
  const int64_t k = wave_append(samp_count, keep ? 1 : 0);
  if (keep && k < samp_cap) samp[k] = it;
}

// FP64 one-arctan segment-pair term (reference compute_link.cpp:151-175) of
// segment p0->p1 against q0->q1, times 4 pi.
__device__ __forceinline__ double pair_term_x4pi_f64(double4 p0, double4 p1, double4 q0, double4 q1) {
  const double ax = q0.x - p0.x, ay = q0.y - p0.y, az = q0.z - p0.z;
  const double bx = q0.x - p1.x, by = q0.y - p1.y, bz = q0.z - p1.z;
  const double cx = q1.x - p1.x, cy = q1.y - p1.y, cz = q1.z - p1.z;
  const double dx = q1.x - p0.x, dy = q1.y - p0.y, dz = q1.z - p0.z;
  const double la = sqrt(ax * ax + ay * ay + az * az), lb = sqrt(bx * bx + by * by + bz * bz);
  const double lc = sqrt(cx * cx + cy * cy + cz * cz), ld = sqrt(dx * dx + dy * dy + dz * dz);
  const double ac = cx * ax + cy * ay + cz * az;
  const double div1 = la * lb * lc + (ax * bx + ay * by + az * bz) * lc + ac * lb + (cx * bx + cy * by + cz * bz) * la;
  const double div2 = la * ld * lc + (ax * dx + ay * dy + az * dz) * lc + ac * ld + (cx * dx + cy * dy + cz * dz) * la;
  const double det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx);
  const double xp = div1 * div2 - det * det, yp = det * (div1 + div2);
  double v = 2.0 * atan2(yp, xp);
  if (yp * det < 0) v += (det > 0 ? 1.0 : -1.0) * 12.566370614359172953850573533118;
  return v;
}

// One wave per sample: exact FP64 sum over the two nodes' segment pairs, the
// FP32 far field, features and the label log10 |exact - far field| (>= -14).
__global__ __launch_bounds__(256) void bh_sample_labels(
    const BhItem *__restrict__ samp, int64_t n, const BhGeo *__restrict__ geo,
    const BhMom *__restrict__ mom, const uint32_t *__restrict__ order,
    const double4 *__restrict__ pts, float eps, float *__restrict__ x, float *__restrict__ y) {
  const int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int l = threadIdx.x & 63;
  if (w >= n) return;
  const BhItem it = samp[w];
  const BhGeo A = geo[it.a], B = geo[it.b];
  double acc = 0.0;
  const int64_t total = (int64_t)A.nseg * B.nseg;
  for (int64_t k = l; k < total; k += 64) {
    const uint32_t va = order[A.seg0 + (int)(k / B.nseg)], vb = order[B.seg0 + (int)(k % B.nseg)];
    acc += pair_term_x4pi_f64(pts[va], pts[va + 1], pts[vb], pts[vb + 1]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (l == 0) {
    const double exact = acc * 0.07957747154594766788444188168625718;
    const F3 r = f3((B.cx - A.cx) + (B.lx - A.lx), (B.cy - A.cy) + (B.ly - A.ly),
                    (B.cz - A.cz) + (B.lz - A.lz));
    const float dsq = dot3(r, r) + eps;
    float e;
    const float ff = far_field(node_mom(mom, it.a, A), node_mom(mom, it.b, B), A, B, r, dsq, e);
    const double d = fabs(exact - (double)ff);
    y[w] = (float)fmax(log10(d), -14.0);
    float f[FLK_MLP_NFEAT];
    mlp_features(A, B, dsq, f);
    for (int k2 = 0; k2 < FLK_MLP_NFEAT; ++k2) x[w * FLK_MLP_NFEAT + k2] = f[k2];
  }
}

__global__ void bh_roots(const int32_t *__restrict__ ra, const int32_t *__restrict__ rb, int64_t n,
                         BhItem *__restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) out[k] = BhItem{(int32_t)k, ra[k], rb[k], 0};
}

// Start of a batch's traversal: its root items, both passes' counters and every
// copy of the sums cleared (a kernel rather than memsets, so it can be
// captured), and the first pass's root count.
__global__ __launch_bounds__(256) void bh_begin(const int32_t *__restrict__ ra, const int32_t *__restrict__ rb,
                                                int64_t nb, BhItem *__restrict__ items,
                                                unsigned long long *__restrict__ cnt, int words, int64_t nsums,
                                                double *__restrict__ sum, double *__restrict__ err) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nb) items[k] = BhItem{(int32_t)k, ra[k], rb[k], 0};
  if (k < 2 * words) cnt[k] = k == 4 ? (unsigned long long)nb : 0ull;
  if (k < nsums) sum[k] = err[k] = 0.0;
}

// The copies of one sum, added in order.
__device__ __forceinline__ double fold_copies(const double *p, int copies, int64_t stride) {
  double v = p[0];
  if (copies == 8) {  // a walk's, in flight at once
    double u[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) u[k] = p[(k + 1) * stride];
#pragma unroll
    for (int k = 0; k < 7; ++k) v += u[k];
    return v;
  }
  for (int k = 1; k < copies; ++k) v += p[k * stride];
  return v;
}

// The re-run decision after a batch's first pass, on the device.  Beta
// (reference linking_number_certificate.cpp:165-184): the estimate scaled by
// err_scale gives the target beta = min(beta_init (E / target)^(1/4),
// beta_limit), and a pair whose target exceeds beta_init is re-run with it.
// Learned criterion: the root-sum-square of the accepted predictions is the
// estimate, and a pair above a tenth of the target is re-run (one decade
// stricter, by the caller's second pass).  One block walks the pairs in order
// and compacts the re-runs with a block scan, so the list is deterministic:
// root items (pair = position in the list), beta^2, and every pair's position
// in it (-1: not re-run).  Sets the second pass's root count.
__global__ __launch_bounds__(1024) void bh_adapt(int64_t nb, const int32_t *__restrict__ ra,
                                                const int32_t *__restrict__ rb, const double *__restrict__ err1,
                                                int copies, int64_t copy_stride, int mlp, double err_scale,
                                                double target_error, double beta_init, double beta_limit,
                                                BhItem *__restrict__ items2, float *__restrict__ beta2_2,
                                                int32_t *__restrict__ redo, unsigned long long *__restrict__ n_redo) {
  __shared__ int sw[16];
  int carry = 0;
  for (int64_t c0 = 0; c0 < nb; c0 += 1024) {
    const int64_t t = c0 + threadIdx.x;
    int flag = 0;
    float b2 = 0.f;
    const double e1 = t < nb ? fold_copies(err1 + t, copies, copy_stride) : 0.0;
    if (t < nb) {
      const double excess = e1 * err_scale / target_error;
      if (!mlp && excess < 0.99 && beta_init > 0.0) {
        // a fourth root below 1: the target lies below beta_init, without the pow
      } else if (!mlp) {
        const double want = pow(excess, 0.25) * beta_init;
        const double target = beta_limit < want ? beta_limit : want;  // std::min: a NaN estimate stays NaN
        if (target > beta_init) {
          flag = 1;
          b2 = (float)(target * target);
        }
      } else if (sqrt(e1) > 0.1 * target_error) {
        flag = 1;
        b2 = (float)(beta_init * beta_init);
      }
    }
    int tot = 0;
    const int pos = carry + block_scan<16>(flag, &tot, sw);
    if (flag) {
      items2[pos] = BhItem{pos, ra[t], rb[t], 0};
      beta2_2[pos] = b2;
    }
    if (t < nb) redo[t] = flag ? pos : -1;
    carry += tot;
  }
  if (threadIdx.x == 0) *n_redo = (unsigned long long)carry;
}

// Per-pair results of a batch: the first pass's sum and estimate (scaled by
// err_scale for beta, the root-sum-square for the learned criterion), or the
// second pass's for a re-run pair; sums of the second pass are at + nb.
// With counters (cnt, null for a host-driven batch) one block more, which makes
// both device-scheduled passes' kPassHead words of them (behind the results of
// block 0 they took it 1 us longer).  levels: how many a level pass has, 0 when walked
// in `rounds`.  An overflow is noted where a queue is over its capacity (its
// segment's share of it), the leaf list is over its own, or items were left after
// the last level.
__global__ __launch_bounds__(256) void bh_merge(int64_t nb, const int32_t *__restrict__ redo,
                                                const double *__restrict__ sum, const double *__restrict__ err,
                                                int copies, int64_t copy_stride, int mlp, double err_scale,
                                                double *__restrict__ v, double *__restrict__ e,
                                                uint32_t *__restrict__ f, unsigned long long *__restrict__ heads,
                                                unsigned long long *__restrict__ cnt, int64_t cap, int levels, int rounds) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < nb) {
    const int32_t r = redo[t];
    const int64_t at = r < 0 ? t : nb + r;
    const double es = fold_copies(err + at, copies, copy_stride);
    v[t] = fold_copies(sum + at, copies, copy_stride);
    e[t] = mlp ? sqrt(es) : es * err_scale;
    f[t] = r < 0 ? 0u : FLK_PAIR_RETRY;
  }
  if (cnt == nullptr || blockIdx.x + 1 != gridDim.x || threadIdx.x >= 2 * kSegs) return;
  const int seg = threadIdx.x & (kSegs - 1), pass = threadIdx.x / kSegs;
  unsigned long long *c = cnt + pass * pass_words(rounds);
  unsigned long long x[kPassHead] = {0, 0, 0, 0, seg == 0 ? c[4] : 0, 0, 0, 0};
  if (levels) {
    for (int d = seg; d <= levels; d += kSegs) {
      const unsigned long long n = c[4 + 2 * d];
      if (d < levels) x[0] += n;
      if (d > 0) x[1] += n / 2;
      if ((int64_t)n > cap || (d == levels && n)) x[6] = 1;
    }
    if (seg == 0) {
      x[2] = c[2];
      x[3] = c[3];
      x[5] = c[5];
      if ((int64_t)c[5] > cap) x[6] = 1;
    }
  } else {
    const unsigned long long *tot = seg_totals(c, seg);
    x[0] = tot[0];
    x[1] = tot[1];
    x[2] = tot[4];
    x[5] = min(tot[3], (unsigned long long)(cap / kSegs));
    if (c[6]) x[6] = 1;
    for (int r = 1; r <= rounds; r += 6) {  // six loads in flight
      unsigned long long most = 0;
#pragma unroll
      for (int k = 0; k < 6; ++k) most = max(most, *seg_round(c, min(r + k, rounds), seg));
      if ((int64_t)most > cap / kSegs) x[6] = 1;
    }
  }
#pragma unroll
  for (int i = 0; i < kPassHead; ++i) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x[i] += __shfl_xor(x[i], d, 64);
    if (seg == 0) heads[pass * kPassHead + i] = x[i];
  }
}

}  // namespace

// ---------------------------------------------------------------- host side
namespace {

// Node records of the trees of one call; the buffers are the context's.

struct Forest {
  int32_t nnodes = 0;
  int32_t depth = 0;          // node levels of the deepest tree
  std::vector<int32_t> root;  // per curve (-1 if no tree)
  DevBuf &geo, &mom, &order;
  explicit Forest(BhScratch &b) : geo(b.geo), mom(b.mom), order(b.order) {}
};

// Host plan of a forest build: the curves with trees (rank order), their
// segment and vertex offsets, key boxes, roots and the level structure, all
// known before anything runs on the device.  plan_forest also reserves every
// buffer the build writes; enqueue_forest then only enqueues (no allocation,
// no read-back), so the build can be captured.  The host arrays are read by
// the build's copies when they run: the plan outlives them.
struct ForestPlan {
  int leaf = 1, direct = kDirectSegments;
  std::vector<int32_t> cs;
  std::vector<int64_t> seg_off, vtx_off;
  std::vector<double> cbox;
  std::vector<RadixTile> tiles;  // the segmented sort's tiles (one curve each)
  std::vector<int32_t> tcurve;   // each tile's curve rank
  std::vector<int32_t> small[kSmallSorts];  // ranks of the curves that one block sorts (see kSmallSort)
  int64_t S = 0;
  std::vector<int32_t> level_base, level_n;
  std::vector<int64_t> level_split, level_max;
  int32_t total = 0;
  int lev_top = 0;
  // the arrays' device addresses (PlanUpload)
  const int64_t *d_seg = nullptr, *d_vtx = nullptr;
  const double *d_box = nullptr;
  const RadixTile *d_tiles = nullptr;
  const int32_t *d_tcurve = nullptr, *d_small[kSmallSorts] = {};
};

// Host arrays of the plans on their way to the device: gathered in one pinned
// buffer and sent as one copy, and the kernels read them where they land (ten
// uploads and ten device copies into scratch took 10 us each).  The buffers are
// the context's: a captured graph's plans are sent again before each launch.
class PlanUpload {
 public:
  template <typename T> void add(const std::vector<T> &v, const T *&where) {
    parts_.push_back({v.data(), sizeof(T) * v.size(), total_, reinterpret_cast<const void **>(&where)});
    total_ += (sizeof(T) * v.size() + 15) & ~size_t(15);
  }
  void send(flk_ctx *ctx, hipStream_t s) {
    BhScratch &B = ctx->bh;
    B.pack.reserve(std::max<size_t>(total_, 16));
    B.pack_host.reserve(std::max<size_t>(total_, 16));
    for (const Part &p : parts_) {
      if (p.bytes) std::memcpy(B.pack_host.as<unsigned char>() + p.off, p.src, p.bytes);
      *p.where = B.pack.as<unsigned char>() + p.off;
    }
    if (total_) FLK_HIP(hipMemcpyAsync(B.pack.ptr, B.pack_host.ptr, total_, hipMemcpyHostToDevice, s));
  }

 private:
  struct Part {
    const void *src;
    size_t bytes, off;
    const void **where;
  };
  std::vector<Part> parts_;
  size_t total_ = 0;
};

void add_forest(PlanUpload &up, ForestPlan &P) {
  up.add(P.seg_off, P.d_seg);
  up.add(P.vtx_off, P.d_vtx);
  up.add(P.cbox, P.d_box);
  up.add(P.tiles, P.d_tiles);
  up.add(P.tcurve, P.d_tcurve);
  for (int k = 0; k < kSmallSorts; ++k) up.add(P.small[k], P.d_small[k]);
}

// The planned curves' key boxes, the one part of a plan that their coordinates
// decide.  Sort keys: a Morton code of 10 bits per axis relative to the curve's
// box (a curve's tree never depends on the batch around it), sorted within each
// curve's range by the segmented sort: 30-bit keys, four passes, whatever the
// number of curves.
void plan_boxes(const Curves &cv, ForestPlan &P) {
  constexpr double cells = 1024.0;
  for (size_t k = 0; k < P.cs.size(); ++k)
    for (int d = 0; d < 3; ++d) {
      const double lo = (cv.box[6 * P.cs[k] + d] - cv.origin[d]) * cv.scale;
      const double hi = (cv.box[6 * P.cs[k] + 3 + d] - cv.origin[d]) * cv.scale;
      P.cbox[6 * k + d] = lo;
      P.cbox[6 * k + 3 + d] = hi > lo ? cells / (hi - lo) : 0.0;
    }
}

void plan_forest(flk_ctx *ctx, const std::vector<int32_t> &curves_in, int leaf, ForestPlan &P) {
  Curves &cv = ctx->curves;
  P = ForestPlan{};
  P.leaf = leaf;
  P.direct = std::max(leaf, kDirectSegments);
  for (int32_t c : curves_in)
    if (cv.n[c] >= 2) P.cs.push_back(c);
  const int32_t nc = (int32_t)P.cs.size();
  if (nc == 0) return;
  if (cv.nvert_dev >= (int64_t)UINT32_MAX) throw Error(FLK_ERR_ARG, "too many vertices for Barnes-Hut");
  P.seg_off.assign(nc + 1, 0);
  P.vtx_off.assign(nc, 0);
  P.cbox.assign(6 * (size_t)nc, 0.0);
  for (int32_t k = 0; k < nc; ++k) {
    P.seg_off[k + 1] = P.seg_off[k] + cv.n[P.cs[k]];
    P.vtx_off[k] = cv.off[P.cs[k]];
  }
  plan_boxes(cv, P);
  const int64_t S = P.S = P.seg_off[nc];
  if (S >= INT32_MAX / 2) throw Error(FLK_ERR_ARG, "too many Barnes-Hut segments");
  for (int32_t k = 0; k < nc; ++k) {
    const int64_t n = P.seg_off[k + 1] - P.seg_off[k];
    int cls = 0;
    while (cls < kSmallSorts && n > kSmallSort[cls]) ++cls;
    if (cls < kSmallSorts) P.small[cls].push_back(k);
  }
  // the shortest join the next class's launch where both are resident at once
  if (!P.small[1].empty() && P.small[0].size() + P.small[1].size() <= 2 * (size_t)std::max(1, ctx->num_cus)) {
    P.small[1].insert(P.small[1].end(), P.small[0].begin(), P.small[0].end());
    P.small[0].clear();
  }
  const int64_t ntiles = segmented_tiles(P.seg_off.data(), nc, kSmallSort[kSmallSorts - 1], P.tiles);
  P.tcurve.resize(ntiles);
  for (int32_t k = 0, t = 0; t < ntiles; ++t) {
    while (P.seg_off[k + 1] <= P.tiles[t].start) ++k;
    P.tcurve[t] = k;
  }
  // Splits per level from the segment counts alone: a range of m > leaf
  // segments splits into floor(m/2) and m - floor(m/2), so every level of a
  // curve's tree holds at most two distinct range sizes (m and m + 1).  With
  // the counts known, the levels are enqueued without reading anything back.
  {
    std::vector<std::pair<int64_t, int64_t>> sizes;  // (range size, count) of the current level
    std::vector<std::pair<int64_t, int64_t>> next;
    for (int32_t k = 0; k < nc; ++k) sizes.emplace_back(P.seg_off[k + 1] - P.seg_off[k], 1);
    for (;;) {
      int64_t split = 0, mx = 0;
      for (const auto &sc : sizes) mx = std::max(mx, sc.first);
      P.level_max.push_back(mx);
      next.clear();
      for (const auto &sc : sizes) {
        if (sc.first <= leaf) continue;
        split += sc.second;
        next.emplace_back(sc.first / 2, sc.second);
        next.emplace_back(sc.first - sc.first / 2, sc.second);
      }
      P.level_split.push_back(split);
      if (split == 0) break;
      // merge equal sizes (keeps the list at two entries per distinct size pair)
      std::sort(next.begin(), next.end());
      sizes.clear();
      for (const auto &sc : next) {
        if (!sizes.empty() && sizes.back().first == sc.first) sizes.back().second += sc.second;
        else sizes.push_back(sc);
      }
    }
  }
  P.level_base.assign(1, 0);
  P.level_n.assign(1, nc);
  int32_t total = nc;
  for (size_t lev = 0; lev < P.level_split.size(); ++lev) {
    const int32_t nsplit = (int32_t)P.level_split[lev];
    if (nsplit == 0) break;
    P.level_base.push_back(total);
    P.level_n.push_back(2 * nsplit);
    total += 2 * nsplit;
  }
  P.total = total;
  // the bottom levels (every range within `direct`) run as one launch
  P.lev_top = (int)P.level_base.size();
  for (int lev = 0; lev < (int)P.level_base.size() && lev < (int)P.level_max.size(); ++lev)
    if (P.level_max[lev] <= P.direct) {
      P.lev_top = lev;
      break;
    }
  // FP64 records exist only for nodes above `direct` segments: node ids are
  // assigned level by level, so they all fall below the first level whose
  // ranges are all that small
  const int64_t m64_nodes = P.lev_top < (int)P.level_base.size() ? P.level_base[P.lev_top] : total;
  BhScratch &B = ctx->bh;
  B.keys0.reserve(sizeof(uint32_t) * S);
  B.keys1.reserve(sizeof(uint32_t) * S);
  B.ids0.reserve(sizeof(uint32_t) * S);
  B.order.reserve(sizeof(uint32_t) * S);
  B.loff.reserve(sizeof(int32_t) * P.level_base.size() * nc);
  B.vals.reserve(sizeof(uint32_t) * S);
  B.tmp.reserve(radix_temp_bytes(S, ntiles));
  B.sp.reserve(sizeof(double2) * 3 * S);
  B.range.reserve(sizeof(BhRange) * (2 * S + nc));
  B.child.reserve(sizeof(int2) * (2 * S + nc));
  B.m64.reserve(sizeof(Mom64) * std::max<int64_t>(m64_nodes, 1));
  B.geo.reserve(sizeof(BhGeo) * total);
  B.mom.reserve(sizeof(BhMom) * total);
}

// Every curve's segments in the order of their keys, and the end points staged
// in it.  Curves within kSmallSort are sorted by a block each, the others by the
// segmented sort.
template <typename SP, typename VP>
void enqueue_sort(flk_ctx *ctx, const ForestPlan &P, const VP *pts, SP *sp, hipStream_t s) {
  BhScratch &B = ctx->bh;
  const int64_t ntiles = (int64_t)P.tiles.size();
  const auto sort = [&](auto kernel, int k) {
    if (!P.small[k].empty())
      hipLaunchKernelGGL(kernel, dim3((unsigned)P.small[k].size()), dim3(kSmallThreads[k]), 0, s, pts, P.d_seg,
                         P.d_vtx, P.d_box, P.d_small[k], B.order.as<uint32_t>(), ntiles ? (SP *)nullptr : sp);
  };
  sort(bh_sort_small<SP, VP, kSmallThreads[0], kSmallSort[0]>, 0);
  sort(bh_sort_small<SP, VP, kSmallThreads[1], kSmallSort[1]>, 1);
  sort(bh_sort_small<SP, VP, kSmallThreads[2], kSmallSort[2]>, 2);
  FLK_HIP(hipGetLastError());
  if (ntiles == 0) return;
  hipLaunchKernelGGL(bh_keys<VP>, dim3((unsigned)ntiles), dim3(256), 0, s, pts, P.d_seg, P.d_vtx, P.d_box, P.d_tiles,
                     P.d_tcurve, B.keys0.as<uint32_t>(), B.ids0.as<uint32_t>());
  FLK_HIP(hipGetLastError());
  radix_sort_pairs<uint32_t>(B.keys0.as<uint32_t>(), B.keys1.as<uint32_t>(), B.ids0.as<uint32_t>(),
                             B.vals.as<uint32_t>(), B.order.as<uint32_t>(), P.S, 30, B.tmp.ptr, s, P.d_tiles, ntiles);
  hipLaunchKernelGGL((bh_stage_segments<SP, VP>), dim3((unsigned)((P.S + 255) / 256)), dim3(256), 0, s,
                     B.order.as<uint32_t>(), pts, P.S, sp);
  FLK_HIP(hipGetLastError());
}

// The nodes' ranges and children and the moments of a planned forest, with the
// segments' end points staged as SP.
template <typename SP>
void enqueue_moments(flk_ctx *ctx, const ForestPlan &P, SP *sp, hipStream_t s) {
  BhScratch &B = ctx->bh;
  const int32_t nc = (int32_t)P.cs.size();
  BhLevels L{};
  L.depth = (int32_t)P.level_base.size();
  int64_t units = nc;
  for (int lev = 0; lev < L.depth; ++lev) {
    L.base[lev] = P.level_base[lev];
    if (lev) units += P.level_n[lev] / 2;
  }
  L.base[L.depth] = P.total;
  hipLaunchKernelGGL(bh_level_offsets, dim3((unsigned)L.depth), dim3(256), 0, s, P.d_seg, nc, P.leaf,
                     B.loff.as<int32_t>());
  hipLaunchKernelGGL(bh_topology, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s, P.d_seg, nc,
                     P.leaf, L, B.loff.as<int32_t>(), B.range.as<BhRange>(), B.child.as<int2>());
  FLK_HIP(hipGetLastError());
  if (P.lev_top < (int)P.level_base.size()) {
    const int32_t b0 = P.level_base[P.lev_top], nd = P.total - b0;
    hipLaunchKernelGGL(bh_moments_direct<SP>, dim3((unsigned)((nd + 255) / 256)), dim3(256), 0, s,
                       B.range.as<BhRange>(), b0, nd, B.child.as<int2>(), (const SP *)sp, B.geo.as<BhGeo>(),
                       B.mom.as<BhMom>());
    FLK_HIP(hipGetLastError());
  }
  for (int lev = P.lev_top - 1; lev >= kTopLevels; --lev) {
    const int32_t n = P.level_n[lev];
    hipLaunchKernelGGL(bh_moments<SP>, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, s, B.range.as<BhRange>(),
                       n, P.level_base[lev], P.direct, B.child.as<int2>(), (const SP *)sp, B.m64.as<Mom64>(),
                       B.geo.as<BhGeo>(), B.mom.as<BhMom>());
  }
  if (P.lev_top > 0)
    hipLaunchKernelGGL(bh_moments_top<SP>, dim3((unsigned)nc), dim3(128), 0, s, B.range.as<BhRange>(), nc, L,
                       B.loff.as<int32_t>(), std::min(P.lev_top, kTopLevels) - 1, P.direct, B.child.as<int2>(),
                       (const SP *)sp, B.m64.as<Mom64>(), B.geo.as<BhGeo>(), B.mom.as<BhMom>());
  FLK_HIP(hipGetLastError());
}

void enqueue_forest(flk_ctx *ctx, const ForestPlan &P, hipStream_t s) {
  const int32_t nc = (int32_t)P.cs.size();
  if (nc == 0) return;
  Curves &cv = ctx->curves;
  BhScratch &B = ctx->bh;
  if (cv.inexact) {
    enqueue_sort(ctx, P, cv.dpts.as<double4>(), B.sp.as<double2>(), s);
    enqueue_moments(ctx, P, B.sp.as<double2>(), s);
  } else {  // every coordinate exact in FP32: the FP32 copies, the same values
    enqueue_sort(ctx, P, cv.hi.as<float4>(), B.sp.as<float2>(), s);
    enqueue_moments(ctx, P, B.sp.as<float2>(), s);
  }
}

void forest_from_plan(flk_ctx *ctx, const ForestPlan &P, Forest &F) {
  F.root.assign(ctx->curves.ncurves, -1);
  F.nnodes = P.total;
  F.depth = (int32_t)P.level_base.size();
  if (P.cs.empty()) F.depth = 0;
  for (size_t k = 0; k < P.cs.size(); ++k) F.root[P.cs[k]] = (int32_t)k;  // roots are nodes 0..nc-1
}

void build_forest(flk_ctx *ctx, const std::vector<int32_t> &curves_in, int leaf, Forest &F) {
  ForestPlan P;
  plan_forest(ctx, curves_in, leaf, P);
  PlanUpload up;
  add_forest(up, P);
  up.send(ctx, ctx->stream);
  enqueue_forest(ctx, P, ctx->stream);
  FLK_HIP(hipStreamSynchronize(ctx->stream));
  forest_from_plan(ctx, P, F);
}

// Items per thread of the level and leaf kernels: the tuned value, or by
// criterion (0): 8 for beta, 4 for the learned criterion, whose network
// staging in LDS would hold 8 items per thread to 2 blocks per CU (measured
// on 2 x 8M random walks: beta 21.4 ms at 8 against 21.8 at 4, learned 12.5
// at 4 against 15.1 at 8).
int items_per_thread(const flk_ctx *ctx, bool use_mlp) {
  const int t = ctx->tune.bh_items_per_thread;
  return (t == 2 || t == 4 || t == 8) ? t : (use_mlp ? 4 : 8);
}

// The level kernel for a criterion and a number of items per thread.
using LevelKernel = void (*)(const int4 *, int64_t, const unsigned long long *, int, const BhGeo *, const BhMom *,
                             const float *, float, const InferImage *, float, unsigned long long *,
                             int4 *, unsigned long long *, int64_t, BhItem *, unsigned long long *, int64_t,
                             double *, double *);
LevelKernel level_kernel(int ipt, bool use_mlp) {
  if (use_mlp) return ipt == 2 ? bh_level<2, true> : ipt == 8 ? bh_level<8, true> : bh_level<4, true>;
  return ipt == 2 ? bh_level<2, false> : ipt == 8 ? bh_level<8, false> : bh_level<4, false>;
}

// Traverses the given pairs (indices into the forest roots) with per-pair
// beta; adds into psum/perr (device, per pair).
//
// Items live in level buffers processed in chunks of up to kChunk items; a
// level that fits one chunk is consumed whole and its buffer swapped with the
// next level's (breadth-first, two buffers), a wider one pushes the next
// level on a LIFO stack so memory stays bounded by depth x chunk.  The host
// reads the queue counts (pinned memory) once per round of up to four levels;
// the device counters rotate through a pre-zeroed array instead of a clear
// per launch.
void traverse(flk_ctx *ctx, Forest &F, const std::vector<int32_t> &ra, const std::vector<int32_t> &rb,
              const std::vector<float> &beta2, float eps, double *d_sum, double *d_err,
              unsigned long long stats[4], bool use_mlp, float log_tol, bool timing) {
  hipStream_t s = ctx->stream;
  BhScratch &B = ctx->bh;
  const int64_t np = (int64_t)ra.size();
  if (np == 0) return;
  constexpr int64_t kChunk = 1 << 24;
  constexpr int kSlots = 1024;  // count pairs per zeroing of the counter array
  constexpr int kRound = 4;     // levels per host round trip (at most)
  // items per thread of the level/leaf kernels: 2, 4 or 8 (grid and kernel agree)
  const int ipt = items_per_thread(ctx, use_mlp);
  B.roots_a.reserve(sizeof(int32_t) * np);
  B.roots_b.reserve(sizeof(int32_t) * np);
  B.beta2.reserve(sizeof(float) * np);
  B.cnt.reserve(sizeof(unsigned long long) * (4 + 2 * kSlots));
  if (!B.host_cnt) FLK_HIP(hipHostMalloc((void **)&B.host_cnt, 2 * kRound * sizeof(unsigned long long)));
  FLK_HIP(hipMemcpyAsync(B.roots_a.ptr, ra.data(), sizeof(int32_t) * np, hipMemcpyHostToDevice, s));
  FLK_HIP(hipMemcpyAsync(B.roots_b.ptr, rb.data(), sizeof(int32_t) * np, hipMemcpyHostToDevice, s));
  FLK_HIP(hipMemcpyAsync(B.beta2.ptr, beta2.data(), sizeof(float) * np, hipMemcpyHostToDevice, s));
  // [2] leaf segment pairs, [3] network evaluations, [4 + 2k] queues
  unsigned long long *cnt = B.cnt.as<unsigned long long>();
  FLK_HIP(hipMemsetAsync(cnt, 0, sizeof(unsigned long long) * (4 + 2 * kSlots), s));

  struct Level {
    DevBuf *buf;
    int64_t n;
    bool roots;
  };
  std::vector<Level> stack;
  size_t used = 0;  // level buffers handed out from B.levels
  auto level_buf = [&](int64_t items) -> DevBuf * {
    if (B.levels.size() <= used) B.add_level();
    DevBuf *b = B.levels[used++].get();
    b->reserve(sizeof(BhItem) * std::max<int64_t>(items, 1));
    return b;
  };
  stack.push_back(Level{level_buf(np), np, true});
  hipLaunchKernelGGL(bh_roots, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, s,
                     B.roots_a.as<int32_t>(), B.roots_b.as<int32_t>(), np, stack[0].buf->as<BhItem>());
  FLK_HIP(hipGetLastError());
  DevBuf *spare = level_buf(2 * std::min(np, kChunk));
  if (use_mlp) mlp_upload(ctx);
  const InferImage *mlp_img = use_mlp ? ctx->mlp.d_image.as<InferImage>() : nullptr;
  unsigned long long visits = 0, far = 0;
  int slot_next = 0;
  DevBuf *alt = nullptr;  // second output buffer of a multi-level round
  while (!stack.empty()) {
    Level &top = stack.back();
    if (top.n == 0) {
      spare = top.buf;  // an emptied level's buffer is reused
      stack.pop_back();
      continue;
    }
    const int64_t take = std::min<int64_t>(top.n, kChunk);
    top.n -= take;
    const int4 *src = top.buf->as<int4>() + (top.roots ? top.n : top.n / 2);  // two items a record past the roots
    const bool roots = top.roots;
    // Levels enqueued before the next read-back: the first from its exact
    // count and, when it is consumed whole, up to kRound - 1 more, level d
    // sized for its bound take * 2^d (a level at most doubles) and reading
    // its true count from the previous level's counter on the device.  The
    // last level's bound keeps its output within 2 * kChunk items.  With
    // per-launch timing every level is its own round.
    int D = 1;
    if (!timing && top.n == 0)
      while (D < kRound && (take << (D + 1)) <= 2 * kChunk) ++D;
    const int64_t out_cap = take << D;  // items: bound of the last level's output
    spare->reserve(sizeof(BhItem) * out_cap);
    if (D > 1) {
      if (!alt) alt = level_buf(out_cap);
      alt->reserve(sizeof(BhItem) * out_cap);
    }
    const int64_t leaf_cap = (int64_t)((1LL << D) - 1) * take;  // sum of the level bounds
    if (B.leaves.bytes < sizeof(BhItem) * leaf_cap) {
      FLK_HIP(hipStreamSynchronize(s));  // the previous leaf launch may still read it
      B.leaves.reserve(sizeof(BhItem) * leaf_cap);
    }
    if (slot_next + D > kSlots) {
      FLK_HIP(hipMemsetAsync(cnt + 4, 0, sizeof(unsigned long long) * 2 * kSlots, s));
      slot_next = 0;
    }
    unsigned long long *qc = cnt + 4 + 2 * slot_next;  // per level [0] next items; [1] of level 0: leaves
    slot_next += D;
    DevBuf *outb[kRound];
    for (int d = 0; d < D; ++d) {
      outb[d] = (d % 2 == 0) ? spare : alt;
      const int4 *in = d == 0 ? src : outb[d - 1]->as<int4>();
      const int64_t bound = take << d;
      const unsigned long long *n_dev = d == 0 ? nullptr : qc + 2 * (d - 1);
      // with timing, start/stop events ride on the dispatch itself
      const dim3 grid((unsigned)((bound + ipt * kTravBlock - 1) / (ipt * kTravBlock)));
      launch_timed(timing ? ctx->ev1 : nullptr, timing ? ctx->ev2 : nullptr, level_kernel(ipt, use_mlp), grid,
                   dim3(kTravBlock), s, in, bound, n_dev, (int)(roots && d == 0), F.geo.as<BhGeo>(), F.mom.as<BhMom>(),
                   (const float *)B.beta2.as<float>(), eps, mlp_img, log_tol, cnt + 3,
                   outb[d]->as<int4>(), qc + 2 * d, 2 * bound, B.leaves.as<BhItem>(), qc + 1, leaf_cap, d_sum,
                   d_err);
      FLK_HIP(hipGetLastError());
    }
    FLK_HIP(hipMemcpyAsync(B.host_cnt, qc, 2 * D * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    FLK_HIP(hipStreamSynchronize(s));
    if (timing) {
      float ms_level = 0.f;
      FLK_HIP(hipEventElapsedTime(&ms_level, ctx->ev1, ctx->ev2));
      if (use_mlp) ctx->stats.ms_mlp += ms_level;  // the network runs inside the level kernels
      ctx->stats.ms_bh_level += ms_level;
    }
    // every item is exactly one of: leaf pair, far field, split (two children)
    int64_t in_n = take;
    for (int d = 0; d < D; ++d) {
      const unsigned long long nn = B.host_cnt[2 * d];
      if ((int64_t)nn > 2 * (take << d)) throw Error(FLK_ERR_STATE, "Barnes-Hut level buffer overflow");
      visits += (unsigned long long)in_n;
      far += (unsigned long long)in_n - nn / 2;
      in_n = (int64_t)nn;
    }
    const unsigned long long nleaf = B.host_cnt[1];
    if ((int64_t)nleaf > leaf_cap) throw Error(FLK_ERR_STATE, "Barnes-Hut leaf buffer overflow");
    far -= nleaf;
    if (nleaf > 0) {
      const Curves &cv = ctx->curves;
      auto leafk = ipt == 2 ? bh_leaf_pairs<2> : ipt == 8 ? bh_leaf_pairs<8> : bh_leaf_pairs<4>;
      hipLaunchKernelGGL(leafk, dim3((unsigned)((nleaf + ipt * kTravBlock - 1) / (ipt * kTravBlock))),
                         dim3(kTravBlock), 0, s, B.leaves.as<BhItem>(), (int64_t)nleaf, (unsigned long long *)nullptr, 0,
                         F.geo.as<BhGeo>(), F.order.as<uint32_t>(), cv.hi.as<float4>(), cv.lo.as<float4>(),
                         cv.ed.as<float4>(), d_sum, d_err, cnt + 2, 1, (int64_t)0);
      FLK_HIP(hipGetLastError());
    }
    DevBuf *last = outb[D - 1];
    if (top.n == 0) {
      // the level is consumed: the last level's output replaces it, the
      // consumed buffer and the round's other output buffer are free
      DevBuf *consumed = top.buf;
      top.buf = last;
      top.n = in_n;
      top.roots = false;
      if (D > 1) alt = (last == spare) ? alt : spare;
      spare = consumed;
    } else if (in_n > 0) {
      stack.push_back(Level{last, in_n, false});  // D == 1: last is spare
      spare = level_buf(2 * kChunk);
    }
  }
  unsigned long long st[4];
  FLK_HIP(hipMemcpyAsync(st, cnt, sizeof st, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  stats[0] += visits;
  stats[1] += far;
  stats[2] += st[2];
  stats[3] += st[3];  // learned-criterion network evaluations
}

// Blocks of `kernel` resident on the whole chip at once (the persistent grid
// of a device-scheduled pass).
int resident_grid(flk_ctx *ctx, const void *kernel) {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, kTravBlock, 0) != hipSuccess || nb < 1) nb = 1;
  return nb * std::max(1, ctx->num_cus);
}

// Device schedule of a batch's traversal passes.  A pass enqueues every
// level at once: level d reads its item count from the counter that level
// d - 1 incremented, on a persistent grid whose blocks stride over the
// level's chunks, so no count returns to the host until the batch has ended.
// Every split deepens one of the two trees, so a pass has fewer than
// 2 * depth + 1 levels; launched levels past the last nonempty one see a
// count of 0 and exit at once.  Both level buffers and the leaf list hold
// `cap` items.  A level or leaf list beyond that, or items left after the
// last launched level, mark the pass as overflowed: its sums are incomplete,
// and the batch is re-run on the host-driven schedule.
// Or, with few segments a pair, by some launches of bh_walk, each taking
// what the one before left in the queue.  The line lies where the walk's gain
// in launches is spent: a pair of random walks of 5,000 vertices each takes
// 0.58 ms walked and 0.68 by levels, 30,000 1.14 and 1.13, 100,000 1.66 and
// 1.48 (the levels' blocks classify eight items a thread between barriers, a
// walk's waves one a step).  The learned criterion's network leaves too little
// LDS for a walk's stacks.
constexpr int64_t kWalkSegmentsPerPair = 32768;
// The last round ends with its longest subtree, so a large pair among small ones
// takes more rounds to share out, two for each doubling.  Beside 380 pairs of
// rings, a pair of tangled walks of 60,000 takes 3.8 ms in 6 rounds, 2.0 in 12 and
// 2.1 in 24, one of 300,000 25, 5.9 and 4.2, of 1,000,000 187, 26 and 10.7, of
// 4,000,000 beside one of 100,000 1,003, 136 and 19.6; by levels 2.0, 3.7, 9.0
// and 90 (where pairs mix there, every far field is an atomic).  48 rounds gain
// nothing over 24; a round that finds nothing takes 4 us.
constexpr int kWalkRounds = 6;
inline int walk_rounds(int64_t largest_pair) {
  int rounds = kWalkRounds;
  for (int64_t n = kWalkSegmentsPerPair; n < largest_pair; n *= 2) rounds += 2;
  return rounds;
}

struct PassShape {
  int64_t cap = 0;
  bool walk = false;
  int D = 0, rounds = 0, ipt = 4;
  int copies = 1;  // of the per-pair sums: a walk's blocks of different XCDs add to different ones
  unsigned grid_lev = 1, grid_leaf = 1;
};

// Counter words of the host-driven schedule (traverse); a batch's re-run
// count lives in the 8 words after them.
constexpr int kHostCounterWords = 4 + 2 * 1024;

// Sizes the device schedule of a batch of nb pairs on trees of `segments`
// segments, the deepest with `depth` node levels, and reserves its buffers;
// false when it cannot hold the batch (the host-driven schedule runs it
// instead).  largest_pair: the most segments of any pair, each curve counted
// with those of the shorter (a short curve meets little of a long one).
bool plan_device_passes(flk_ctx *ctx, int64_t nb, int64_t segments, int64_t largest_pair, int depth, bool use_mlp,
                        PassShape &P) {
  BhScratch &B = ctx->bh;
  P.walk = !use_mlp && segments <= nb * kWalkSegmentsPerPair;
  P.D = P.walk ? 0 : 2 * depth + 1;
  P.rounds = P.walk ? walk_rounds(largest_pair) : 0;
  if (P.D > kMaxLevels) return false;
  if (B.dev_cap == 0) {
    // two level buffers and the leaf list (16 B per item), within a tenth of
    // the free memory, at most 2^26 items each
    size_t free_b = 0, total_b = 0;
    FLK_HIP(hipMemGetInfo(&free_b, &total_b));
    int64_t cap = int64_t(1) << 26;
    while (cap > (int64_t(1) << 20) && (double)cap * 52.0 > 0.1 * (double)free_b) cap >>= 1;
    B.dev_cap = cap;
  }
  P.cap = ctx->tune.bh_level_capacity > 0 ? (int64_t)ctx->tune.bh_level_capacity : B.dev_cap;
  if (nb > P.cap) return false;
  P.ipt = items_per_thread(ctx, use_mlp);
  P.copies = P.walk && nb <= 4096 ? 8 : 1;
  while (B.levels.size() < 2) B.add_level();
  // a walk's items, or a level's records of two items each
  const size_t level_bytes = P.walk ? sizeof(BhItem) * P.cap : sizeof(int4) * (P.cap / 2 + 1);
  B.levels[0]->reserve(level_bytes);
  B.levels[1]->reserve(level_bytes);
  B.leaves.reserve(sizeof(BhItem) * P.cap);
  auto leafk = P.ipt == 2 ? bh_leaf_pairs<2> : P.ipt == 8 ? bh_leaf_pairs<8> : bh_leaf_pairs<4>;
  const int64_t items_per_block = (int64_t)P.ipt * kTravBlock;
  const int64_t chunks = (P.cap + items_per_block - 1) / items_per_block;
  const int lev = resident_grid(ctx, P.walk ? (const void *)bh_walk : (const void *)level_kernel(P.ipt, use_mlp));
  const int leaf = resident_grid(ctx, (const void *)leafk);
  if (P.walk) {
    // whole multiples of the segments' number: a segment's waves are on one
    // XCD, and the segments have as many each
    P.grid_lev = (unsigned)std::max(kSegs, lev / kSegs * kSegs);
    P.grid_leaf = (unsigned)std::max(kSegs, leaf / kSegs * kSegs);
  } else {
    P.grid_lev = (unsigned)std::min<int64_t>(lev, chunks);
    P.grid_leaf = (unsigned)std::min<int64_t>(leaf, chunks);
  }
  return true;
}

// Enqueues one pass on the device schedule: counters at cnt (bh_begin has
// cleared them, and the root count is at cnt[4]), root items at items0,
// per-pair beta^2 and sums indexed by the items' pair field.
void enqueue_pass(flk_ctx *ctx, const PassShape &P, const BhItem *items0, const float *beta2, float eps,
                  bool use_mlp, float log_tol, unsigned long long *cnt, double *d_sum, double *d_err,
                  int64_t copy_stride, hipStream_t s) {
  BhScratch &B = ctx->bh;
  const Curves &cv = ctx->curves;
  BhItem *buf[2] = {B.levels[0]->as<BhItem>(), B.levels[1]->as<BhItem>()};
  const InferImage *mlp_img = use_mlp ? ctx->mlp.d_image.as<InferImage>() : nullptr;
  const LevelKernel lev = level_kernel(P.ipt, use_mlp);
  auto leafk = P.ipt == 2 ? bh_leaf_pairs<2> : P.ipt == 8 ? bh_leaf_pairs<8> : bh_leaf_pairs<4>;
  for (int d = 0; d < (P.walk ? P.rounds : P.D); ++d) {
    const BhItem *in = d == 0 ? items0 : buf[(d - 1) & 1];
    if (P.walk)
      hipLaunchKernelGGL(bh_walk, dim3(P.grid_lev), dim3(kTravBlock), 0, s, in, P.cap, B.geo.as<BhGeo>(),
                         B.mom.as<BhMom>(), beta2, eps, cnt, d, (int)(d + 1 == P.rounds), buf[d & 1], B.leaves.as<BhItem>(), d_sum,
                         d_err, P.copies, copy_stride);
    else
      hipLaunchKernelGGL(lev, dim3(P.grid_lev), dim3(kTravBlock), 0, s, reinterpret_cast<const int4 *>(in), P.cap,
                         (const unsigned long long *)(cnt + 4 + 2 * d), (int)(d == 0), B.geo.as<BhGeo>(), B.mom.as<BhMom>(), beta2,
                         eps, mlp_img, log_tol, cnt + 3, reinterpret_cast<int4 *>(buf[d & 1]), cnt + 4 + 2 * (d + 1), P.cap,
                         B.leaves.as<BhItem>(), cnt + 5, P.cap, d_sum, d_err);
    FLK_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(leafk, dim3(P.grid_leaf), dim3(kTravBlock), 0, s, B.leaves.as<BhItem>(), P.cap, cnt,
                     (int)P.walk, B.geo.as<BhGeo>(), B.order.as<uint32_t>(), cv.hi.as<float4>(), cv.lo.as<float4>(),
                     cv.ed.as<float4>(), d_sum, d_err, cnt, P.copies, copy_stride);
  FLK_HIP(hipGetLastError());
}

// Adds a device-scheduled pass's visits, far fields, leaf segment pairs and
// network evaluations (from its head h) to st; false when it overflowed.
// Every item is exactly one of: leaf pair, far field, split (two children).
bool pass_counts(const unsigned long long *h, unsigned long long st[4]) {
  if (h[6] != 0) return false;
  st[0] += h[0];
  st[1] += h[0] - h[1] - h[5];
  st[2] += h[2];
  st[3] += h[3];
  return true;
}

}  // namespace

int64_t mlp_samples(flk_ctx *ctx, int32_t a, int32_t b, int64_t cap, uint64_t seed, float *x,
                    float *y) {
  Curves &cv = ctx->curves;
  hipStream_t s = ctx->stream;
  if (cap <= 0) return 0;
  if (cv.n[a] < 2 || cv.n[b] < 2) return 0;
  Forest F(ctx->bh);
  std::vector<int32_t> cs{std::min(a, b), std::max(a, b)};
  if (a == b) cs.resize(1);
  build_forest(ctx, cs, 1, F);
  const float eps = (float)(1e-24 * cv.scale * cv.scale);
  const float stop2 = 36.0f;                // samples up to |r| = 6 (r1 + r2)
  const int64_t max_pairs = 1 << 20;        // exact-label cost cap per sample
  const int64_t chunk = 1 << 22;
  DevBuf d_cnt, d_samp, d_a, d_b;
  d_cnt.reserve(sizeof(unsigned long long) * 4);
  d_a.reserve(sizeof(BhItem) * 2 * chunk);
  d_b.reserve(sizeof(BhItem) * 2 * chunk);
  d_samp.reserve(sizeof(BhItem) * cap);
  unsigned long long *cnt = d_cnt.as<unsigned long long>();
  auto run = [&](double p, int64_t samp_cap) -> int64_t {
    // breadth-first over levels; a level wider than the chunk is thinned by
    // keeping a random subset (the samples stay spread over all depths)
    FLK_HIP(hipMemsetAsync(cnt, 0, sizeof(unsigned long long) * 4, s));
    BhItem root{0, F.root[a], F.root[b], 0};
    FLK_HIP(hipMemcpyAsync(d_a.ptr, &root, sizeof root, hipMemcpyHostToDevice, s));
    int64_t n = 1;
    DevBuf *cur = &d_a, *nxt = &d_b;
    while (n > 0) {
      const int64_t take = std::min(n, chunk);
      FLK_HIP(hipMemsetAsync(cnt, 0, sizeof(unsigned long long), s));
      hipLaunchKernelGGL(bh_sample_level, dim3((unsigned)((take + 255) / 256)), dim3(256), 0, s,
                         cur->as<BhItem>(), take, F.geo.as<BhGeo>(), eps, stop2, p, seed, max_pairs,
                         nxt->as<BhItem>(), cnt, d_samp.as<BhItem>(), cnt + 1, samp_cap);
      FLK_HIP(hipGetLastError());
      unsigned long long nn = 0;
      FLK_HIP(hipMemcpyAsync(&nn, cnt, sizeof nn, hipMemcpyDeviceToHost, s));
      FLK_HIP(hipStreamSynchronize(s));
      n = (int64_t)nn;
      std::swap(cur, nxt);
    }
    unsigned long long ns = 0;
    FLK_HIP(hipMemcpyAsync(&ns, cnt + 1, sizeof ns, hipMemcpyDeviceToHost, s));
    FLK_HIP(hipStreamSynchronize(s));
    return (int64_t)ns;
  };
  const int64_t eligible = run(1.0, 0);
  if (eligible == 0) return 0;
  const double p = std::min(1.0, 1.05 * (double)cap / (double)eligible);
  const int64_t got = std::min(run(p, cap), cap);
  DevBuf dx, dy;
  dx.reserve(sizeof(float) * FLK_MLP_NFEAT * got);
  dy.reserve(sizeof(float) * got);
  hipLaunchKernelGGL(bh_sample_labels, dim3((unsigned)((got * 64 + 255) / 256)), dim3(256), 0, s,
                     d_samp.as<BhItem>(), got, F.geo.as<BhGeo>(), F.mom.as<BhMom>(),
                     F.order.as<uint32_t>(), cv.dpts.as<double4>(), eps, dx.as<float>(), dy.as<float>());
  FLK_HIP(hipGetLastError());
  FLK_HIP(hipMemcpyAsync(x, dx.ptr, sizeof(float) * FLK_MLP_NFEAT * got, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipMemcpyAsync(y, dy.ptr, sizeof(float) * got, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  return got;
}

void tree_export(flk_ctx *ctx, int32_t curve, int32_t leaf, std::vector<flk_tree_node> &nodes,
                 std::vector<int32_t> &seg_order) {
  Curves &cv = ctx->curves;
  hipStream_t s = ctx->stream;
  nodes.clear();
  seg_order.clear();
  if (cv.n[curve] < 2) return;
  Forest F(ctx->bh);
  build_forest(ctx, std::vector<int32_t>{curve}, leaf, F);
  const int32_t nn = F.nnodes, nseg = cv.n[curve];
  std::vector<BhGeo> g(nn);
  std::vector<BhMom> m(nn);
  std::vector<uint32_t> ord(nseg);
  FLK_HIP(hipMemcpyAsync(g.data(), F.geo.ptr, sizeof(BhGeo) * nn, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipMemcpyAsync(m.data(), F.mom.ptr, sizeof(BhMom) * nn, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipMemcpyAsync(ord.data(), F.order.ptr, sizeof(uint32_t) * nseg, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  // stored = (input - origin) * scale with a power-of-two scale: the
  // conversions back are exact apart from the origin's addition
  const double is = 1.0 / cv.scale, is2 = is * is, is3 = is2 * is;
  nodes.resize(nn);
  for (int32_t k = 0; k < nn; ++k) {
    const BhGeo &a = g[k];
    const BhMom b = is_leaf_segment(a) ? leaf_segment_mom(a) : m[k];
    flk_tree_node &o = nodes[k];
    std::memset(&o, 0, sizeof o);
    const double ctr[3] = {(double)a.cx + (double)a.lx, (double)a.cy + (double)a.ly, (double)a.cz + (double)a.lz};
    for (int d = 0; d < 3; ++d) o.center[d] = cv.origin[d] + ctr[d] * is;
    o.radius = (double)a.radius * is;
    o.rsq = (double)a.rsq * is2;
    for (int d = 0; d < 3; ++d) o.c[d] = (double)b.c[d] * is;
    for (int t = 0; t < 9; ++t) o.D[t] = (double)b.D[t] * is2;
    for (int kk = 0; kk < 3; ++kk)
      for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) o.Q[9 * kk + 3 * i + j] = (double)b.Q[6 * kk + qidx(i, j)] * is3;
    o.cn = (double)a.cn * is;
    o.dn = (double)geo_dn(a) * is2;
    o.qn = (double)a.qn * is3;
    o.child[0] = a.c0 < 0 ? -1 : a.c0;
    o.child[1] = a.c0 < 0 ? -1 : a.c1;
    o.seg0 = a.seg0;
    o.nseg = a.nseg;
  }
  seg_order.resize(nseg);
  for (int32_t t = 0; t < nseg; ++t) seg_order[t] = (int32_t)((int64_t)ord[t] - cv.off[curve]);
}

namespace {

// One batch of Barnes–Hut pairs (indices into the call's pair list): its
// forest plan, root nodes, first-pass beta^2, the device schedule's shape,
// and the results and counters the batch's read-back fills.
struct BatchPlan {
  std::vector<int64_t> idx;
  ForestPlan forest;
  std::vector<int32_t> ra, rb;
  std::vector<float> beta2;
  PassShape shape;
  bool device = false;  // the device schedule holds it
  std::vector<double> v, e;
  std::vector<uint32_t> f;
  std::vector<unsigned long long> counts;  // both passes' heads
  // What bh_merge writes, pinned: v, e, counts, f.
  HostBuf res;
  size_t res_bytes() const { return 20 * idx.size() + 8 * counts.size(); }
  // the arrays' device addresses (PlanUpload)
  const int32_t *d_ra = nullptr, *d_rb = nullptr;
  const float *d_beta2 = nullptr;
  void add(PlanUpload &up) {
    add_forest(up, forest);
    up.add(ra, d_ra);
    up.add(rb, d_rb);
    up.add(beta2, d_beta2);
  }
  const unsigned long long *heads() const {
    return reinterpret_cast<const unsigned long long *>(res.as<double>() + 2 * idx.size());
  }
  void collect() {  // res into the vectors
    const double *hv = res.as<double>();
    std::copy(hv, hv + v.size(), v.begin());
    hv += v.size();
    std::copy(hv, hv + e.size(), e.begin());
    const auto *hc = reinterpret_cast<const unsigned long long *>(hv + e.size());
    std::copy(hc, hc + counts.size(), counts.begin());
    const auto *hf = reinterpret_cast<const uint32_t *>(hc + counts.size());
    std::copy(hf, hf + f.size(), f.begin());
  }
};

void plan_batch(flk_ctx *ctx, const int32_t *pairs, std::vector<int64_t> idx, const flk_params &prm,
                BatchPlan &bp) {
  Curves &cv = ctx->curves;
  const bool use_mlp = prm.criterion == FLK_CRIT_MLP;
  bp.idx = std::move(idx);
  std::vector<char> used(cv.ncurves, 0);
  for (int64_t k : bp.idx) used[pairs[2 * k]] = used[pairs[2 * k + 1]] = 1;
  std::vector<int32_t> cs;
  for (int32_t c = 0; c < cv.ncurves; ++c)
    if (used[c]) cs.push_back(c);
  plan_forest(ctx, cs, std::max(1, prm.leaf_size), bp.forest);
  std::vector<int32_t> root(cv.ncurves, -1);
  for (size_t k = 0; k < bp.forest.cs.size(); ++k) root[bp.forest.cs[k]] = (int32_t)k;
  const int64_t nb = (int64_t)bp.idx.size();
  bp.ra.resize(nb);
  bp.rb.resize(nb);
  bp.beta2.assign(nb, (float)(prm.beta_init * prm.beta_init));
  int64_t largest = 0;
  for (int64_t t = 0; t < nb; ++t) {
    const int32_t a = pairs[2 * bp.idx[t]], b = pairs[2 * bp.idx[t] + 1];
    bp.ra[t] = root[a];
    bp.rb[t] = root[b];
    largest = std::max<int64_t>(largest, 2 * (int64_t)std::min(cv.n[a], cv.n[b]));
  }
  bp.device = plan_device_passes(ctx, nb, bp.forest.S, largest, (int)bp.forest.level_base.size(), use_mlp, bp.shape);
  BhScratch &B = ctx->bh;
  B.beta2.reserve(sizeof(float) * 2 * nb);
  B.items0.reserve(sizeof(BhItem) * nb);
  B.redo.reserve(sizeof(int32_t) * nb);
  B.sum.reserve(sizeof(double) * 2 * nb * bp.shape.copies);
  B.err.reserve(sizeof(double) * 2 * nb * bp.shape.copies);
  B.cnt.reserve(sizeof(unsigned long long) * std::max(2 * pass_words(bp.shape.rounds), kHostCounterWords + 8));
  if (use_mlp) mlp_upload(ctx);
  bp.v.assign(nb, 0.0);
  bp.e.assign(nb, 0.0);
  bp.f.assign(nb, 0u);
  bp.counts.assign(2 * kPassHead, 0ull);
  bp.res.reserve(bp.res_bytes());
}

// The batch's merge of both passes into per-pair results, in pinned memory.
// cnt: the device-scheduled passes' counters, null for a host-driven batch.
void enqueue_merge(flk_ctx *ctx, BatchPlan &bp, const flk_params &prm, unsigned long long *cnt, hipStream_t s) {
  BhScratch &B = ctx->bh;
  const int64_t nb = (int64_t)bp.idx.size();
  double *v = bp.res.as<double>(), *e = v + nb;
  auto *heads = reinterpret_cast<unsigned long long *>(e + nb);
  auto *f = reinterpret_cast<uint32_t *>(heads + bp.counts.size());
  hipLaunchKernelGGL(bh_merge, dim3((unsigned)((nb + 255) / 256) + (cnt ? 1 : 0)), dim3(256), 0, s, nb,
                     (const int32_t *)B.redo.as<int32_t>(), (const double *)B.sum.as<double>(),
                     (const double *)B.err.as<double>(), bp.shape.copies, 2 * nb,
                     prm.criterion == FLK_CRIT_MLP ? 1 : 0, prm.err_scale, v, e, f, heads, cnt, bp.shape.cap,
                     bp.shape.D, bp.shape.rounds);
  FLK_HIP(hipGetLastError());
}

void enqueue_adapt(flk_ctx *ctx, const BatchPlan &bp, const flk_params &prm, unsigned long long *n_redo,
                   hipStream_t s) {
  BhScratch &B = ctx->bh;
  const int64_t nb = (int64_t)bp.idx.size();
  hipLaunchKernelGGL(bh_adapt, dim3(1), dim3(1024), 0, s, nb, bp.d_ra, bp.d_rb,
                     (const double *)B.err.as<double>(), bp.shape.copies,
                     2 * nb, prm.criterion == FLK_CRIT_MLP ? 1 : 0, prm.err_scale, prm.target_error, prm.beta_init,
                     prm.beta_limit, B.items0.as<BhItem>(), B.beta2.as<float>() + nb, B.redo.as<int32_t>(), n_redo);
  FLK_HIP(hipGetLastError());
}

// Clears the sums and both passes' counters and lists the root items.
void enqueue_begin(flk_ctx *ctx, const BatchPlan &bp, hipStream_t s) {
  BhScratch &B = ctx->bh;
  const int64_t nb = (int64_t)bp.idx.size(), nsums = 2 * nb * bp.shape.copies;
  const int words = pass_words(bp.shape.rounds);
  hipLaunchKernelGGL(bh_begin, dim3((unsigned)((std::max<int64_t>(nsums, 2 * words) + 255) / 256)), dim3(256), 0, s,
                     bp.d_ra, bp.d_rb, nb, B.items0.as<BhItem>(), B.cnt.as<unsigned long long>(), words, nsums,
                     B.sum.as<double>(), B.err.as<double>());
  FLK_HIP(hipGetLastError());
}

// Traversal of a planned batch on the device schedule, after its forest:
// first pass, the re-run decision (bh_adapt), second pass over the re-run
// list and the merge of results and counters.  Kernels only, so it can be
// captured.  `first` and `second` pick the passes to enqueue (a merge follows
// either).
void enqueue_traversal(flk_ctx *ctx, BatchPlan &bp, const flk_params &prm, hipStream_t s, bool first = true,
                       bool second = true) {
  BhScratch &B = ctx->bh;
  const Curves &cv = ctx->curves;
  const bool use_mlp = prm.criterion == FLK_CRIT_MLP;
  const int64_t nb = (int64_t)bp.idx.size();
  const PassShape &P = bp.shape;
  const float eps = (float)(prm.eps_sq * cv.scale * cv.scale);
  const float log_tol = (float)prm.mlp_log_tol;
  double *sum = B.sum.as<double>(), *err = B.err.as<double>();
  unsigned long long *c1 = B.cnt.as<unsigned long long>(), *c2 = c1 + pass_words(P.rounds);
  if (first) {
    enqueue_begin(ctx, bp, s);
    enqueue_pass(ctx, P, B.items0.as<BhItem>(), bp.d_beta2, eps, use_mlp, log_tol, c1, sum, err, 2 * nb, s);
    enqueue_adapt(ctx, bp, prm, c2 + 4, s);
  }
  if (second)
    enqueue_pass(ctx, P, B.items0.as<BhItem>(), B.beta2.as<float>() + nb, eps, use_mlp, log_tol - 1.0f, c2, sum + nb,
                 err + nb, 2 * nb, s);
  enqueue_merge(ctx, bp, prm, c1, s);
}

// Results and statistics of a batch whose read-back has arrived; false when
// a pass overflowed the device schedule (nothing is written then).
bool finish_batch(flk_ctx *ctx, const BatchPlan &bp, std::vector<double> &lk, std::vector<double> &err,
                  std::vector<uint32_t> &flags) {
  unsigned long long st[4] = {0, 0, 0, 0};
  const unsigned long long *h = bp.counts.data();
  if (!pass_counts(h, st) || !pass_counts(h + kPassHead, st)) return false;
  for (size_t t = 0; t < bp.idx.size(); ++t) {
    lk[bp.idx[t]] = bp.v[t];
    err[bp.idx[t]] = bp.e[t];
    flags[bp.idx[t]] |= bp.f[t];
  }
  ctx->stats.retries += (int64_t)h[kPassHead + 4];
  ctx->stats.bh_visits += (int64_t)st[0];
  ctx->stats.bh_far += (int64_t)st[1];
  ctx->stats.bh_leaf_pairs += (int64_t)st[2];
  ctx->stats.mlp_evals += (int64_t)st[3];
  return true;
}

// A batch on the host-driven schedule: per-launch timing, or a batch the
// device schedule cannot hold or that overflowed it.  The same re-run
// decision (bh_adapt) and merge; the re-run list comes back to the host.
void bh_batch_host(flk_ctx *ctx, const int32_t *pairs, const std::vector<int64_t> &idx, const flk_params &prm,
                   std::vector<double> &lk, std::vector<double> &err, std::vector<uint32_t> &flags) {
  hipStream_t s = ctx->stream;
  const bool use_mlp = prm.criterion == FLK_CRIT_MLP;
  BatchPlan bp;
  auto t0 = std::chrono::steady_clock::now();
  plan_batch(ctx, pairs, idx, prm, bp);
  PlanUpload up;
  bp.add(up);
  up.send(ctx, s);
  enqueue_forest(ctx, bp.forest, s);
  FLK_HIP(hipStreamSynchronize(s));
  ctx->stats.ms_bh_build +=
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  t0 = std::chrono::steady_clock::now();
  Forest F(ctx->bh);
  forest_from_plan(ctx, bp.forest, F);
  BhScratch &B = ctx->bh;
  const int64_t nb = (int64_t)bp.idx.size();
  const float eps = (float)(prm.eps_sq * ctx->curves.scale * ctx->curves.scale);
  double *sum = B.sum.as<double>(), *err_d = B.err.as<double>();
  enqueue_begin(ctx, bp, s);
  unsigned long long st[4] = {0, 0, 0, 0};
  traverse(ctx, F, bp.ra, bp.rb, bp.beta2, eps, sum, err_d, st, use_mlp, (float)prm.mlp_log_tol, prm.timing != 0);
  unsigned long long *c2 = B.cnt.as<unsigned long long>() + kHostCounterWords;
  enqueue_adapt(ctx, bp, prm, c2 + 4, s);
  unsigned long long nr = 0;
  FLK_HIP(hipMemcpyAsync(&nr, c2 + 4, sizeof nr, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  int passes = 1;
  if (nr > 0) {
    std::vector<BhItem> it(nr);
    std::vector<float> b2(nr);
    FLK_HIP(hipMemcpyAsync(it.data(), B.items0.ptr, sizeof(BhItem) * nr, hipMemcpyDeviceToHost, s));
    FLK_HIP(hipMemcpyAsync(b2.data(), B.beta2.as<float>() + nb, sizeof(float) * nr, hipMemcpyDeviceToHost, s));
    FLK_HIP(hipStreamSynchronize(s));
    std::vector<int32_t> ra2(nr), rb2(nr);
    for (size_t k = 0; k < nr; ++k) {
      ra2[k] = it[k].a;
      rb2[k] = it[k].b;
    }
    traverse(ctx, F, ra2, rb2, b2, eps, sum + nb, err_d + nb, st, use_mlp, (float)prm.mlp_log_tol - 1.0f,
             prm.timing != 0);
    passes = 2;
  }
  enqueue_merge(ctx, bp, prm, nullptr, s);
  FLK_HIP(hipStreamSynchronize(s));
  bp.collect();
  for (size_t t = 0; t < bp.idx.size(); ++t) {
    lk[bp.idx[t]] = bp.v[t];
    err[bp.idx[t]] = bp.e[t];
    flags[bp.idx[t]] |= bp.f[t];
  }
  ctx->stats.retries += (int64_t)nr;
  ctx->stats.bh_host_passes += passes;
  ctx->stats.bh_visits += (int64_t)st[0];
  ctx->stats.bh_far += (int64_t)st[1];
  ctx->stats.bh_leaf_pairs += (int64_t)st[2];
  ctx->stats.mlp_evals += (int64_t)st[3];
  ctx->stats.ms_bh_traverse +=
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

// Trees, traversal and the adaptive-beta / learned-criterion re-run for one
// batch of Barnes–Hut pairs, launched eagerly; results into lk/err/flags.
void bh_batch(flk_ctx *ctx, const int32_t *pairs, const std::vector<int64_t> &idx, const flk_params &prm,
              std::vector<double> &lk, std::vector<double> &err, std::vector<uint32_t> &flags) {
  if (prm.timing) {
    bh_batch_host(ctx, pairs, idx, prm, lk, err, flags);
    return;
  }
  hipStream_t s = ctx->stream;
  BatchPlan bp;
  auto t0 = std::chrono::steady_clock::now();
  plan_batch(ctx, pairs, idx, prm, bp);
  if (!bp.device) {
    bh_batch_host(ctx, pairs, idx, prm, lk, err, flags);
    return;
  }
  PlanUpload up;
  bp.add(up);
  up.send(ctx, s);
  enqueue_forest(ctx, bp.forest, s);
  FLK_HIP(hipStreamSynchronize(s));
  ctx->stats.ms_bh_build +=
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  t0 = std::chrono::steady_clock::now();
  enqueue_traversal(ctx, bp, prm, s);
  FLK_HIP(hipStreamSynchronize(s));
  bp.collect();
  ctx->stats.ms_bh_traverse +=
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  if (!finish_batch(ctx, bp, lk, err, flags)) bh_batch_host(ctx, pairs, idx, prm, lk, err, flags);
}

// Device bytes the trees and their build records take per segment: two
// 192-byte node records (384), 288-byte FP64 records for the nodes above 8
// segments (about one node in eight: ~72), ranges and children (32), sort keys,
// values, ids and order (20), the staged segment endpoints (48) and sort scratch,
// with headroom.
constexpr double kBhBytesPerSegment = 648.0;

// Batches of Barnes–Hut pairs whose curves' trees fit the device: the
// segment budget is bh_batch_ksegs thousand, or what free memory (plus the
// scratch this context already holds) allows when a curve set first runs
// Barnes–Hut -- kept for later calls on the same curves, so repeated
// certificates form the same batches and reuse the same scratch.  A curve
// shared by two batches is built in both.
std::vector<std::vector<int64_t>> form_batches(flk_ctx *ctx, const int32_t *pairs, const std::vector<int64_t> &bh_idx,
                                               const flk_params &prm) {
  Curves &cv = ctx->curves;
  int64_t budget;
  if (prm.bh_batch_ksegs > 0) {
    budget = (int64_t)prm.bh_batch_ksegs * 1000;
  } else {
    if (cv.bh_budget <= 0) {
      size_t free_b = 0, total_b = 0;
      FLK_HIP(hipMemGetInfo(&free_b, &total_b));
      cv.bh_budget = (int64_t)(0.6 * (double)(free_b + ctx->bh.bytes()) / kBhBytesPerSegment);
    }
    budget = cv.bh_budget;
  }
  budget = std::max<int64_t>(budget, 1);
  std::vector<std::vector<int64_t>> out;
  std::vector<char> in_batch(cv.ncurves, 0);
  std::vector<int32_t> members;
  std::vector<int64_t> batch;
  int64_t segs = 0;
  auto flush = [&]() {
    if (batch.empty()) return;
    out.push_back(batch);
    for (int32_t c : members) in_batch[c] = 0;
    members.clear();
    batch.clear();
    segs = 0;
  };
  for (int64_t k : bh_idx) {
    const int32_t a = pairs[2 * k], b = pairs[2 * k + 1];
    const int64_t add = (in_batch[a] ? 0 : cv.n[a]) + (in_batch[b] || a == b ? 0 : cv.n[b]);
    if (!batch.empty() && segs + add > budget) flush();
    for (int32_t c : {a, b})
      if (!in_batch[c]) {
        in_batch[c] = 1;
        members.push_back(c);
        segs += cv.n[c];
      }
    batch.push_back(k);
  }
  flush();
  return out;
}

}  // namespace

// A whole Barnes–Hut certificate as one captured graph: the direct-sum batch
// of the pairs below the threshold (persistent tile kernel, reduction) and, per Barnes–Hut batch, the forest build (sort,
// topology, moments), both traversal passes with the device re-run decision
// between them and the merge, results straight to pinned memory: kernels only.  The device pointers it holds
// belong to the context's scratch: it is replayed only while no DevBuf has
// been allocated or freed since its capture (g_devbuf_epoch).  Its plans follow
// from the pairs and the curves' sizes but for the key boxes, so new positions
// of the same curves replay it too, with the plans sent again: capturing and
// instantiating 50-100 nodes for each step of a simulation took longer than
// running them.  With one Barnes–Hut batch the second pass is a graph of its own
// (`again`), launched when the first has pairs to re-run, which is known after
// it: 7 launches of a walk or 45-50 of levels that would find nothing take 36 or
// 250 us.  A certificate that had re-runs is launched with it at once.
struct CertGraph {
  GraphKey key;
  uint64_t epoch = 0;
  hipGraphExec_t exec = nullptr, again = nullptr;
  bool reran = false;  // the last launch had pairs to re-run
  std::vector<int64_t> ds_idx;
  DsGraph ds;
  std::vector<BatchPlan> batches;
  ~CertGraph() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (again) (void)hipGraphExecDestroy(again);
  }
};

namespace {

// What `body` enqueues on s, captured and instantiated.
template <typename F> hipGraphExec_t captured(hipStream_t s, F &&body) {
  hipGraph_t graph = nullptr;
  FLK_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  t_capturing = true;
  try {
    body();
  } catch (...) {
    t_capturing = false;
    (void)hipStreamEndCapture(s, &graph);
    if (graph) (void)hipGraphDestroy(graph);
    throw;
  }
  t_capturing = false;
  FLK_HIP(hipStreamEndCapture(s, &graph));
  hipGraphExec_t exec = nullptr;
  const hipError_t ie = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (ie != hipSuccess) throw Error(FLK_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(ie));
  return exec;
}

// Most batches of one graph (about 7,000 nodes in a chain; a call that would
// have captured hundreds of thousands, 5e5 pairs in batches of 250 curves, ended in
// a segmentation fault on the host).  The largest benchmark has two.
constexpr size_t kGraphBatches = 64;

// Captures (or finds) the certificate graph for these pairs and launches it;
// false when a batch does not fit the device schedule, or there are too many
// (the caller then runs the eager path).
bool bh_run_graph(flk_ctx *ctx, const int32_t *pairs, int64_t npairs, const flk_params &prm,
                  const std::vector<int64_t> &ds_idx, const std::vector<int32_t> &ds_pairs,
                  const std::vector<int64_t> &bh_idx, std::vector<double> &lk, std::vector<double> &err,
                  std::vector<uint32_t> &flags) {
  hipStream_t s = ctx->stream;
  const bool use_mlp = prm.criterion == FLK_CRIT_MLP;
  const float eps = (float)(prm.eps_sq * ctx->curves.scale * ctx->curves.scale);  // as the traversal has it
  GraphKey key(ctx, pairs, npairs);
  key.add(std::array<double, 6>{prm.beta_init, prm.beta_limit, prm.target_error, prm.err_scale, prm.mlp_log_tol, eps});
  key.add(std::array<int64_t, 5>{prm.criterion, prm.bh_direct_threshold, prm.leaf_size, prm.fp64, prm.bh_batch_ksegs});
  key.add(ctx->tune);
  CertGraph *G = ctx->cert_graph.get();
  PlanUpload up;
  if (!(G && G->key == key && G->epoch == g_devbuf_epoch.load())) {
    auto formed = form_batches(ctx, pairs, bh_idx, prm);
    if (formed.size() > kGraphBatches) return false;
    auto NG = std::make_shared<CertGraph>();
    if (G) NG->ds.take_buffers(G->ds);
    ctx->cert_graph.reset();
    NG->key = std::move(key);
    NG->ds_idx = ds_idx;
    for (auto &idx : formed) {
      NG->batches.emplace_back();
      BatchPlan &bp = NG->batches.back();
      plan_batch(ctx, pairs, std::move(idx), prm, bp);
      if (!bp.device) return false;
    }
    for (BatchPlan &bp : NG->batches) bp.add(up);
    up.send(ctx, s);
    if (!ds_idx.empty()) {
      // Beside the Barnes-Hut branch the direct-sum kernel takes a share of
      // its resident blocks, the direct sum's fraction of the two parts'
      // estimated times alone: its segment pairs at 1.2e12 per second (FP64:
      // 4.5e11), and 0.19 ns per Barnes-Hut tree segment for build and
      // traversal.  Both rates are the 10,000-loop lattice's (5.6e10 direct
      // pairs, 3.2e8 tree segments; share 0.43, 3 of the 8 blocks per CU),
      // whose certificate took 109 ms with the parts in sequence, 97 ms as two
      // branches at full residency, 87, 84 and 97 ms with 4, 3 and 2 blocks.
      double share = 1.0;
      if (!NG->batches.empty()) {
        const std::vector<int32_t> &n = ctx->curves.n;
        double work = 0.0, bh_segments = 0.0;
        for (size_t k = 0; k + 1 < ds_pairs.size(); k += 2)
          work += (double)n[ds_pairs[k]] * (double)n[ds_pairs[k + 1]];
        for (const BatchPlan &bp : NG->batches) bh_segments += (double)bp.forest.S;
        const double t_ds = work / (prm.fp64 ? 4.5e11 : 1.2e12), t_bh = bh_segments * 0.19e-9;
        share = t_ds / (t_ds + t_bh);
      }
      ds_capture_prepare(ctx, ds_pairs.data(), (int64_t)ds_idx.size(), prm.fp64 != 0, NG->ds, share);
    }
    FLK_HIP(hipStreamSynchronize(s));
    // A hybrid certificate's direct-sum part (VALU-bound) and its Barnes-Hut
    // batches (memory-bound builds and traversals) share nothing they write:
    // the direct sum is a branch of its own, forked from the capture stream
    // onto the context's second stream and joined before the capture ends.
    const bool fork = !ds_idx.empty() && !NG->batches.empty();
    NG->exec = captured(s, [&]() {
      bool forked = false;
      try {
        if (fork) {
          FLK_HIP(hipEventRecord(ctx->ev_fork, s));
          FLK_HIP(hipStreamWaitEvent(ctx->aux, ctx->ev_fork, 0));
          forked = true;
          ds_capture_enqueue(ctx, NG->ds, ctx->aux);
        } else if (!ds_idx.empty()) {
          ds_capture_enqueue(ctx, NG->ds, s);
        }
        for (BatchPlan &bp : NG->batches) {
          enqueue_forest(ctx, bp.forest, s);
          enqueue_traversal(ctx, bp, prm, s, true, NG->batches.size() > 1);
        }
      } catch (...) {
        if (forked) {  // the capture cannot end with a branch left open
          (void)hipEventRecord(ctx->ev_join, ctx->aux);
          (void)hipStreamWaitEvent(s, ctx->ev_join, 0);
        }
        throw;
      }
      if (forked) {
        FLK_HIP(hipEventRecord(ctx->ev_join, ctx->aux));
        FLK_HIP(hipStreamWaitEvent(s, ctx->ev_join, 0));
      }
    });
    NG->epoch = g_devbuf_epoch.load();
    ctx->cert_graph = NG;
    G = NG.get();
  } else {
    if (use_mlp) mlp_upload(ctx);  // the weights as they are now (same buffers)
    for (BatchPlan &bp : G->batches) {
      plan_boxes(ctx->curves, bp.forest);
      bp.add(up);
    }
    up.send(ctx, s);
  }
  FLK_HIP(hipEventRecord(ctx->ev0, s));
  const auto t0 = std::chrono::steady_clock::now();
  FLK_HIP(hipGraphLaunch(G->exec, s));
  ctx->stats.ms_graph_launch =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  const bool at_once = G->again && G->reran;
  if (at_once) FLK_HIP(hipGraphLaunch(G->again, s));
  FLK_HIP(hipEventRecord(ctx->ev1, s));
  FLK_HIP(hipStreamSynchronize(s));
  if (G->batches.size() == 1) {
    const unsigned long long *head = G->batches[0].heads();
    G->reran = head[kPassHead + 4] != 0;
    if (G->reran && !at_once && head[6] == 0) {  // (an overflowed first pass goes to the host)
      if (!G->again)
        G->again = captured(s, [&]() { enqueue_traversal(ctx, G->batches[0], prm, s, false, true); });
      FLK_HIP(hipGraphLaunch(G->again, s));
      FLK_HIP(hipEventRecord(ctx->ev1, s));
      FLK_HIP(hipStreamSynchronize(s));
    }
  }
  float ms = 0.f;
  FLK_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
  ctx->stats.ms_kernel = ms;
  ctx->stats.graph_launches += 1;
  if (!G->ds_idx.empty()) {
    for (size_t t = 0; t < G->ds_idx.size(); ++t) lk[G->ds_idx[t]] = G->ds.h_out.as<double>()[t];
    ctx->stats.ds_seg_pairs += G->ds.work;
    ctx->stats.ds_launches += G->ds.tasks.empty() ? 0 : 1;
    ctx->stats.ds_waves = G->ds.waves;
  }
  // keep the graph alive while batches that overflowed re-run eagerly (their
  // allocations retire it for the next call)
  std::shared_ptr<CertGraph> hold = ctx->cert_graph;
  for (BatchPlan &bp : G->batches) {
    bp.collect();
    if (!finish_batch(ctx, bp, lk, err, flags)) bh_batch_host(ctx, pairs, bp.idx, prm, lk, err, flags);
  }
  return true;
}

}  // namespace

void bh_run(flk_ctx *ctx, const int32_t *pairs, int64_t npairs, const flk_params &prm,
            std::vector<double> &lk, std::vector<double> &err, std::vector<uint32_t> &flags) {
  Curves &cv = ctx->curves;
  lk.assign(npairs, 0.0);
  err.assign(npairs, 0.0);
  flags.assign(npairs, 0u);
  if (npairs == 0) return;
  const bool use_mlp = prm.criterion == FLK_CRIT_MLP;
  if (use_mlp && !ctx->mlp.loaded)
    throw Error(FLK_ERR_STATE, "the learned criterion needs weights (flk_mlp_set_weights)");
  // Pairs below the direct threshold (or with a curve too short for a tree)
  // go to the direct sum; the rest to Barnes–Hut.
  std::vector<int64_t> ds_idx, bh_idx;
  std::vector<int32_t> ds_pairs;
  for (int64_t k = 0; k < npairs; ++k) {
    const int32_t a = pairs[2 * k], b = pairs[2 * k + 1];
    const int64_t work = (int64_t)cv.n[a] * cv.n[b];
    if (cv.n[a] < 2 || cv.n[b] < 2 || work < prm.bh_direct_threshold) {
      ds_idx.push_back(k);
      ds_pairs.push_back(a);
      ds_pairs.push_back(b);
      flags[k] |= FLK_PAIR_DIRECT;
    } else {
      bh_idx.push_back(k);
    }
  }
  // Default: the whole certificate (direct-sum part and every Barnes–Hut
  // batch) as one graph launch.
  if (prm.graph && !prm.timing && !bh_idx.empty() &&
      bh_run_graph(ctx, pairs, npairs, prm, ds_idx, ds_pairs, bh_idx, lk, err, flags))
    return;
  if (!ds_idx.empty()) {
    std::vector<double> v;
    float ms = 0.f;
    ds_run(ctx, ds_pairs.data(), (int64_t)ds_idx.size(), prm.fp64 != 0, v, &ms, prm.graph != 0);
    ctx->stats.ms_ds_kernel += ms;
    for (size_t t = 0; t < ds_idx.size(); ++t) lk[ds_idx[t]] = v[t];
  }
  for (const auto &idx : form_batches(ctx, pairs, bh_idx, prm)) bh_batch(ctx, pairs, idx, prm, lk, err, flags);
}

}  // namespace flk
