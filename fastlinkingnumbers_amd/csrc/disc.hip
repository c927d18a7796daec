// Discretization of spline curves into polylines on the device (reference
// src/discretize.cpp:102-281).
//
// Every segment of every curve starts as one piece (curve, segment, t_lo = 0,
// t_hi = 1) with its exact FP64 box.  Each round builds an implicit BVH over the
// boxes of the live pieces, in the list's own order, which runs along the curves,
// or, where curves have many potential links, in Morton order; one query per piece
// walks it and, for every overlapping piece that belongs to a different curve of
// a potentially linked pair, counts the pair once and marks both pieces.  Marked
// pieces are bisected at the parameter midpoint (two new
// pieces with their boxes), the others retire.  The loop ends when a round
// finds no overlap, and fails after 55 rounds or when a new piece's box
// diagonal falls below eps * mean |q| / sqrt(3), as the reference does.  The
// retired pieces, radix-sorted by (curve segment, t_lo), give each curve's
// polyline vertices.
//
// Boxes and points use the reference's formulas (cubic bases, cancellation-
// free quadratic for the derivative roots, closed-interval overlap) in FP64
// with floating-point contraction off, so every box and every overlap decision
// is the same as the host restatement's, bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <limits>

#include "flk_internal.h"

#pragma clang fp contract(off)

namespace flk {

namespace {

// Segment types in the order of VerifyCurves::SegmentType (2 is Bezier).
constexpr int kBSpline = 0, kCatmullRom = 1, kPolyline = 3;

struct DCurve {
  int64_t q0;    // first control point in the packed array
  int32_t n;     // control points
  int32_t type;  // segment type
  int32_t nseg;  // segments (looped: n; open: n - 1 polyline, n - 3 spline)
  int32_t seg0;  // global index of the first segment
};

struct PBox {
  double mn[3], mx[3];
};

__device__ __forceinline__ double dmin(double a, double b) { return (b < a) ? b : a; }  // std::min
__device__ __forceinline__ double dmax(double a, double b) { return (a < b) ? b : a; }  // std::max

// One coordinate of a cubic segment in the power basis and its exact range
// over [t0, t1]: endpoint values and the derivative roots inside
// (reference curve.cpp:197-277; complex roots give NaN, rejected by every
// comparison).
__device__ void coord_range(int type, double a, double b, double c, double d, double t0, double t1, double &lo,
                            double &hi) {
  double k3, k2, k1, k0;
  if (type == kBSpline) {
    k3 = -(1.0 / 6.0) * a + 0.5 * b - 0.5 * c + (1.0 / 6.0) * d;
    k2 = 0.5 * a - b + 0.5 * c;
    k1 = -0.5 * a + 0.5 * c;
    k0 = (1.0 / 6.0) * a + (2.0 / 3.0) * b + (1.0 / 6.0) * c;
  } else if (type == kCatmullRom) {
    k3 = -0.5 * a + 1.5 * b - 1.5 * c + 0.5 * d;
    k2 = 1.0 * a - 2.5 * b + 2.0 * c - 0.5 * d;
    k1 = -0.5 * a + 0.5 * c;
    k0 = 1.0 * b;
  } else {
    k3 = -1.0 * a + 3.0 * b - 3.0 * c + 1.0 * d;
    k2 = 3.0 * a - 6.0 * b + 3.0 * c;
    k1 = -3.0 * a + 3.0 * b;
    k0 = 1.0 * a;
  }
  auto f = [&](double t) { return ((k3 * t + k2) * t + k1) * t + k0; };
  lo = f(t0);
  hi = f(t1);
  if (hi < lo) {
    const double s = lo;
    lo = hi;
    hi = s;
  }
  auto take = [&](double t) {
    if (t >= t0 && t <= t1) {
      const double v = f(t);
      lo = dmin(lo, v);
      hi = dmax(hi, v);
    }
  };
  const double disc = 4 * k2 * k2 - 12 * k1 * k3;
  if (disc == 0) {
    take(-2 * k2 / (6 * k3));
  } else {
    const double r = k2 >= 0 ? -2 * k2 - sqrt(disc) : -2 * k2 + sqrt(disc);
    take(r / (6 * k3));
    take(2 * k1 / r);
  }
}

// Point of segment i at parameter t (reference curve.cpp:99-131).
__device__ void curve_point(const double *__restrict__ q, const DCurve &C, int i, double t, double p[3]) {
  const int n = C.n;
  const double *a = q + 3 * (C.q0 + i), *b = q + 3 * (C.q0 + (i + 1) % n);
  if (C.type == kPolyline) {
    for (int d = 0; d < 3; ++d) p[d] = (1.0 - t) * a[d] + t * b[d];
    return;
  }
  double B[4];
  if (C.type == kBSpline) {
    B[0] = ((-(1.0 / 6) * t + (1.0 / 2)) * t - (1.0 / 2)) * t + (1.0 / 6);
    B[1] = ((1.0 / 2) * t - 1.0) * (t * t) + (2.0 / 3);
    B[2] = ((-(1.0 / 2) * t + (1.0 / 2)) * t + (1.0 / 2)) * t + (1.0 / 6);
    B[3] = (1.0 / 6) * (t * t) * t;
  } else if (C.type == kCatmullRom) {
    B[0] = ((-0.5 * t + 1.0) * t - 0.5) * t;
    B[1] = (1.5 * t - 2.5) * (t * t) + 1.0;
    B[2] = ((-1.5 * t + 2.0) * t + 0.5) * t;
    B[3] = (0.5 * t - 0.5) * (t * t);
  } else {
    B[0] = ((-1.0 * t + 3.0) * t - 3.0) * t + 1.0;
    B[1] = ((3.0 * t - 6.0) * t + 3.0) * t;
    B[2] = (-3.0 * t + 3.0) * (t * t);
    B[3] = 1.0 * t * t * t;
  }
  const double *c = q + 3 * (C.q0 + (i + 2) % n), *e = q + 3 * (C.q0 + (i + 3) % n);
  for (int d = 0; d < 3; ++d) p[d] = B[0] * a[d] + B[1] * b[d] + B[2] * c[d] + B[3] * e[d];
}

// Exact box of segment i over [tlo, thi] (reference curve.cpp:293-324).
__device__ PBox seg_box(const double *__restrict__ q, const DCurve &C, int i, double tlo, double thi) {
  PBox b;
  if (C.type == kPolyline) {
    double pa[3], pb[3];
    curve_point(q, C, i, tlo, pa);
    curve_point(q, C, i, thi, pb);
    for (int d = 0; d < 3; ++d) {
      b.mn[d] = dmin(pa[d], pb[d]);
      b.mx[d] = dmax(pa[d], pb[d]);
    }
  } else {
    const int n = C.n;
    for (int d = 0; d < 3; ++d)
      coord_range(C.type, q[3 * (C.q0 + i) + d], q[3 * (C.q0 + (i + 1) % n) + d], q[3 * (C.q0 + (i + 2) % n) + d],
                  q[3 * (C.q0 + (i + 3) % n) + d], tlo, thi, b.mn[d], b.mx[d]);
  }
  for (int d = 0; d < 3; ++d) {
    b.mn[d] -= 0.0;
    b.mx[d] += 0.0;
  }
  return b;
}

__device__ __forceinline__ double box_diag(const PBox &b) {
  const double x = b.mx[0] - b.mn[0], y = b.mx[1] - b.mn[1], z = b.mx[2] - b.mn[2];
  return sqrt(x * x + y * y + z * z);
}

__device__ __forceinline__ bool overlap(const PBox &a, const PBox &b) {
  return a.mn[0] <= b.mx[0] && a.mn[1] <= b.mx[1] && a.mn[2] <= b.mx[2] && b.mn[0] <= a.mx[0] &&
         b.mn[1] <= a.mx[1] && b.mn[2] <= a.mx[2];
}

__device__ __forceinline__ int curve_of(const DCurve *__restrict__ cs, int nc, int64_t g) {
  int lo = 0, hi = nc;  // last c with seg0 <= g
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cs[mid].seg0 <= g) lo = mid;
    else hi = mid;
  }
  return lo;
}

// One piece per segment: (curve, segment, 0, 1), its box and diagonal.
// Also reduced per block: the sum of the segments' first points' norms, the
// first smallest box diagonal and whether any is NaN,
// and those by disc_fold, so the host reads 32 bytes instead of every point and diagonal: with
// the scratch kept between calls, a discretization of 8.8e5 splines took 16.2 ms
// and takes 2.3.
struct InitPart {
  double sum, md;
  int64_t mg;
  int64_t nan;
};
__device__ __forceinline__ void fold_part(InitPart &a, const InitPart &b) {
  a.sum += b.sum;
  a.nan |= b.nan;
  if (b.md < a.md || (b.md == a.md && b.mg < a.mg)) {
    a.md = b.md;
    a.mg = b.mg;
  }
}
// Thread 0's r becomes the block's (WAVES waves, as many entries of LDS).
template <int WAVES> __device__ __forceinline__ void fold_block(InitPart &r, InitPart *sp) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    InitPart u;
    u.sum = __shfl_down(r.sum, o, 64);
    u.md = __shfl_down(r.md, o, 64);
    u.mg = __shfl_down(r.mg, o, 64);
    u.nan = __shfl_down(r.nan, o, 64);
    fold_part(r, u);
  }
  if ((threadIdx.x & 63) == 0) sp[threadIdx.x >> 6] = r;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 1; k < WAVES; ++k) fold_part(r, sp[k]);
}
__global__ __launch_bounds__(256) void disc_init(const double *__restrict__ q, const DCurve *__restrict__ cs,
                                                 int32_t nc, int64_t nseg, int32_t *__restrict__ pc,
                                                 int32_t *__restrict__ ps, double *__restrict__ plo,
                                                 double *__restrict__ phi, PBox *__restrict__ pbox,
                                                 double *__restrict__ diag, InitPart *__restrict__ part) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  InitPart r{0.0, __builtin_inf(), INT64_MAX, 0};
  if (g < nseg) {
    const int c = curve_of(cs, nc, g);
    const DCurve C = cs[c];
    const int s = (int)(g - C.seg0);
    const PBox b = seg_box(q, C, s, 0.0, 1.0);
    const double d = box_diag(b);
    pc[g] = c;
    ps[g] = s;
    plo[g] = 0.0;
    phi[g] = 1.0;
    pbox[g] = b;
    diag[g] = d;
    const double *p0 = q + 3 * (C.q0 + s);
    r.sum = sqrt(p0[0] * p0[0] + p0[1] * p0[1] + p0[2] * p0[2]);
    r.nan = d != d;
    r.md = d;
    r.mg = g;
  }
  __shared__ InitPart sp[4];
  fold_block<4>(r, sp);
  if (threadIdx.x == 0) part[blockIdx.x] = r;
}

// The blocks' folded, straight into pinned memory.
__global__ __launch_bounds__(1024) void disc_fold(const InitPart *__restrict__ part, int64_t n,
                                                  InitPart *__restrict__ host) {
  InitPart r{0.0, __builtin_inf(), INT64_MAX, 0};
  for (int64_t k = threadIdx.x; k < n; k += 1024) fold_part(r, part[k]);
  __shared__ InitPart sp[16];
  fold_block<16>(r, sp);
  if (threadIdx.x == 0) *host = r;
}

// A round's overlaps and marked pieces into pinned memory.
__global__ void disc_report(const unsigned long long *__restrict__ cnt, const int32_t *__restrict__ nhit,
                            unsigned long long *__restrict__ host) {
  host[0] = cnt[0];
  host[1] = (unsigned long long)*nhit;
}

// A node of the implicit tree: its box about a point of the model, rounded
// outward to FP32 (32 bytes instead of 48; the leaves' pieces are tested again
// in FP64).  About 0 a model at 1e7, where an FP32 number is 1 from the next, had
// long runs of pieces to test: 256 rings of 400 segments 5.4 ms, 1.3 at 0.  The
// difference is rounded, but no bound overtakes another by it, so boxes that
// overlap still do.
struct FBox {
  float4 mn, mx;
};
__device__ __forceinline__ FBox outward(const PBox &b, const double3 &o) {
  return FBox{make_float4(__double2float_rd(b.mn[0] - o.x), __double2float_rd(b.mn[1] - o.y),
                          __double2float_rd(b.mn[2] - o.z), 0.f),
              make_float4(__double2float_ru(b.mx[0] - o.x), __double2float_ru(b.mx[1] - o.y),
                          __double2float_ru(b.mx[2] - o.z), 0.f)};
}
__device__ __forceinline__ bool overlap(const FBox &a, const FBox &b) {
  return a.mn.x <= b.mx.x && a.mn.y <= b.mx.y && a.mn.z <= b.mx.z && b.mn.x <= a.mx.x && b.mn.y <= a.mx.y &&
         b.mn.z <= a.mx.z;
}

// Cells of a piece's box centre in the model's box, 10 bits an axis, interleaved.
__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  return (v | (v << 2)) & 0x09249249u;
}
__global__ __launch_bounds__(256) void disc_morton(const PBox *__restrict__ pbox, int64_t n, double3 lo, double3 cells,
                                                   uint32_t *__restrict__ keys, uint32_t *__restrict__ ids) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const PBox b = pbox[i];
  auto cell = [](double mn, double mx, double first, double per) {  // NaN: 0
    return (uint32_t)fmin(fmax((0.5 * (mn + mx) - first) * per, 0.0), 1023.0);
  };
  keys[i] = spread10(cell(b.mn[0], b.mx[0], lo.x, cells.x)) << 2 | spread10(cell(b.mn[1], b.mx[1], lo.y, cells.y)) << 1 |
            spread10(cell(b.mn[2], b.mx[2], lo.z, cells.z));
  ids[i] = (uint32_t)i;
}

// Eight levels of the tree a launch: a block takes 256 nodes of level M (heap
// slots [M, 2M); with LEAVES it makes them of the pieces' boxes, empty ones
// padding to the power of two M) and writes the unions above them (slot k: of
// slots 2k and 2k + 1).  LEAVES takes the pieces in `order`, or in the list's own
// and then also notes where each curve's pieces lie.
template <bool LEAVES>
__global__ __launch_bounds__(256) void disc_tree(const PBox *__restrict__ pbox, const int32_t *__restrict__ pc,
                                                 const uint32_t *__restrict__ order, int64_t n, double3 origin,
                                                 int64_t M, FBox *__restrict__ heap, int2 *__restrict__ range) {
  __shared__ FBox sb[256];
  const int t = threadIdx.x, cnt = (int)min((int64_t)256, M);
  const int64_t i = (int64_t)blockIdx.x * 256 + t;
  FBox b{make_float4(FLT_MAX, FLT_MAX, FLT_MAX, 0.f), make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, 0.f)};
  if (t < cnt) {
    if (!LEAVES) b = heap[M + i];
    else {
      if (i < n) {
        b = outward(pbox[order ? order[i] : i], origin);
        if (!order) {
          const int c = pc[i];
          if (i == 0 || pc[i - 1] != c) range[c].x = (int32_t)i;
          if (i + 1 == n || pc[i + 1] != c) range[c].y = (int32_t)(i + 1);
        }
      }
      heap[M + i] = b;
    }
    sb[t] = b;
  }
  int64_t at = (M + (int64_t)blockIdx.x * 256) >> 1;
  for (int w = cnt >> 1; w >= 1; w >>= 1, at >>= 1) {
    __syncthreads();
    if (t < w) {
      const FBox l = sb[2 * t], r = sb[2 * t + 1];
      b = FBox{make_float4(fminf(l.mn.x, r.mn.x), fminf(l.mn.y, r.mn.y), fminf(l.mn.z, r.mn.z), 0.f),
               make_float4(fmaxf(l.mx.x, r.mx.x), fmaxf(l.mx.y, r.mx.y), fmaxf(l.mx.z, r.mx.z), 0.f)};
      heap[at + t] = b;
    }
    __syncthreads();
    if (t < w) sb[t] = b;
  }
}

// Potential link between curves a < b: binary search of the sorted keys.
__device__ __forceinline__ bool linked(const uint64_t *__restrict__ keys, int64_t m, int a, int b) {
  const uint64_t key = ((uint64_t)(uint32_t)min(a, b) << 32) | (uint32_t)max(a, b);
  int64_t lo = 0, hi = m;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo < m && keys[lo] == key;
}

// Leaves [at, end) of the tree whose boxes overlap q's, each given to `leaf`.  The
// walk keeps no stack: it takes the largest subtree that starts at `at` and ends
// by `end`, goes down to the left where boxes overlap and else on behind the
// subtree.
template <typename F>
__device__ __forceinline__ void walk_leaves(const FBox *__restrict__ heap, uint32_t L, uint32_t at, uint32_t end,
                                            const FBox &q, F &&leaf) {
  if (at >= end) return;
  auto largest = [&]() { return min(__builtin_ctz(L + at), 31 - __builtin_clz(end - at)); };
  int h = largest();
  for (;;) {
    if (overlap(heap[(L + at) >> h], q)) {
      if (h > 0) {
        --h;
        continue;
      }
      leaf((int64_t)at);
    }
    at += 1u << h;
    if (at >= end) return;
    h = largest();
  }
}

// One query per piece, over a tree of the pieces in the list's own order, which
// runs along the curves: the pieces of its curve's partners, one partner after
// the other (each potential link is asked from one of its curves).  What a query
// costs does not depend on the order of the curves: walking every piece
// behind its own curve, 10,000 rings of 60 segments in random order took 156 ms
// and take 2.2, as in order (the query of 8.8e5 pieces of 576 curves 100 us -> 60).
// SORTED: where a curve asks more than kMostPartners, a tree of the pieces in
// Morton order; a query takes the pieces behind its own and looks their curves
// up among the links.  Whole calls on closed curves through one another, listed and
// sorted: 20 of 5,000 segments 0.87 and 1.24 ms, 50 of 200 2.7 and 2.3, 500 of 500
// 24 and 5.9 (58 by walking the list), 100 of 40 beside 3,600 rings 5.8 and 4.5;
// chain mail of 1,600 rings (2 partners) 1.5 and 3.0.
constexpr int32_t kMostPartners = 32;
template <bool SORTED>
__global__ __launch_bounds__(256) void disc_query(const FBox *__restrict__ heap, const PBox *__restrict__ pbox,
                                                  int64_t n, double3 origin, int64_t L,
                                                  const int32_t *__restrict__ pc, const uint32_t *__restrict__ order,
                                                  const uint64_t *__restrict__ links, int64_t nlinks,
                                                  const int2 *__restrict__ range, const int32_t *__restrict__ first,
                                                  const int32_t *__restrict__ partner,
                                                  uint8_t *__restrict__ hit, unsigned long long *__restrict__ count) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int found = 0;
  if (t < n) {
    const int64_t i = SORTED ? order[t] : t;
    const int c = pc[i];
    const PBox me = pbox[i];
    const FBox q = outward(me, origin);
    auto both = [&](int64_t o) {
      ++found;
      hit[i] = 1;
      hit[o] = 1;
    };
    if (SORTED) {
      walk_leaves(heap, (uint32_t)L, (uint32_t)t + 1, (uint32_t)n, q, [&](int64_t at) {
        const int64_t o = order[at];
        if (pc[o] != c && overlap(pbox[o], me) && linked(links, nlinks, c, pc[o])) both(o);
      });
    } else {
      for (int32_t k = first[c]; k < first[c + 1]; ++k) {
        const int2 r = range[partner[k]];
        walk_leaves(heap, (uint32_t)L, (uint32_t)r.x, (uint32_t)r.y, q, [&](int64_t o) {
          if (overlap(pbox[o], me)) both(o);
        });
      }
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) found += __shfl_xor(found, off, 64);
  __shared__ int sf[4];
  if ((threadIdx.x & 63) == 0) sf[threadIdx.x >> 6] = found;
  __syncthreads();
  if (threadIdx.x == 0) {
    found = sf[0] + sf[1] + sf[2] + sf[3];
    if (found) atomicAdd(count, (unsigned long long)found);
  }
}

__global__ __launch_bounds__(256) void disc_flags(const uint8_t *__restrict__ hit, int64_t n,
                                                  int32_t *__restrict__ f) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) f[i] = hit[i] ? 1 : 0;
}

// Marked pieces split at the midpoint into slots 2 s, 2 s + 1 of the next
// list (s = marked pieces before this one); unmarked pieces retire to slot
// r0 + i - s of the retired list.  too_small is set when a new box's
// diagonal is below the threshold.
__global__ __launch_bounds__(256) void disc_split(const double *__restrict__ q, const DCurve *__restrict__ cs,
                                                  int64_t n, const uint8_t *__restrict__ hit,
                                                  const int32_t *__restrict__ scan, const int32_t *__restrict__ pc,
                                                  const int32_t *__restrict__ ps, const double *__restrict__ plo,
                                                  const double *__restrict__ phi, int32_t *__restrict__ nc_,
                                                  int32_t *__restrict__ ns_, double *__restrict__ nlo,
                                                  double *__restrict__ nhi, PBox *__restrict__ nbox,
                                                  int64_t r0, int32_t *__restrict__ rc, int32_t *__restrict__ rs,
                                                  double *__restrict__ rlo, double *__restrict__ rhi,
                                                  double threshold, int32_t *__restrict__ too_small) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = pc[i], s = ps[i];
  const double lo = plo[i], hi = phi[i];
  const int64_t before = scan[i];
  if (hit[i]) {
    const DCurve C = cs[c];
    const double mid = 0.5 * (lo + hi);
    const PBox b1 = seg_box(q, C, s, lo, mid), b2 = seg_box(q, C, s, mid, hi);
    if (!(box_diag(b1) >= threshold) || !(box_diag(b2) >= threshold)) *too_small = 1;
    const int64_t o = 2 * before;
    nc_[o] = c;
    ns_[o] = s;
    nlo[o] = lo;
    nhi[o] = mid;
    nbox[o] = b1;
    nc_[o + 1] = c;
    ns_[o + 1] = s;
    nlo[o + 1] = mid;
    nhi[o + 1] = hi;
    nbox[o + 1] = b2;
  } else {
    const int64_t o = r0 + (i - before);
    rc[o] = c;
    rs[o] = s;
    rlo[o] = lo;
    rhi[o] = hi;
  }
}

// Sort keys of a retired piece, for two stable passes: t_lo as the integer
// t_lo * 2^R (t_lo is a dyadic fraction with at most R <= 55 bits), then the
// global segment index.  Two passes keep the order (segment, t_lo) for any
// segment count and round count the reference allows.
__global__ __launch_bounds__(256) void disc_keys(const DCurve *__restrict__ cs, const int32_t *__restrict__ rc,
                                                 const int32_t *__restrict__ rs, const double *__restrict__ rlo,
                                                 int64_t n, int R, uint64_t *__restrict__ tkey,
                                                 uint32_t *__restrict__ ids, int32_t *__restrict__ per_curve) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    tkey[i] = (uint64_t)ldexp(rlo[i], R);
    ids[i] = (uint32_t)i;
  }
  // pieces of each curve: one atomic per curve in the wave (most often one)
  const int c = i < n ? rc[i] : -1;
  uint64_t left = __ballot(c >= 0);
  while (left) {
    const int lead = __builtin_ctzll(left);
    const int cl = __shfl(c, lead, 64);
    const uint64_t same = __ballot(c == cl);
    if ((int)(threadIdx.x & 63) == lead) atomicAdd(per_curve + cl, __popcll(same));
    left &= ~same;
  }
}

// Second pass's keys in the first pass's order: the global segment of piece
// perm[k].
__global__ __launch_bounds__(256) void disc_seg_keys(const DCurve *__restrict__ cs, const int32_t *__restrict__ rc,
                                                     const int32_t *__restrict__ rs, const uint32_t *__restrict__ perm,
                                                     int64_t n, uint32_t *__restrict__ gkey) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t i = perm[k];
  gkey[k] = (uint32_t)(cs[rc[i]].seg0 + rs[i]);
}

// Output vertex of sorted retired piece k: its start point at out[k + the
// number of open curves before its curve]; an open curve's last piece also
// writes its end point after it.
__global__ __launch_bounds__(256) void disc_points(const double *__restrict__ q, const DCurve *__restrict__ cs,
                                                   const int32_t *__restrict__ order, const int32_t *__restrict__ rc,
                                                   const int32_t *__restrict__ rs, const double *__restrict__ rlo,
                                                   const double *__restrict__ rhi, int64_t n,
                                                   const int32_t *__restrict__ open_before,
                                                   const int32_t *__restrict__ is_open, double *__restrict__ out) {
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int32_t p = order[k];
  const int c = rc[p];
  const DCurve C = cs[c];
  double v[3];
  curve_point(q, C, rs[p], rlo[p], v);
  const int64_t o = k + open_before[c];
  for (int d = 0; d < 3; ++d) out[3 * o + d] = v[d];
  if (is_open[c]) {
    const bool last = k + 1 == n || rc[order[k + 1]] != c;
    if (last) {
      curve_point(q, C, rs[p], rhi[p], v);
      for (int d = 0; d < 3; ++d) out[3 * (o + 1) + d] = v[d];
    }
  }
}

unsigned blocks_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + 255) / 256); }

}  // namespace

// The output polylines become the context's curve set (device to device);
// res.xyz receives a host copy when host_copy is set.
void discretize_run(flk_ctx *ctx, const double *ctrl, const int64_t *offsets, const int32_t *types,
                    const uint8_t *looped, int32_t nc, const int32_t *pairs, int64_t npairs, DiscResult &res,
                    bool host_copy) {
  hipStream_t s = ctx->stream;
  DiscScratch &D = ctx->disc_scratch;
  struct GiveBack {
    DiscScratch &D;
    hipStream_t s;
    ~GiveBack() {
      if (D.bytes() <= DiscScratch::kKept) return;
      (void)hipStreamSynchronize(s);
      D = DiscScratch{};
    }
  } give_back{D, s};
  res = DiscResult{};
  // curves and their segments
  std::vector<DCurve> cs(nc);
  int64_t nseg = 0;
  for (int32_t c = 0; c < nc; ++c) {
    const int64_t n = offsets[c + 1] - offsets[c];
    if (n < 0 || n > INT32_MAX / 2) throw Error(FLK_ERR_ARG, "bad curve offsets");
    if (types[c] < 0 || types[c] > 3) throw Error(FLK_ERR_ARG, "invalid segment type");
    const int32_t ns = looped[c] ? (int32_t)n : (int32_t)std::max<int64_t>(0, types[c] == kPolyline ? n - 1 : n - 3);
    cs[c] = DCurve{offsets[c], (int32_t)n, types[c], ns, (int32_t)nseg};
    nseg += ns;
    if (nseg > INT32_MAX / 4) throw Error(FLK_ERR_ARG, "too many segments to discretize");
  }
  res.segments = nseg;
  res.out_offsets.assign(nc + 1, 0);
  if (nseg == 0) {
    try {
      curves_layout(ctx, res.out_offsets.data(), nc);
      curves_finish(ctx);
    } catch (...) {
      curves_clear(ctx);
      throw;
    }
    return;
  }
  // potential links as sorted (min << 32 | max) keys
  std::vector<uint64_t> lk;
  lk.reserve(npairs);
  for (int64_t k = 0; k < npairs; ++k) {
    const int32_t a = pairs[2 * k], b = pairs[2 * k + 1];
    if (a < 0 || b < 0 || a >= nc || b >= nc) throw Error(FLK_ERR_ARG, "pair index out of range");
    if (a != b) lk.push_back(((uint64_t)(uint32_t)std::min(a, b) << 32) | (uint32_t)std::max(a, b));
  }
  std::sort(lk.begin(), lk.end());
  lk.erase(std::unique(lk.begin(), lk.end()), lk.end());

  // Each link is asked from its curve with fewer links (then with fewer segments):
  // the partners of curve c are partner[first[c]..first[c + 1]).
  std::vector<int32_t> first(nc + 1, 0), links_of(nc, 0);
  for (const uint64_t l : lk) {
    ++links_of[l >> 32];
    ++links_of[l & 0xffffffffu];
  }
  auto asks = [&](uint64_t l, int32_t &other) {
    const int32_t a = (int32_t)(l >> 32), b = (int32_t)(l & 0xffffffffu);
    const bool from_a = links_of[a] != links_of[b] ? links_of[a] < links_of[b] : cs[a].nseg <= cs[b].nseg;
    other = from_a ? b : a;
    return from_a ? a : b;
  };
  int32_t other = 0, most = 0;
  for (const uint64_t l : lk) most = std::max(most, ++first[asks(l, other) + 1]);
  const bool sorted = most > kMostPartners;
  std::vector<int32_t> partner(sorted ? 0 : lk.size());
  if (!sorted) {
    for (int32_t c = 0; c < nc; ++c) first[c + 1] += first[c];
    std::vector<int32_t> at(first.begin(), first.end() - 1);
    for (const uint64_t l : lk) {
      const int32_t c = asks(l, other);
      partner[at[c]++] = other;
    }
  }

  const int64_t nctrl = offsets[nc];
  DevBuf &d_cs = D.cs, &d_links = D.links, &d_cnt = D.cnt;
  d_cs.reserve(sizeof(DCurve) * nc);
  const size_t link_words = sorted ? lk.size() : (nc + 1 + lk.size() + 1) / 2;  // 8 bytes each
  d_links.reserve(sizeof(uint64_t) * std::max<size_t>(link_words, 1));
  d_cnt.reserve(sizeof(unsigned long long) * 2);
  // the control points: the current curve set's input array, or the caller's
  const double *q = ctx->curves.raw.as<double>();
  if (ctrl) {
    D.q.reserve(sizeof(double) * 3 * std::max<int64_t>(nctrl, 1));
    D.land.reserve(sizeof(float) * 3 * std::max<int64_t>(nctrl, 1));
    ingest_points(ctx, ctrl, false, nctrl, D.q.as<double>(), D.land.as<float>(), D.land.bytes);
    q = D.q.as<double>();
  }
  // The reference's guard threshold, eps times the mean first point's norm over
  // sqrt 3, its sum in the reference's order on the host: only where the
  // device's sum, in another order, cannot decide.
  const double eps = std::numeric_limits<double>::epsilon();
  auto threshold_of = [&](double sum) { return eps * (sum / (nseg * 1.73205080757)); };
  auto exact_threshold = [&]() {
    std::vector<double> current;
    const double *p0 = ctrl;
    if (!p0) {
      current.resize(3 * (size_t)nctrl);
      FLK_HIP(hipMemcpyAsync(current.data(), q, sizeof(double) * current.size(), hipMemcpyDeviceToHost, s));
      FLK_HIP(hipStreamSynchronize(s));
      p0 = current.data();
    }
    double sum = 0.0;
    for (int32_t c = 0; c < nc; ++c)
      for (int32_t k = 0; k < cs[c].nseg; ++k) {
        const double *p = p0 + 3 * (offsets[c] + k);
        sum += std::sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
      }
    return threshold_of(sum);
  };
  constexpr double kUnsure = 1e-6;  // far above either sum's rounding
  // everything small goes through pinned memory
  D.host.reserve(sizeof(InitPart) + 2 * sizeof(unsigned long long) + sizeof(uint64_t) * link_words +
                 (sizeof(DCurve) + 3 * sizeof(int32_t)) * (size_t)nc);
  InitPart *h_part = D.host.as<InitPart>();
  auto *h_report = reinterpret_cast<unsigned long long *>(h_part + 1);
  auto *h_links = reinterpret_cast<uint64_t *>(h_report + 2);
  auto *h_cs = reinterpret_cast<DCurve *>(h_links + link_words);
  auto *per_curve = reinterpret_cast<int32_t *>(h_cs + nc);
  int32_t *open_before = per_curve + nc, *is_open = open_before + nc;
  if (sorted) {
    std::copy(lk.begin(), lk.end(), h_links);
  } else {
    std::copy(first.begin(), first.end(), reinterpret_cast<int32_t *>(h_links));
    std::copy(partner.begin(), partner.end(), reinterpret_cast<int32_t *>(h_links) + nc + 1);
  }
  std::copy(cs.begin(), cs.end(), h_cs);
  FLK_HIP(hipMemcpyAsync(d_cs.ptr, h_cs, sizeof(DCurve) * nc, hipMemcpyHostToDevice, s));
  if (link_words)
    FLK_HIP(hipMemcpyAsync(d_links.ptr, h_links, sizeof(uint64_t) * link_words, hipMemcpyHostToDevice, s));
  const int32_t *d_first = d_links.as<int32_t>(), *d_partner = d_first + nc + 1;
  const DCurve *dcs = d_cs.as<DCurve>();
  unsigned long long *cnt = d_cnt.as<unsigned long long>();  // [0] overlaps, [1] too-small flag

  // live pieces (two generations) and retired pieces
  auto reserve_gen = [](DiscScratch::Gen &g, int64_t n) {
    g.c.reserve(sizeof(int32_t) * n);
    g.s.reserve(sizeof(int32_t) * n);
    g.lo.reserve(sizeof(double) * n);
    g.hi.reserve(sizeof(double) * n);
    g.box.reserve(sizeof(PBox) * n);
  };
  DiscScratch::Gen(&gen)[2] = D.gen;
  DiscScratch::Gen &ret = D.ret;
  // the retired list accumulates over rounds: grow it keeping its contents
  auto grow_kept = [&](DevBuf &b, size_t used, size_t need) {
    if (need <= b.bytes) return;
    DevBuf nb;
    nb.reserve(std::max(need, 2 * b.bytes));
    if (used) FLK_HIP(hipMemcpyAsync(nb.ptr, b.ptr, used, hipMemcpyDeviceToDevice, s));
    FLK_HIP(hipStreamSynchronize(s));
    b = std::move(nb);
  };
  auto grow_retired = [&](int64_t used, int64_t need) {
    grow_kept(ret.c, sizeof(int32_t) * used, sizeof(int32_t) * need);
    grow_kept(ret.s, sizeof(int32_t) * used, sizeof(int32_t) * need);
    grow_kept(ret.lo, sizeof(double) * used, sizeof(double) * need);
    grow_kept(ret.hi, sizeof(double) * used, sizeof(double) * need);
  };
  reserve_gen(gen[0], nseg);
  bool exact = false;  // `threshold` is the reference's to the bit
  double threshold;
  {
    const int64_t nb = blocks_for(nseg);
    D.diag.reserve(sizeof(double) * nseg);
    D.part.reserve(sizeof(InitPart) * nb);
    hipLaunchKernelGGL(disc_init, dim3((unsigned)nb), dim3(256), 0, s, q, dcs, nc, nseg, gen[0].c.as<int32_t>(),
                       gen[0].s.as<int32_t>(), gen[0].lo.as<double>(), gen[0].hi.as<double>(),
                       gen[0].box.as<PBox>(), D.diag.as<double>(), D.part.as<InitPart>());
    FLK_HIP(hipGetLastError());
    hipLaunchKernelGGL(disc_fold, dim3(1), dim3(1024), 0, s, (const InitPart *)D.part.as<InitPart>(), nb, h_part);
    FLK_HIP(hipGetLastError());
    FLK_HIP(hipStreamSynchronize(s));
    double md = h_part->md;
    int64_t mg = h_part->mg;
    const bool nan = h_part->nan != 0;
    threshold = threshold_of(h_part->sum) * (1 + kUnsure);
    // the reference's input guard, in its order (first smallest, NaN taken)
    if (nan) {
      std::vector<double> diag(nseg);
      FLK_HIP(hipMemcpyAsync(diag.data(), D.diag.ptr, sizeof(double) * nseg, hipMemcpyDeviceToHost, s));
      FLK_HIP(hipStreamSynchronize(s));
      md = std::numeric_limits<double>::infinity();
      mg = -1;
      for (int64_t g = 0; g < nseg; ++g)
        if (!(diag[g] >= md)) {
          md = diag[g];
          mg = g;
        }
    }
    if (!(md >= threshold)) {
      threshold = exact_threshold();
      exact = true;
    }
    if (!(md >= threshold)) {
      int c = 0;
      while (c + 1 < nc && cs[c + 1].seg0 <= mg) ++c;
      res.small_curve = c;
      res.small_segment = (int32_t)(mg - cs[c].seg0);
      res.small_size = md;
      throw Error(FLK_ERR_ARG, "Discretize: Smallest input segment is smaller than eps * avg coordinate. Consider "
                               "combining.");
    }
  }
  // a point of the model, for the tree's boxes: the first control point, or the
  // corner of its curve's box
  double3 origin = make_double3(0, 0, 0);
  {
    int32_t c = 0;
    while (cs[c].n == 0) ++c;  // nseg > 0
    const double *p = ctrl ? ctrl : ctx->curves.box.data() + 6 * (size_t)c;
    if (std::isfinite(p[0]) && std::isfinite(p[1]) && std::isfinite(p[2])) origin = make_double3(p[0], p[1], p[2]);
  }
  // the control points' box, for the sorted tree's keys
  double3 key_lo{}, key_cells{};
  if (sorted) {
    double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (int64_t k = 0; k < (ctrl ? nctrl : (int64_t)nc); ++k)
      for (int d = 0; d < 3; ++d) {
        const double *b = ctrl ? ctrl + 3 * k : ctx->curves.box.data() + 6 * k;
        lo[d] = std::min(lo[d], b[d]);
        hi[d] = std::max(hi[d], b[ctrl ? d : 3 + d]);
      }
    auto cells = [&](int d) { return hi[d] > lo[d] ? 1024.0 / (hi[d] - lo[d]) : 0.0; };
    key_lo = make_double3(lo[0], lo[1], lo[2]);
    key_cells = make_double3(cells(0), cells(1), cells(2));
  }
  int64_t n = nseg, nret = 0;
  int cur = 0;
  DevBuf &d_heap = D.heap, &d_hit = D.hit, &d_flag = D.flag, &d_scan = D.scan, &d_tmp = D.tmp;
  unsigned long long host_cnt[2] = {0, 0};
  for (int round = 0; round < 55; ++round) {
    DiscScratch::Gen &G = gen[cur];
    int64_t L = 1;
    while (L < n) L <<= 1;
    d_heap.reserve(sizeof(FBox) * 2 * L);
    const size_t range_bytes = sorted ? 0 : sizeof(int2) * (size_t)nc;  // before the marks: cleared together
    d_hit.reserve(range_bytes + n);
    int2 *range = d_hit.as<int2>();
    uint8_t *hit = d_hit.as<uint8_t>() + range_bytes;
    d_flag.reserve(sizeof(int32_t) * (n + 1));
    d_scan.reserve(sizeof(int32_t) * (n + 1));
    FBox *heap = d_heap.as<FBox>();
    FLK_HIP(hipMemsetAsync(d_hit.ptr, 0, range_bytes + n, s));
    FLK_HIP(hipMemsetAsync(cnt, 0, sizeof(unsigned long long) * 2, s));
    const uint32_t *order = nullptr;
    if (sorted) {
      for (DevBuf *b : {&D.k0, &D.k1, &D.i0, &D.i1, &D.i2}) b->reserve(sizeof(uint32_t) * n);
      d_tmp.reserve(std::max<size_t>(radix_temp_bytes(n), 16));
      hipLaunchKernelGGL(disc_morton, dim3(blocks_for(n)), dim3(256), 0, s, G.box.as<PBox>(), n, key_lo, key_cells,
                         D.k0.as<uint32_t>(), D.i0.as<uint32_t>());
      FLK_HIP(hipGetLastError());
      radix_sort_pairs<uint32_t>(D.k0.as<uint32_t>(), D.k1.as<uint32_t>(), D.i0.as<uint32_t>(), D.i1.as<uint32_t>(),
                                 D.i2.as<uint32_t>(), n, 30, d_tmp.ptr, s);
      order = D.i2.as<uint32_t>();
    }
    hipLaunchKernelGGL(disc_tree<true>, dim3(blocks_for(L)), dim3(256), 0, s, G.box.as<PBox>(), G.c.as<int32_t>(),
                       order, n, origin, L, heap, range);
    for (int64_t M = L / 256; M > 1; M /= 256)
      hipLaunchKernelGGL(disc_tree<false>, dim3(blocks_for(M)), dim3(256), 0, s, G.box.as<PBox>(),
                         G.c.as<int32_t>(), order, n, origin, M, heap, range);
    FLK_HIP(hipGetLastError());
    hipLaunchKernelGGL(sorted ? disc_query<true> : disc_query<false>, dim3(blocks_for(n)), dim3(256), 0, s, heap,
                       G.box.as<PBox>(), n, origin, L, G.c.as<int32_t>(), order, d_links.as<uint64_t>(),
                       (int64_t)lk.size(), range, d_first, d_partner, hit, cnt);
    FLK_HIP(hipGetLastError());
    // positions: scan of the marks (a trailing zero makes scan[n] the count)
    hipLaunchKernelGGL(disc_flags, dim3(blocks_for(n)), dim3(256), 0, s, hit, n,
                       d_flag.as<int32_t>());
    FLK_HIP(hipMemsetAsync(d_flag.as<int32_t>() + n, 0, sizeof(int32_t), s));
    d_tmp.reserve(scan_temp_bytes(n + 1));
    exclusive_scan(d_flag.as<int32_t>(), d_scan.as<int32_t>(), n + 1, d_tmp.as<int32_t>(), s);
    hipLaunchKernelGGL(disc_report, dim3(1), dim3(1), 0, s, cnt, d_scan.as<int32_t>() + n, h_report);
    FLK_HIP(hipGetLastError());
    FLK_HIP(hipStreamSynchronize(s));
    const int32_t nhit = (int32_t)h_report[1];
    host_cnt[0] = h_report[0];
    host_cnt[1] = 0;
    res.overlaps.push_back((int64_t)host_cnt[0]);
    // bisect the marked pieces, retire the rest
    DiscScratch::Gen &N = gen[cur ^ 1];
    reserve_gen(N, std::max<int64_t>(2 * (int64_t)nhit, 1));
    grow_retired(nret, std::max<int64_t>(nret + (n - nhit), 1));
    for (;;) {
      hipLaunchKernelGGL(disc_split, dim3(blocks_for(n)), dim3(256), 0, s, q, dcs, n, hit,
                         d_scan.as<int32_t>(), G.c.as<int32_t>(), G.s.as<int32_t>(), G.lo.as<double>(),
                         G.hi.as<double>(), N.c.as<int32_t>(), N.s.as<int32_t>(), N.lo.as<double>(),
                         N.hi.as<double>(), N.box.as<PBox>(), nret, ret.c.as<int32_t>(), ret.s.as<int32_t>(),
                         ret.lo.as<double>(), ret.hi.as<double>(), threshold, reinterpret_cast<int32_t *>(cnt + 1));
      FLK_HIP(hipGetLastError());
      host_cnt[1] = 0;
      if (nhit == 0) break;  // no new boxes
      FLK_HIP(hipMemcpyAsync(host_cnt + 1, cnt + 1, sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
      FLK_HIP(hipStreamSynchronize(s));
      if (host_cnt[1] == 0 || exact) break;
      // too small by the device's threshold: again with the reference's
      threshold = exact_threshold();
      exact = true;
      FLK_HIP(hipMemsetAsync(cnt + 1, 0, sizeof(unsigned long long), s));
    }
    nret += n - nhit;
    if (host_cnt[1] != 0)
      throw Error(FLK_ERR_ARG, "Discretize: Smallest segment is smaller than eps * avg coordinate. Perhaps curves "
                               "are too close.");
    if (host_cnt[0] == 0) break;
    n = 2 * (int64_t)nhit;
    cur ^= 1;
  }
  res.rounds = (int32_t)res.overlaps.size();
  if (res.overlaps.back() > 0)
    throw Error(FLK_ERR_ARG, "Reached max recursion (curves are too close) in Discretize().");

  // sort the retired pieces by (global segment, t_lo) and evaluate the vertices
  const int R = res.rounds;
  int gbits = 1;
  while (gbits < 32 && ((int64_t)1 << gbits) < nseg) ++gbits;
  DevBuf &d_k0 = D.k0, &d_k1 = D.k1, &d_i0 = D.i0, &d_i1 = D.i1, &d_i2 = D.i2, &d_open = D.open,
         &d_out = D.out, &d_per = D.per_curve;
  d_k0.reserve(sizeof(uint64_t) * nret);
  d_k1.reserve(sizeof(uint64_t) * nret);
  d_i0.reserve(sizeof(uint32_t) * nret);
  d_i1.reserve(sizeof(uint32_t) * nret);
  d_i2.reserve(sizeof(uint32_t) * nret);
  d_tmp.reserve(std::max<size_t>(radix_temp_bytes(nret), 16));
  d_per.reserve(sizeof(int32_t) * nc);
  FLK_HIP(hipMemsetAsync(d_per.ptr, 0, sizeof(int32_t) * nc, s));
  hipLaunchKernelGGL(disc_keys, dim3(blocks_for(nret)), dim3(256), 0, s, dcs, ret.c.as<int32_t>(),
                     ret.s.as<int32_t>(), ret.lo.as<double>(), nret, R, d_k0.as<uint64_t>(),
                     (R > 1 ? d_i0 : d_i1).as<uint32_t>(), d_per.as<int32_t>());
  FLK_HIP(hipGetLastError());
  // stable by t_lo (R bits), then stable by segment: d_i1 = the order.  After one
  // round nothing was split, and the pieces have retired in that order (17
  // launches, 230 us for 8.8e5 pieces).
  if (R > 1) {
    radix_sort_pairs<uint64_t>(d_k0.as<uint64_t>(), d_k1.as<uint64_t>(), d_i0.as<uint32_t>(), d_i1.as<uint32_t>(),
                               d_i2.as<uint32_t>(), nret, R, d_tmp.ptr, s);
    hipLaunchKernelGGL(disc_seg_keys, dim3(blocks_for(nret)), dim3(256), 0, s, dcs, ret.c.as<int32_t>(),
                       ret.s.as<int32_t>(), d_i2.as<uint32_t>(), nret, d_k0.as<uint32_t>());
    FLK_HIP(hipGetLastError());
    radix_sort_pairs<uint32_t>(d_k0.as<uint32_t>(), d_k1.as<uint32_t>(), d_i2.as<uint32_t>(), d_i0.as<uint32_t>(),
                               d_i1.as<uint32_t>(), nret, gbits, d_tmp.ptr, s);
  }
  FLK_HIP(hipMemcpyAsync(per_curve, d_per.ptr, sizeof(int32_t) * nc, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  int32_t opens = 0;
  res.out_offsets.assign(nc + 1, 0);
  for (int32_t c = 0; c < nc; ++c) {
    open_before[c] = opens;
    is_open[c] = (!looped[c] && per_curve[c] > 0) ? 1 : 0;
    opens += is_open[c];
    res.out_offsets[c + 1] = res.out_offsets[c] + per_curve[c] + is_open[c];
  }
  res.retired = nret;
  const int64_t nout = res.out_offsets[nc];
  d_open.reserve(sizeof(int32_t) * 2 * nc);
  d_out.reserve(sizeof(double) * 3 * std::max<int64_t>(nout, 1));
  FLK_HIP(hipMemcpyAsync(d_open.ptr, open_before, sizeof(int32_t) * 2 * nc, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(disc_points, dim3(blocks_for(nret)), dim3(256), 0, s, q, dcs, d_i1.as<int32_t>(),
                     ret.c.as<int32_t>(), ret.s.as<int32_t>(), ret.lo.as<double>(), ret.hi.as<double>(), nret,
                     d_open.as<int32_t>(), d_open.as<int32_t>() + nc, d_out.as<double>());
  FLK_HIP(hipGetLastError());
  if (host_copy) {
    res.xyz.resize(3 * nout);
    FLK_HIP(hipMemcpyAsync(res.xyz.data(), d_out.ptr, sizeof(double) * 3 * nout, hipMemcpyDeviceToHost, s));
  }
  FLK_HIP(hipStreamSynchronize(s));
  // install the polylines: the output array becomes the curve set's input
  // array (it holds 3 nout doubles, so the layout's reserve keeps it)
  std::swap(ctx->curves.raw, d_out);
  try {
    curves_layout(ctx, res.out_offsets.data(), nc);
    curves_finish(ctx);
  } catch (...) {
    curves_clear(ctx);
    throw;
  }
}

}  // namespace flk
