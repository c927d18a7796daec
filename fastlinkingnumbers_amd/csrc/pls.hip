// Curve boxes, vertex staging and the potential-link search (gfx950).
//
// Potential-link search (reference src/potential_link_search.cpp:88-127): all
// unordered curve pairs whose FP64 bounding boxes overlap as closed intervals.
// Up to kAllPairsCurves curves every pair is tested: the curves' boxes fit the
// caches, and counts, their prefix sum and a second sweep that writes put the
// pairs in ascending order without a sort.  Beyond that the device builds an
// implicit BVH over the curve boxes: boxes are sorted by
// the 30-bit Morton code of their centres, padded to a power of two, and the
// levels of a complete binary tree (heap layout, root = 1, children 2k and
// 2k+1) are unions of their children.  One thread per curve then walks the
// tree with a private stack (a wavefront of independent queries), appending
// every overlapping pair with a lower first index to a global list, which is
// radix-sorted into the reference's ascending order.  All box tests are FP64
// on the exact input boxes, so the pair set is exactly the reference's.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "flk_internal.h"

namespace flk {

namespace {

struct Box6 {
  double mn[3], mx[3];
};

__device__ __forceinline__ bool box_overlap(const Box6 &a, const Box6 &b) {
  return a.mn[0] <= b.mx[0] && a.mn[1] <= b.mx[1] && a.mn[2] <= b.mx[2] && b.mn[0] <= a.mx[0] &&
         b.mn[1] <= a.mx[1] && b.mn[2] <= a.mx[2];
}

// FP64 min/max of each curve's vertices (the polyline case of reference
// curve.cpp:331-343; an empty curve gets the empty box) in two passes: one
// block per chunk of at most kBoxChunk vertices of one curve, then one wave per
// curve folding its chunks (a thread took 115 us for 490 chunks), so a curve of millions of vertices is spread
// over the whole chip; where every curve is one chunk the first pass is all.
// The boxes also go to pinned memory (`host`) without a copy, and the last pass
// clears the flag that stage_vertices sets.
constexpr int64_t kBoxChunk = 4096;

// Coordinates that came as FP32 are read there and written to xyz as FP64 on the
// way (a pass of its own read and wrote them again: 215 us for 3.1e7 vertices).
// A block of 1,024 threads with four vertices each in flight: for a few curves of
// thousands of vertices the pass is as long as one chunk.  Launching such a block
// takes 14 ns, so for more than kManyChunks chunks it has as many threads as a
// chunk has fours on average, in quarters: 200,000 curves of 16 vertices 2,887 ->
// 370 us, 20,000 of 400 302 -> 79, 3,000 of 100 53 -> 11, 1,100 of 900 28 -> 16.
constexpr int64_t kManyChunks = 1024;
template <bool LANDED, int THREADS>
__global__ __launch_bounds__(THREADS) void curve_box_chunks(double *__restrict__ xyz, const float *__restrict__ land,
                                                        const int64_t *__restrict__ chunk_v,
                                                        double *__restrict__ part, double *__restrict__ host,
                                                        int32_t *__restrict__ inexact) {
  const int64_t c = blockIdx.x;
  if (host && c == 0 && threadIdx.x == 0) *inexact = 0;
  const int64_t v0 = chunk_v[2 * c], v1 = chunk_v[2 * c + 1];
  double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (int64_t base = v0 + threadIdx.x; base < v1; base += 4 * THREADS) {
    double x[4][3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t v = min(base + THREADS * k, v1 - 1);  // the last again past the end
#pragma unroll
      for (int d = 0; d < 3; ++d) x[k][d] = LANDED ? (double)land[3 * v + d] : xyz[3 * v + d];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        if (LANDED && base + THREADS * k < v1) xyz[3 * (base + THREADS * k) + d] = x[k][d];
        mn[d] = fmin(mn[d], x[k][d]);
        mx[d] = fmax(mx[d], x[k][d]);
      }
  }
  __shared__ double smn[3][THREADS / 64], smx[3][THREADS / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    for (int o = 32; o > 0; o >>= 1) {
      mn[d] = fmin(mn[d], __shfl_xor(mn[d], o, 64));
      mx[d] = fmax(mx[d], __shfl_xor(mx[d], o, 64));
    }
    if (lane == 0) {
      smn[d][w] = mn[d];
      smx[d][w] = mx[d];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int d = 0; d < 3; ++d) {
      double lo = smn[d][0], hi = smx[d][0];
      for (int k = 1; k < THREADS / 64; ++k) {
        lo = fmin(lo, smn[d][k]);
        hi = fmax(hi, smx[d][k]);
      }
      part[6 * c + d] = lo;
      part[6 * c + 3 + d] = hi;
      if (host) {
        host[6 * c + d] = lo;
        host[6 * c + 3 + d] = hi;
      }
    }
  }
}

__global__ __launch_bounds__(256) void curve_box_merge(const double *__restrict__ part,
                                                       const int64_t *__restrict__ coff, int32_t ncurves,
                                                       double *__restrict__ boxes, double *__restrict__ host,
                                                       int32_t *__restrict__ inexact) {
  const int c = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
  if (c == 0 && lane == 0) *inexact = 0;
  if (c >= ncurves) return;
  double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (int64_t k = coff[c] + lane; k < coff[c + 1]; k += 64)
    for (int d = 0; d < 3; ++d) {
      mn[d] = fmin(mn[d], part[6 * k + d]);
      mx[d] = fmax(mx[d], part[6 * k + 3 + d]);
    }
#pragma unroll
  for (int d = 0; d < 3; ++d)
    for (int o = 32; o > 0; o >>= 1) {
      mn[d] = fmin(mn[d], __shfl_xor(mn[d], o, 64));
      mx[d] = fmax(mx[d], __shfl_xor(mx[d], o, 64));
    }
  if (lane) return;
  for (int d = 0; d < 3; ++d) {
    boxes[6 * c + d] = host[6 * c + d] = mn[d];
    boxes[6 * c + 3 + d] = host[6 * c + 3 + d] = mx[d];
  }
}

// Device vertex v (curve c, local index l <= n_c) takes input vertex l, or
// vertex 0 for the closing copy l == n_c; coordinates are (x - origin) * scale.
// Beside the FP64 vertex go its FP32 hi/lo split and the FP32 edge to the next
// vertex of the array (the FP64 difference rounded, with -|edge|^2 / 2), and
// with a curve's first vertex the scaled diagonal of its box; any
// vertex that FP32 cannot hold sets the flag.  One pass instead of a second over
// the FP64 vertices: 3.1e7 vertices took 523 + 433 us in two.
__global__ __launch_bounds__(256) void stage_vertices(const double *__restrict__ xyz,
                                                      const int64_t *__restrict__ in_off,
                                                      const int64_t *__restrict__ dev_off,
                                                      const double *__restrict__ boxes,
                                                      int32_t ncurves, int64_t ndev, double ox,
                                                      double oy, double oz, double scale,
                                                      double4 *__restrict__ out, float4 *__restrict__ hi,
                                                      float4 *__restrict__ lo, float4 *__restrict__ ed,
                                                      int32_t *__restrict__ inexact,
                                                      int32_t *__restrict__ inexact_host) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool bad = false;
  if (v < ndev) {
    int c = 0, end = ncurves;  // last c with dev_off[c] <= v
    while (end - c > 1) {
      const int mid = (c + end) >> 1;
      if (dev_off[mid] <= v) c = mid;
      else end = mid;
    }
    auto staged = [&](int k, int64_t l) {  // vertex l of curve k, (0, 0, 0) for an empty one
      const int64_t first = in_off[k], n = in_off[k + 1] - first;
      if (n == 0) return make_double4(0, 0, 0, 0);
      const double *p = xyz + 3 * (first + (l < n ? l : 0));
      return make_double4((p[0] - ox) * scale, (p[1] - oy) * scale, (p[2] - oz) * scale, 0.0);
    };
    const int64_t l = v - dev_off[c];
    double4 p = staged(c, l);
    if (l == 0 && in_off[c + 1] > in_off[c]) {
      const double *b = boxes + 6 * (int64_t)c;
      const double dx = (b[3] - b[0]) * scale, dy = (b[4] - b[1]) * scale, dz = (b[5] - b[2]) * scale;
      p.w = sqrt(dx * dx + dy * dy + dz * dz);
    }
    out[v] = p;
    const float hx = (float)p.x, hy = (float)p.y, hz = (float)p.z;
    const float lx = (float)(p.x - (double)hx), ly = (float)(p.y - (double)hy), lz = (float)(p.z - (double)hz);
    hi[v] = make_float4(hx, hy, hz, 0.f);
    lo[v] = make_float4(lx, ly, lz, 0.f);
    bad = (lx != 0.f) || (ly != 0.f) || (lz != 0.f);
    if (v + 1 < ndev) {
      const double4 q = v + 1 < dev_off[c + 1] ? staged(c, l + 1) : staged(c + 1, 0);
      const double ex = q.x - p.x, ey = q.y - p.y, ez = q.z - p.z;
      ed[v] = make_float4((float)ex, (float)ey, (float)ez, (float)(-0.5 * (ex * ex + ey * ey + ez * ez)));
    } else {
      ed[v] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  // Plain stores by the blocks that read the flag clear (writers agree, and a
  // stale read costs another store): an atomic for every wave serialises on its
  // address, 180 us for the 8.8e5 vertices of a discretized knit.
  if (__syncthreads_or(bad) && threadIdx.x == 0 &&
      __hip_atomic_load(inexact, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) {
    __hip_atomic_store(inexact, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    *inexact_host = 1;
  }
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v = (v * 0x00010001u) & 0xFF0000FFu;
  v = (v * 0x00000101u) & 0x0F00F00Fu;
  v = (v * 0x00000011u) & 0xC30C30C3u;
  v = (v * 0x00000005u) & 0x49249249u;
  return v;
}

__global__ __launch_bounds__(256) void morton_keys(const double *__restrict__ boxes, int32_t n,
                                                   double lx, double ly, double lz, double ix,
                                                   double iy, double iz,
                                                   uint32_t *__restrict__ keys,
                                                   int32_t *__restrict__ ids) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *b = boxes + 6 * (int64_t)i;
  uint32_t k = 0;
  if (b[0] <= b[3]) {  // non-empty
    const double c[3] = {0.5 * (b[0] + b[3]), 0.5 * (b[1] + b[4]), 0.5 * (b[2] + b[5])};
    const double lo[3] = {lx, ly, lz}, inv[3] = {ix, iy, iz};
    uint32_t q[3];
    for (int d = 0; d < 3; ++d) {
      double u = (c[d] - lo[d]) * inv[d];
      u = fmin(fmax(u, 0.0), 1.0);
      q[d] = (uint32_t)fmin(u * 1024.0, 1023.0);
    }
    k = (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
  }
  keys[i] = k;
  ids[i] = i;
}

// Heap slot L + i holds the box of the i-th curve in Morton order (empty
// boxes pad to a power of two).
__global__ __launch_bounds__(256) void bvh_leaves(const double *__restrict__ boxes,
                                                  const int32_t *__restrict__ order, int32_t n,
                                                  int32_t L, Box6 *__restrict__ heap) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= L) return;
  Box6 b;
  if (i < n) {
    const double *s = boxes + 6 * (int64_t)order[i];
    for (int d = 0; d < 3; ++d) {
      b.mn[d] = s[d];
      b.mx[d] = s[3 + d];
    }
  } else {
    for (int d = 0; d < 3; ++d) {
      b.mn[d] = DBL_MAX;
      b.mx[d] = -DBL_MAX;
    }
  }
  heap[L + i] = b;
}

__global__ __launch_bounds__(256) void bvh_level(Box6 *__restrict__ heap, int32_t first,
                                                 int32_t count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int k = first + i;
  const Box6 a = heap[2 * k], b = heap[2 * k + 1];
  Box6 u;
  for (int d = 0; d < 3; ++d) {
    u.mn[d] = fmin(a.mn[d], b.mn[d]);
    u.mx[d] = fmax(a.mx[d], b.mx[d]);
  }
  heap[k] = u;
}

// One query per curve (Morton position i): stack walk of the heap, append
// (min id, max id) for every overlap whose partner has a larger curve id.
__global__ __launch_bounds__(256) void bvh_query(const Box6 *__restrict__ heap,
                                                 const int32_t *__restrict__ order, int32_t n,
                                                 int32_t L, int64_t cap,
                                                 unsigned long long *__restrict__ count,
                                                 uint64_t *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Box6 q = heap[L + i];
  const int32_t me = order[i];
  int stack[64];
  int sp = 0;
  stack[sp++] = 1;
  while (sp > 0) {
    const int k = stack[--sp];
    if (!box_overlap(heap[k], q)) continue;
    if (k >= L) {
      const int j = k - L;
      if (j < n) {
        const int32_t other = order[j];
        if (other > me) {
          const unsigned long long slot = atomicAdd(count, 1ull);
          if ((int64_t)slot < cap) out[slot] = ((uint64_t)(uint32_t)me << 32) | (uint32_t)other;
        }
      }
    } else if (sp + 2 <= 64) {
      stack[sp++] = 2 * k + 1;
      stack[sp++] = 2 * k;
    }
  }
}

// Every pair of curves tested.  A wave takes kRowsPerWave rows (curves i) and
// one chunk of kColChunk columns (curves j > i), 64 columns a step; a cell is
// one row's part in one chunk.  Counting: cells[i * chunks + chunk] receives
// the cell's overlaps.  Writing: cells holds their exclusive prefix sum, and
// the pairs go to their places, which are ascending in (i, j), straight into
// the caller's pinned memory (slots past cap are dropped, the host sees the
// total).  Bound by latency for the sizes at hand: 16 steps a wave, each six
// 8-byte loads from the caches for kRowsPerWave tests.
constexpr int kRowsPerWave = 4;
constexpr int kColChunk = 1024;
template <bool kWrite>
__global__ __launch_bounds__(256) void pls_all_pairs(const double *__restrict__ boxes, int32_t n, int32_t chunks,
                                                     int32_t *__restrict__ cells, int64_t cap,
                                                     int2 *__restrict__ out, int64_t *__restrict__ total) {
  const int lane = threadIdx.x & 63;
  const int i0 = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)) * kRowsPerWave;
  const int c0 = (int)blockIdx.y * kColChunk;
  if (kWrite && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *total = cells[(int64_t)n * chunks];
  if (!kWrite && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) cells[(int64_t)n * chunks] = 0;
  if (i0 >= n) return;
  Box6 row[kRowsPerWave];
  int cnt[kRowsPerWave];
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const double *b = boxes + 6 * (int64_t)min(i0 + r, n - 1);
    for (int d = 0; d < 3; ++d) {
      row[r].mn[d] = b[d];
      row[r].mx[d] = b[3 + d];
    }
    cnt[r] = kWrite && i0 + r < n ? cells[(int64_t)(i0 + r) * chunks + blockIdx.y] : 0;
  }
  const int end = min(n, c0 + kColChunk);
  // from the 64-column step that holds the first column past row i0
  for (int j0 = max(c0, c0 + (i0 + 1 - c0) / 64 * 64); j0 < end; j0 += 64) {
    const int j = j0 + lane;
    const double *b = boxes + 6 * (int64_t)min(j, n - 1);
    Box6 q;
    for (int d = 0; d < 3; ++d) {
      q.mn[d] = b[d];
      q.mx[d] = b[3 + d];
    }
#pragma unroll
    for (int r = 0; r < kRowsPerWave; ++r) {
      const int i = i0 + r;
      const bool hit = j < end && j > i && i < n && box_overlap(row[r], q);
      const unsigned long long m = __ballot(hit);
      if (kWrite && hit) {
        const int64_t slot = (int64_t)cnt[r] + __popcll(m & ((1ull << lane) - 1ull));
        if (slot < cap) out[slot] = make_int2(i, j);
      }
      cnt[r] += __popcll(m);
    }
  }
  if (!kWrite && lane < kRowsPerWave && i0 + lane < n) {
    int v = cnt[0];
#pragma unroll
    for (int r = 1; r < kRowsPerWave; ++r) v = lane == r ? cnt[r] : v;
    cells[(int64_t)(i0 + lane) * chunks + blockIdx.y] = v;
  }
}

// Most curves of the all-pairs search.  Whole calls on lattices of four pairs a
// curve, the tree (with its two library sorts, an allocation per array and one
// atomic per pair) against all pairs: 137 and 25 us for 10 curves, 270 and 44
// for 400, 393 and 77 for 1,600, 587 and 237 for 10,000, 727 and 250 for
// 16,384, 1,052 and 636 for 30,000; the sweep grows with the square.  With a pair
// for every four curves the two meet at 28,000 (537 and 530 us; 32,000: 546 and 658), with
// two pairs a curve all pairs are ahead at 32,000 still (979 and 665).
constexpr int32_t kAllPairsCurves = 32768;

// Up to kOneBlockCurves curves in one launch: the boxes in LDS, a row a wave at a
// time, counted and, after a scan of the rows' counts, written.  For ten curves
// the three launches were most of the call.
constexpr int32_t kOneBlockCurves = 256;
__global__ __launch_bounds__(1024) void pls_one_block(const double *__restrict__ boxes, int32_t n, int64_t cap,
                                                      int2 *__restrict__ out, int64_t *__restrict__ total) {
  __shared__ double box[6][kOneBlockCurves];
  __shared__ int first[kOneBlockCurves];
  __shared__ int sum[kOneBlockCurves / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, waves = (int)(blockDim.x >> 6);
  for (int t = threadIdx.x; t < 6 * n; t += (int)blockDim.x) box[t % 6][t / 6] = boxes[t];
  __syncthreads();
  auto row = [&](int i, auto found) {  // found(mask of the overlaps from column j0)
    Box6 a;
    for (int d = 0; d < 3; ++d) {
      a.mn[d] = box[d][i];
      a.mx[d] = box[3 + d][i];
    }
    for (int j0 = (i + 1) / 64 * 64; j0 < n; j0 += 64) {
      const int j = j0 + lane;
      Box6 b;
      for (int d = 0; d < 3; ++d) {
        b.mn[d] = box[d][min(j, n - 1)];
        b.mx[d] = box[3 + d][min(j, n - 1)];
      }
      found(j0, __ballot(j > i && j < n && box_overlap(a, b)));
    }
  };
  for (int i = w; i < n; i += waves) {
    int cnt = 0;
    row(i, [&](int, uint64_t m) { cnt += __popcll(m); });
    if (lane == 0) first[i] = cnt;
  }
  __syncthreads();
  int mine = 0, inc = 0;  // the rows' counts, scanned
  if (threadIdx.x < kOneBlockCurves) {
    mine = inc = (int)threadIdx.x < n ? first[threadIdx.x] : 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = __shfl_up(inc, d, 64);
      if (lane >= d) inc += u;
    }
    if (lane == 63) sum[w] = inc;
  }
  __syncthreads();
  if (threadIdx.x < kOneBlockCurves) {
    for (int k = 0; k < w; ++k) inc += sum[k];
    first[threadIdx.x] = inc - mine;
    if (threadIdx.x == kOneBlockCurves - 1) *total = inc;
  }
  __syncthreads();
  for (int i = w; i < n; i += waves) {
    int at = first[i];
    row(i, [&](int j0, uint64_t m) {
      const int slot = at + __popcll(m & ((1ull << lane) - 1ull));
      if (((m >> lane) & 1ull) && slot < cap) out[slot] = make_int2(i, j0 + lane);
      at += __popcll(m);
    });
  }
}

// Pinned memory of the search that a call may leave behind.
constexpr size_t kKeptPinned = size_t(64) << 20;

void pls_small(flk_ctx *ctx, const double *d_boxes, int32_t n, std::vector<int32_t> &out) {
  hipStream_t s = ctx->stream;
  const bool one = n <= kOneBlockCurves;
  const int32_t chunks = (n + kColChunk - 1) / kColChunk;
  const int64_t ncells = (int64_t)n * chunks;
  const dim3 grid((unsigned)((n + 4 * kRowsPerWave - 1) / (4 * kRowsPerWave)), (unsigned)chunks);
  int32_t *cells = nullptr;
  if (!one) {
    ctx->d_pls.reserve(sizeof(int32_t) * (ncells + 1) + scan_temp_bytes(ncells + 1));
    cells = ctx->d_pls.as<int32_t>();
    hipLaunchKernelGGL(pls_all_pairs<false>, grid, dim3(256), 0, s, d_boxes, n, chunks, cells, (int64_t)0,
                       (int2 *)nullptr, (int64_t *)nullptr);
    FLK_HIP(hipGetLastError());
    exclusive_scan(cells, cells, ncells + 1, cells + ncells + 1, s);
  }
  // the pairs land in pinned memory behind their total; a second sweep only
  // when there are more than eight pairs a curve (and than ever before)
  int64_t cap = std::max<int64_t>(1024, 8 * (int64_t)n);
  for (;;) {
    ctx->pls_host.reserve(sizeof(int64_t) * (1 + cap));
    cap = (int64_t)(ctx->pls_host.bytes / sizeof(int64_t)) - 1;
    int64_t *total = ctx->pls_host.as<int64_t>();
    int2 *pairs = reinterpret_cast<int2 *>(total + 1);
    if (one)
      hipLaunchKernelGGL(pls_one_block, dim3(1), dim3(1024), 0, s, d_boxes, n, cap, pairs, total);
    else
      hipLaunchKernelGGL(pls_all_pairs<true>, grid, dim3(256), 0, s, d_boxes, n, chunks, cells, cap, pairs, total);
    FLK_HIP(hipGetLastError());
    FLK_HIP(hipStreamSynchronize(s));
    if (*total <= cap) {
      const int32_t *p = reinterpret_cast<const int32_t *>(pairs);
      out.assign(p, p + 2 * *total);
      if (ctx->pls_host.bytes > kKeptPinned) ctx->pls_host.release();
      return;
    }
    cap = *total;
  }
}

}  // namespace

void curve_boxes_run(flk_ctx *ctx, std::vector<double> &boxes, const float *land) {
  Curves &cv = ctx->curves;
  const size_t nc = (size_t)cv.ncurves;
  boxes.assign(6 * nc, 0.0);
  if (nc == 0) return;
  // input and device offsets, the chunk table ((first, end) vertex of every
  // chunk) and each curve's chunks, in pinned memory on their way to the device
  int64_t nchunks = 0;
  for (size_t c = 0; c < nc; ++c) nchunks += (cv.in_off[c + 1] - cv.in_off[c] + kBoxChunk - 1) / kBoxChunk;
  bool single = nchunks <= (int64_t)nc;  // then empty curves have a chunk too
  for (size_t c = 0; single && c < nc; ++c) single = cv.in_off[c + 1] - cv.in_off[c] <= kBoxChunk;
  if (single) nchunks = (int64_t)nc;
  const size_t words = 3 * (nc + 1) + 2 * (size_t)nchunks;
  ctx->curve_host.reserve(sizeof(int64_t) * words + sizeof(double) * 6 * nc + sizeof(int32_t));
  int64_t *meta = ctx->curve_host.as<int64_t>();
  double *host = reinterpret_cast<double *>(meta + words);
  ctx->inexact_host = reinterpret_cast<int32_t *>(host + 6 * nc);
  *ctx->inexact_host = 0;
  std::copy(cv.in_off.begin(), cv.in_off.end(), meta);
  std::copy(cv.off.begin(), cv.off.end(), meta + nc + 1);
  int64_t *coff = meta + 2 * (nc + 1), *chunk = coff + nc + 1, k = 0;
  for (size_t c = 0; c < nc; ++c) {
    coff[c] = k;
    int64_t v = cv.in_off[c];
    const int64_t end = cv.in_off[c + 1];
    if (single && v == end) {
      chunk[2 * k] = chunk[2 * k + 1] = v;
      ++k;
    }
    for (; v < end; v += kBoxChunk, ++k) {
      chunk[2 * k] = v;
      chunk[2 * k + 1] = std::min(v + kBoxChunk, end);
    }
  }
  coff[nc] = nchunks;
  hipStream_t s = ctx->stream;
  ctx->d_boxes.reserve(sizeof(double) * 6 * (nc + std::max<int64_t>(nchunks, 1)));
  ctx->d_misc.reserve(sizeof(int64_t) * words);
  ctx->d_count.reserve(sizeof(int32_t));
  FLK_HIP(hipMemcpyAsync(ctx->d_misc.ptr, meta, sizeof(int64_t) * words, hipMemcpyHostToDevice, s));
  double *d_boxes = ctx->d_boxes.as<double>(), *d_part = d_boxes + 6 * nc;
  const int64_t *d_coff = ctx->d_misc.as<int64_t>() + 2 * (nc + 1), *d_chunk = d_coff + nc + 1;
  int32_t *flag = ctx->d_count.as<int32_t>();
  if (nchunks > 0) {
    const int64_t mean = nchunks > kManyChunks ? cv.in_off[nc] / nchunks : kBoxChunk;
    const auto pass = mean <= 256    ? (land ? curve_box_chunks<true, 64> : curve_box_chunks<false, 64>)
                      : mean <= 1024 ? (land ? curve_box_chunks<true, 256> : curve_box_chunks<false, 256>)
                                     : (land ? curve_box_chunks<true, 1024> : curve_box_chunks<false, 1024>);
    hipLaunchKernelGGL(pass,
                       dim3((unsigned)nchunks), dim3(mean <= 256 ? 64 : mean <= 1024 ? 256 : 1024), 0, s, cv.raw.as<double>(), land, d_chunk,
                       single ? d_boxes : d_part, single ? host : (double *)nullptr, flag);
  }
  if (!single)
    hipLaunchKernelGGL(curve_box_merge, dim3((unsigned)((nc + 3) / 4)), dim3(256), 0, s, d_part, d_coff,
                       cv.ncurves, d_boxes, host, flag);
  FLK_HIP(hipGetLastError());
  FLK_HIP(hipStreamSynchronize(s));
  boxes.assign(host, host + 6 * nc);
}

bool stage_vertices_run(flk_ctx *ctx) {
  Curves &cv = ctx->curves;
  const int64_t blocks = (cv.nvert_dev + 255) / 256;
  const int64_t *d_in = ctx->d_misc.as<int64_t>();
  hipLaunchKernelGGL(stage_vertices, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, cv.raw.as<double>(), d_in,
                     d_in + cv.ncurves + 1, ctx->d_boxes.as<double>(), cv.ncurves, cv.nvert_dev, cv.origin[0], cv.origin[1], cv.origin[2],
                     cv.scale, cv.dpts.as<double4>(), cv.hi.as<float4>(), cv.lo.as<float4>(), cv.ed.as<float4>(),
                     ctx->d_count.as<int32_t>(), ctx->inexact_host);
  FLK_HIP(hipGetLastError());
  FLK_HIP(hipStreamSynchronize(ctx->stream));
  return *ctx->inexact_host != 0;
}

void pls_run(flk_ctx *ctx, const double *boxes, int32_t n, std::vector<int32_t> &out) {
  out.clear();
  if (n < 2) return;
  hipStream_t s = ctx->stream;
  if (n <= kAllPairsCurves) {
    // the uploaded curves' boxes are on the device already
    const double *d_boxes = ctx->d_boxes.as<double>();
    if (boxes != ctx->curves.box.data()) {
      ctx->d_pls_boxes.reserve(sizeof(double) * 6 * (size_t)n);
      FLK_HIP(hipMemcpyAsync(ctx->d_pls_boxes.ptr, boxes, sizeof(double) * 6 * (size_t)n, hipMemcpyHostToDevice, s));
      d_boxes = ctx->d_pls_boxes.as<double>();
    }
    pls_small(ctx, d_boxes, n, out);
    return;
  }
  int32_t L = 1;
  while (L < n) L <<= 1;
  // device scratch layout inside d_pls
  const size_t sz_boxes = sizeof(double) * 6 * (size_t)n;
  const size_t sz_keys = sizeof(uint32_t) * (size_t)n;
  const size_t sz_ids = sizeof(int32_t) * (size_t)n;
  const size_t sz_heap = sizeof(Box6) * 2 * (size_t)L;
  DevBuf d_b, d_k0, d_k1, d_i0, d_i1, d_heap, d_cnt, d_out, d_out2, d_tmp;
  d_b.reserve(sz_boxes);
  d_k0.reserve(sz_keys);
  d_k1.reserve(sz_keys);
  d_i0.reserve(sz_ids);
  d_i1.reserve(sz_ids);
  d_heap.reserve(sz_heap);
  d_cnt.reserve(sizeof(unsigned long long));
  struct Guard {
    DevBuf *b[10];
    ~Guard() {
      for (auto *p : b) p->release();
    }
  } guard{{&d_b, &d_k0, &d_k1, &d_i0, &d_i1, &d_heap, &d_cnt, &d_out, &d_out2, &d_tmp}};
  FLK_HIP(hipMemcpyAsync(d_b.ptr, boxes, sz_boxes, hipMemcpyHostToDevice, s));
  // model box for Morton normalisation
  double lo[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, hi[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
  for (int32_t i = 0; i < n; ++i)
    if (boxes[6 * i] <= boxes[6 * i + 3])
      for (int d = 0; d < 3; ++d) {
        lo[d] = std::min(lo[d], 0.5 * (boxes[6 * i + d] + boxes[6 * i + 3 + d]));
        hi[d] = std::max(hi[d], 0.5 * (boxes[6 * i + d] + boxes[6 * i + 3 + d]));
      }
  double inv[3];
  for (int d = 0; d < 3; ++d) inv[d] = (hi[d] > lo[d]) ? 1.0 / (hi[d] - lo[d]) : 0.0;
  if (!(lo[0] <= hi[0])) lo[0] = lo[1] = lo[2] = 0.0;
  const unsigned nb = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(morton_keys, dim3(nb), dim3(256), 0, s, d_b.as<double>(), n, lo[0], lo[1],
                     lo[2], inv[0], inv[1], inv[2], d_k0.as<uint32_t>(), d_i0.as<int32_t>());
  FLK_HIP(hipGetLastError());
  size_t tmp_bytes = 0;
  FLK_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, d_k0.as<uint32_t>(),
                                             d_k1.as<uint32_t>(), d_i0.as<int32_t>(),
                                             d_i1.as<int32_t>(), n, 0, 30, s));
  d_tmp.reserve(std::max<size_t>(tmp_bytes, 16));
  FLK_HIP(hipcub::DeviceRadixSort::SortPairs(d_tmp.ptr, tmp_bytes, d_k0.as<uint32_t>(),
                                             d_k1.as<uint32_t>(), d_i0.as<int32_t>(),
                                             d_i1.as<int32_t>(), n, 0, 30, s));
  const int32_t *order = d_i1.as<int32_t>();
  hipLaunchKernelGGL(bvh_leaves, dim3((unsigned)((L + 255) / 256)), dim3(256), 0, s,
                     d_b.as<double>(), order, n, L, d_heap.as<Box6>());
  FLK_HIP(hipGetLastError());
  for (int32_t first = L / 2; first >= 1; first /= 2) {
    hipLaunchKernelGGL(bvh_level, dim3((unsigned)((first + 255) / 256)), dim3(256), 0, s,
                       d_heap.as<Box6>(), first, first);
    FLK_HIP(hipGetLastError());
  }
  // query: first pass with a guessed capacity, second pass if it overflowed
  int64_t cap = std::max<int64_t>(1024, 8 * (int64_t)n);
  unsigned long long cnt = 0;
  for (int attempt = 0; attempt < 2; ++attempt) {
    d_out.reserve(sizeof(uint64_t) * cap);
    FLK_HIP(hipMemsetAsync(d_cnt.ptr, 0, sizeof(unsigned long long), s));
    hipLaunchKernelGGL(bvh_query, dim3(nb), dim3(256), 0, s, d_heap.as<Box6>(), order, n, L, cap,
                       d_cnt.as<unsigned long long>(), d_out.as<uint64_t>());
    FLK_HIP(hipGetLastError());
    FLK_HIP(hipMemcpyAsync(&cnt, d_cnt.ptr, sizeof(cnt), hipMemcpyDeviceToHost, s));
    FLK_HIP(hipStreamSynchronize(s));
    if ((int64_t)cnt <= cap) break;
    cap = (int64_t)cnt;
  }
  const int64_t m = (int64_t)cnt;
  if (m == 0) return;
  d_out2.reserve(sizeof(uint64_t) * m);
  tmp_bytes = 0;
  FLK_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tmp_bytes, d_out.as<uint64_t>(),
                                            d_out2.as<uint64_t>(), (int)m, 0, 64, s));
  d_tmp.reserve(std::max<size_t>(tmp_bytes, 16));
  FLK_HIP(hipcub::DeviceRadixSort::SortKeys(d_tmp.ptr, tmp_bytes, d_out.as<uint64_t>(),
                                            d_out2.as<uint64_t>(), (int)m, 0, 64, s));
  std::vector<uint64_t> h(m);
  FLK_HIP(hipMemcpyAsync(h.data(), d_out2.ptr, sizeof(uint64_t) * m, hipMemcpyDeviceToHost, s));
  FLK_HIP(hipStreamSynchronize(s));
  out.resize(2 * m);
  for (int64_t k = 0; k < m; ++k) {
    out[2 * k] = (int32_t)(h[k] >> 32);
    out[2 * k + 1] = (int32_t)(h[k] & 0xffffffffu);
  }
}

}  // namespace flk
