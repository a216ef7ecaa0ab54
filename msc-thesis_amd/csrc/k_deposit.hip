// k_deposit.hip -- charge deposit of a caller's particles in any order (pic_op_deposit;
// thesisCode/collisionless/double/src/pic.cu:99-138) into int64 fixed-point node sums.
//
// The device executes about 24e9 scattered 8-byte atomic adds per second on global memory,
// whatever the number of addresses, which bounded a deposit of four (FP64: eight) of them
// per particle: 1.36 ms for 8,000,009 FP32 particles on 512^2.  The sums are integers, so the
// particles can go in any order, and three forms give the same bits (8,000,009 FP32 particles
// in random order on 512^2: 15.7 + 4.7 + 35.8 + 22.8 us in the last; whole call 1427 -> 89):
//   direct   four global atomics per particle
//   grid     each workgroup sums its share in an LDS copy of the whole grid, then adds the
//            copy's non-zero words to the global one
//   binned   positions grouped by tiles of the grid (tile counts, their scan, one pass that
//            moves each position once), then equal slices of that order are summed in LDS
//            windows of a tile: bound by HBM (each position read three times, written once)
// deposit_plan picks one; the measurements behind its lines are there.
#include <algorithm>
#include <type_traits>
#include "deposit.h"
#include "launch.h"

namespace {

#define DEP_NT 512                  // threads per workgroup
#define DEP_MAX_TILES 1024
#define DEP_LDS_GRID (128 * 1024)   // largest LDS grid copy (of the CU's 160 KB)
#define DEP_LDS_WIN (72 * 1024)     // largest tile window: two workgroups per CU

template <typename R>
using DepPair = typename std::conditional<sizeof(R) == 4, float2, double2>::type;

template <typename R>
__device__ __forceinline__ void lds_add(unsigned long long* hi, unsigned long long* lo, int i,
                                        long long w) {
  if (sizeof(R) == 8) {
    atomicAdd(&hi[i], (unsigned long long)(w >> 30));
    atomicAdd(&lo[i], (unsigned long long)(w & ((1ll << 30) - 1)));
  } else {
    atomicAdd(&hi[i], (unsigned long long)w);
  }
}

template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_dep_direct(const R* __restrict__ x,
                                                       const R* __restrict__ y, int64_t n,
                                                       int nx, int ny, double lx, double ly,
                                                       unsigned long long* hi,
                                                       unsigned long long* lo) {
  const Geo<R> g = make_geo<R>(nx, ny, lx, ly);
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * PIC_WG) {
    int cx, cy;
    long long w[4];
    deposit_weights<R>(x[p], y[p], g, cx, cy, w);
    deposit_global<R>(hi, lo, cx, cy, w, g);
  }
}

// the whole grid in LDS; four positions per thread loaded together (past the end: the last)
template <typename R>
__global__ __launch_bounds__(DEP_NT) void k_dep_grid(const R* __restrict__ x,
                                                     const R* __restrict__ y, int64_t n, int nx,
                                                     int ny, double lx, double ly,
                                                     unsigned long long* hi,
                                                     unsigned long long* lo) {
  extern __shared__ unsigned long long sums[];
  constexpr int U = 4, NQ = (sizeof(R) == 8) ? 2 : 1;
  const Geo<R> g = make_geo<R>(nx, ny, lx, ly);
  const int G = nx * ny;
  unsigned long long *shi = sums, *slo = sums + G;
  for (int i = threadIdx.x; i < NQ * G; i += DEP_NT) sums[i] = 0ull;
  __syncthreads();
  const int64_t stride = (int64_t)gridDim.x * DEP_NT;
  for (int64_t p0 = blockIdx.x * (int64_t)DEP_NT + threadIdx.x; p0 < n; p0 += U * stride) {
    R xv[U], yv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t p = p0 + u * stride;
      const int64_t pl = p < n ? p : n - 1;
      xv[u] = x[pl];
      yv[u] = y[pl];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (p0 + u * stride >= n) continue;
      int cx, cy;
      long long w[4];
      deposit_weights<R>(xv[u], yv[u], g, cx, cy, w);
      const int cxp = pwrap(cx + 1, nx), cyp = pwrap(cy + 1, ny);
      lds_add<R>(shi, slo, cx * ny + cy, w[0]);
      lds_add<R>(shi, slo, cxp * ny + cy, w[1]);
      lds_add<R>(shi, slo, cx * ny + cyp, w[2]);
      lds_add<R>(shi, slo, cxp * ny + cyp, w[3]);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < G; i += DEP_NT) {
    const unsigned long long v = shi[i];
    if (v) atomicAdd(&hi[i], v);
    if (sizeof(R) == 8) {
      const unsigned long long vl = slo[i];
      if (vl) atomicAdd(&lo[i], vl);
    }
  }
}

// tile of a position: any position, as the weights clamp its cell into the grid
template <typename R>
__device__ __forceinline__ int dep_tile(R x, R y, const Geo<R>& g, const DepositPlan& p) {
  int cx, cy;
  R f;
  locate_w(x, g.idx, g.nx, cx, f);
  locate_w(y, g.idy, g.ny, cy, f);
  return (cx >> p.ltx) * p.tiles_y + (cy >> p.lty);
}

// tile counts of each workgroup's positions -> table[tile][workgroup]
template <typename R, int IT>
__global__ __launch_bounds__(DEP_NT) void k_dep_count(const R* __restrict__ x,
                                                      const R* __restrict__ y, int n, int nx,
                                                      int ny, double lx, double ly,
                                                      DepositPlan p, int* __restrict__ table) {
  __shared__ int h[DEP_MAX_TILES];
  const Geo<R> g = make_geo<R>(nx, ny, lx, ly);
  const int p0 = blockIdx.x * (IT * DEP_NT) + threadIdx.x;
  R xv[IT], yv[IT];
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const int q = min(p0 + u * DEP_NT, n - 1);
    xv[u] = x[q];
    yv[u] = y[q];
  }
  for (int t = threadIdx.x; t < p.tiles; t += DEP_NT) h[t] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u)
    if (p0 + u * DEP_NT < n) atomicAdd(&h[dep_tile<R>(xv[u], yv[u], g, p)], 1);
  __syncthreads();
  for (int t = threadIdx.x; t < p.tiles; t += DEP_NT)
    table[(long long)t * gridDim.x + blockIdx.x] = h[t];
}

// Exclusive scan over the workgroup of two values per thread (v0 before v1).
__device__ __forceinline__ int dep_scan2(int v0, int v1, int* wsum) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = v0 + v1;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int s = __shfl_up(inc, o, 64);
    if (lane >= o) inc += s;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int ex = inc - v0 - v1;
  for (int k = 0; k < w; ++k) ex += wsum[k];
  return ex;
}

// Each workgroup groups its positions by tile in LDS (rank: an LDS atomic, the order inside a
// tile is free) and writes each tile's run, (x, y) pairs together, to tile base + scanned
// table entry.  (Runs reserved by an atomic on a cursor per tile, no table: every workgroup's
// 256 atomics met the others' on the same addresses, 82 us for 8,000,009 positions against
// 35 without them.)  The first workgroup also writes the tile offsets.
template <typename R, int IT>
__global__ __launch_bounds__(DEP_NT) void k_dep_move(const R* __restrict__ x,
                                                     const R* __restrict__ y, int n, int nx,
                                                     int ny, double lx, double ly, DepositPlan p,
                                                     const int* __restrict__ table,
                                                     const int* __restrict__ totals,
                                                     int* __restrict__ offs,
                                                     DepPair<R>* __restrict__ out) {
  __shared__ int cnt[DEP_MAX_TILES], first[DEP_MAX_TILES];
  __shared__ int wsum[2][DEP_NT / 64];
  __shared__ DepPair<R> sp[IT * DEP_NT];
  __shared__ unsigned short st[IT * DEP_NT];
  static_assert(DEP_MAX_TILES <= 2 * DEP_NT, "two tiles per thread");
  const Geo<R> g = make_geo<R>(nx, ny, lx, ly);
  const int b0 = blockIdx.x * (IT * DEP_NT);
  const int count = min(n - b0, IT * DEP_NT);
  R xv[IT], yv[IT];
  int tile[IT], rk[IT];
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const int q = min((int)threadIdx.x + u * DEP_NT, count - 1);
    xv[u] = x[b0 + q];
    yv[u] = y[b0 + q];
  }
  for (int t = threadIdx.x; t < p.tiles; t += DEP_NT) cnt[t] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    tile[u] = dep_tile<R>(xv[u], yv[u], g, p);
    rk[u] = (int)threadIdx.x + u * DEP_NT < count ? atomicAdd(&cnt[tile[u]], 1) : -1;
  }
  __syncthreads();
  {
    const int t = 2 * threadIdx.x;
    const bool h0 = t < p.tiles, h1 = t + 1 < p.tiles;
    const int c0 = h0 ? cnt[t] : 0, c1 = h1 ? cnt[t + 1] : 0;
    const int t0 = h0 ? totals[t] : 0, t1 = h1 ? totals[t + 1] : 0;
    const int r0 = h0 ? table[(long long)t * gridDim.x + blockIdx.x] : 0;
    const int r1 = h1 ? table[(long long)(t + 1) * gridDim.x + blockIdx.x] : 0;
    const int ex = dep_scan2(c0, c1, wsum[0]);    // places in this workgroup's order
    const int base = dep_scan2(t0, t1, wsum[1]);  // slots of the tiles
    // cnt: the tile's first place; first: its slot minus that place
    if (h0) {
      cnt[t] = ex;
      first[t] = base + r0 - ex;
    }
    if (h1) {
      cnt[t + 1] = ex + c0;
      first[t + 1] = base + t0 + r1 - ex - c0;
    }
    if (blockIdx.x == 0) {
      if (h0) offs[t] = base;
      if (h1) offs[t + 1] = base + t0;
      if (threadIdx.x == 0) offs[p.tiles] = n;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u)
    if (rk[u] >= 0) {
      const int q = cnt[tile[u]] + rk[u];
      DepPair<R> v;
      v.x = xv[u];
      v.y = yv[u];
      sp[q] = v;
      st[q] = (unsigned short)tile[u];
    }
  __syncthreads();
  for (int q = threadIdx.x; q < count; q += DEP_NT) out[first[st[q]] + q] = sp[q];
}

// Slice blockIdx.x of the tile order: for each tile it meets, the window of the tile's nodes
// is cleared, summed in LDS and added to the global sums.
template <typename R>
__global__ __launch_bounds__(DEP_NT) void k_dep_slices(const DepPair<R>* __restrict__ pos,
                                                       int n, int nx, int ny, double lx,
                                                       double ly, DepositPlan p,
                                                       const int* __restrict__ offs,
                                                       unsigned long long* hi,
                                                       unsigned long long* lo) {
  extern __shared__ unsigned long long sums[];
  constexpr int U = 4, NQ = (sizeof(R) == 8) ? 2 : 1;
  const Geo<R> g = make_geo<R>(nx, ny, lx, ly);
  const int Wy = (1 << p.lty) + 1, nw = ((1 << p.ltx) + 1) * Wy;
  unsigned long long *shi = sums, *slo = sums + nw;
  const int s0 = blockIdx.x * p.slice, s1 = min(s0 + p.slice, n);
  // the tile of slot s0: the last with offs <= s0 (the empty ones before it are passed over)
  int t = 0, hiT = p.tiles;
  while (hiT - t > 1) {
    const int mid = (t + hiT) >> 1;
    if (offs[mid] <= s0) t = mid;
    else hiT = mid;
  }
  for (int a = s0; a < s1; ++t) {
    const int b = min(offs[t + 1], s1);
    if (b <= a) continue;  // an empty tile
    const int x0 = (t / p.tiles_y) << p.ltx, y0 = (t % p.tiles_y) << p.lty;
    for (int i = threadIdx.x; i < NQ * nw; i += DEP_NT) sums[i] = 0ull;
    __syncthreads();
    for (int q0 = a + threadIdx.x; q0 < b; q0 += U * DEP_NT) {
      DepPair<R> v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = pos[min(q0 + u * DEP_NT, b - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (q0 + u * DEP_NT >= b) continue;
        int cx, cy;
        long long w[4];
        deposit_weights<R>(v[u].x, v[u].y, g, cx, cy, w);
        const int i0 = (cx - x0) * Wy + (cy - y0);
        lds_add<R>(shi, slo, i0, w[0]);
        lds_add<R>(shi, slo, i0 + Wy, w[1]);
        lds_add<R>(shi, slo, i0 + 1, w[2]);
        lds_add<R>(shi, slo, i0 + Wy + 1, w[3]);
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nw; i += DEP_NT) {
      const unsigned long long v = shi[i];
      const unsigned long long vl = (sizeof(R) == 8) ? slo[i] : 0ull;
      if (v | vl) {
        const int r = i / Wy, c = i - r * Wy;
        const long long nd = (long long)pwrap(x0 + r, nx) * ny + pwrap(y0 + c, ny);
        if (v) atomicAdd(&hi[nd], v);
        if (sizeof(R) == 8 && vl) atomicAdd(&lo[nd], vl);
      }
    }
    __syncthreads();
    a = b;
  }
}

inline int grid_for(long long n, int nt, int most) {
  const long long b = (n + nt - 1) / nt;
  return (int)(b < 1 ? 1 : (b > most ? most : b));
}

}  // namespace

// Lines measured as whole calls on one card, FP32 / FP64 where they differ (us):
//   grid, 64^2, 65,536 positions: 23 / 29, direct 30 / 43; below 8 positions per node clearing
//   and adding the copy costs what it saves (128^2 FP32: 37 against 30 at 65,536, 37 against 41
//   at 131,072)
//   binned, 512^2: 36 / 41 against 41 / 66 direct at 131,072 positions, 39 / 43 against 30 / 44
//   at 65,536; on larger grids the tiles' windows cost more (2048^2: 68 / 97 against 77 / 134 at
//   262,144, 70 / 91 against 54 / 89 at 131,072)
DepositPlan deposit_plan(int64_t n, int nx, int ny, int fp64, bool scratch) {
  DepositPlan p;
  const long long G = (long long)nx * ny, words = fp64 ? 2 : 1;
  p.ltx = p.lty = 0;
  p.tiles = p.tiles_y = p.slice = p.items = p.groups = 0;
  p.form = DEPOSIT_DIRECT;
  if (G * words * 8 <= DEP_LDS_GRID) {
    if (n >= 8 * G) p.form = DEPOSIT_GRID;
    return p;
  }
  if (!scratch || n * words < std::max(131072ll, G / 16) || n > 0x7fff0000) return p;
  int lnx = 0, lny = 0;
  while ((1 << lnx) < nx) ++lnx;
  while ((1 << lny) < ny) ++lny;
  // tiles of 32 cells a side, larger ones while there are more than 256 and the window fits
  for (int l = 5;; ++l) {
    p.ltx = l < lnx ? l : lnx;
    p.lty = l < lny ? l : lny;
    p.tiles_y = 1 << (lny - p.lty);
    p.tiles = p.tiles_y << (lnx - p.ltx);
    const long long next = ((2ll << p.ltx) + 1) * ((2ll << p.lty) + 1) * words * 8;
    if (p.tiles <= 256 || (p.tiles <= DEP_MAX_TILES && next > DEP_LDS_WIN)) break;
  }
  p.form = DEPOSIT_BINNED;
  // moving pass: groups of 1024 positions until they fill the chip, then of 4096 (longer runs)
  p.items = n <= (1 << 20) ? 2 : 8;
  p.groups = (int)((n + p.items * DEP_NT - 1) / (p.items * DEP_NT));
  // about 1024 slices, of 1024 to 16384 positions
  const long long s = (n + 1023) / 1024;
  p.slice = (int)(s < 1024 ? 1024 : (s > 16384 ? 16384 : s));
  return p;
}

template <typename R>
void launch_op_deposit(hipStream_t s, const DepositPlan& p, const R* x, const R* y, int64_t n,
                       int nx, int ny, double lx, double ly, unsigned long long* hi,
                       unsigned long long* lo, DepositBufs b) {
  if (p.form == DEPOSIT_GRID) {
    const size_t lds = (size_t)nx * ny * 2 * sizeof(R);
    // a workgroup's copy costs a global atomic per node: at least two positions per node
    const long long most = 2 * lds <= 160 * 1024 ? 512 : 256;
    const long long per = std::max<long long>(2 * DEP_NT, 2ll * nx * ny);
    k_dep_grid<R><<<grid_for(n, (int)per, (int)most), DEP_NT, lds, s>>>(x, y, n, nx, ny, lx, ly,
                                                                       hi, lo);
    return;
  }
  if (p.form == DEPOSIT_DIRECT) {
    k_dep_direct<R><<<grid_for(n, PIC_WG, 8192), PIC_WG, 0, s>>>(x, y, n, nx, ny, lx, ly, hi, lo);
    return;
  }
  const int m = (int)n;
  DepPair<R>* pos = reinterpret_cast<DepPair<R>*>(b.pos);
  if (p.items == 2)
    k_dep_count<R, 2><<<p.groups, DEP_NT, 0, s>>>(x, y, m, nx, ny, lx, ly, p, b.table);
  else
    k_dep_count<R, 8><<<p.groups, DEP_NT, 0, s>>>(x, y, m, nx, ny, lx, ly, p, b.table);
  launch_scan_rows(s, b.table, p.tiles, p.groups, b.totals, nullptr);
  if (p.items == 2)
    k_dep_move<R, 2><<<p.groups, DEP_NT, 0, s>>>(x, y, m, nx, ny, lx, ly, p, b.table, b.totals,
                                                 b.offs, pos);
  else
    k_dep_move<R, 8><<<p.groups, DEP_NT, 0, s>>>(x, y, m, nx, ny, lx, ly, p, b.table, b.totals,
                                                 b.offs, pos);
  const size_t lds = ((size_t)(1 << p.ltx) + 1) * ((1 << p.lty) + 1) * 2 * sizeof(R);
  k_dep_slices<R><<<(m + p.slice - 1) / p.slice, DEP_NT, lds, s>>>(pos, m, nx, ny, lx, ly, p,
                                                                  b.offs, hi, lo);
}

#define DEP_INST(R)                                                                           \
  template void launch_op_deposit<R>(hipStream_t, const DepositPlan&, const R*, const R*,     \
                                     int64_t, int, int, double, double, unsigned long long*,  \
                                     unsigned long long*, DepositBufs);
DEP_INST(float)
DEP_INST(double)
