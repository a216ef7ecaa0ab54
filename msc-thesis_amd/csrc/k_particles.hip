// k_particles.hip -- particle-side kernels: tile sort, fused gather+push+deposit, outputs.
//
// Reference stages replaced (thesisCode/collisionless/double/src/pic.cu):
//   currentCell        :69-87    -> cell key computed inside the sort and the push
//   chargeAssignment   :99-138   -> deterministic fixed-point CIC deposit in LDS windows
//   forceCalculation   :298-355  -> bilinear gather fused into the push
//   positionUpdate     :372-420  -> leapfrog push, periodic wrap into [0, L)
#include <algorithm>
#include <climits>
#include <type_traits>
#include "launch.h"
#include "deposit.h"
#include "step_tail.h"

namespace {

// ------------------------------------------------------------ tile sort of the step
// Stable counting sort of the particles by tile (sort bucket):
//   1. k_tile_hist    per chunk of schunk particles: count of each bucket -> table[b][chunk]
//   2. k_tscan_*      exclusive scan of the table in bucket-major order (per run)
//   3. k_tile_scatter the waves of a workgroup walk a chunk's quarters in index order; lanes
//                     with equal buckets get consecutive slots (ballot ranks), so the
//                     order inside a bucket is the previous order: deterministic and
//                     stable without any per-cell sort.
// The bucket of a position is its tile.  Every pass of one sort evaluates this same
// function, so any deterministic cell choice is consistent: the cell comes from the
// reciprocal multiply (locate_w), the tile from shifts (tile sizes are powers of two).  No
// per-particle division: the count and scatter passes run it once per particle.
template <typename R>
__device__ __forceinline__ int bucket_of(R x, R y, const Geo<R>& g, const RunDesc& rd) {
  int cx, cy;
  R f;
  locate_w(x, g.idx, g.nx, cx, f);
  locate_w(y, g.idy, g.ny, cy, f);
  const int sh = __builtin_ctz((unsigned)rd.tile);
  return (cx >> sh) * rd.tiles_y + (cy >> sh);
}

// Key of the tile sorts: the tile of the position extrapolated by rd.sort_lead (about half
// the span of the steps until the next sort; 0 in runs with collisions, whose cell lists
// need the tiles of the positions themselves).  The particles of a tile range then stay
// within about half a cycle's drift of their tile, instead of drifting a whole cycle away
// from it, so far fewer of them leave the tile's LDS windows (gathers and deposits through
// HBM).  Any key gives the same trajectories; both passes of one sort evaluate it on the
// same stored values.
template <typename R>
__device__ __forceinline__ int bucket_lead(R x, R y, R vx, R vy, const Geo<R>& g,
                                           const RunDesc& rd) {
  if (rd.sort_lead == 0.0) return bucket_of<R>(x, y, g, rd);
  const R t = (R)rd.sort_lead;
  return bucket_of<R>(wrap_pos(fmar(t, vx, x), g.Lx), wrap_pos(fmar(t, vy, y), g.Ly), g, rd);
}

// The same key with its place relative to tile (tx, ty), for the scatter step's ranking:
// bits 0-15 the key, bits 16 and up the neighbour code (dx + 1) * 3 + (dy + 1) of a key
// tile within one tile of (tx, ty) along each axis (periodically), else 9.  With fewer than
// 3 tiles along an axis the neighbours are not distinct tiles: every key gets 9.
#define PUSH_NCODES 9
template <typename R>
__device__ __forceinline__ int bucket_lead_code(R x, R y, R vx, R vy, const Geo<R>& g,
                                                const RunDesc& rd, int tx, int ty) {
  if (rd.sort_lead != 0.0) {
    const R t = (R)rd.sort_lead;
    x = wrap_pos(fmar(t, vx, x), g.Lx);
    y = wrap_pos(fmar(t, vy, y), g.Ly);
  }
  int cx, cy;
  R f;
  locate_w(x, g.idx, g.nx, cx, f);
  locate_w(y, g.idy, g.ny, cy, f);
  const int sh = __builtin_ctz((unsigned)rd.tile);
  const int kx = cx >> sh, ky = cy >> sh;
  // tiles per axis: a power of two
  const int dx = pwrap(kx - tx + 1, rd.tiles_x), dy = pwrap(ky - ty + 1, rd.tiles_y);
  const bool near = rd.tiles_x >= 3 && rd.tiles_y >= 3 && dx <= 2 && dy <= 2;
  const int code = near ? dx * 3 + dy : PUSH_NCODES;
  return (kx * rd.tiles_y + ky) | (code << 16);
}

// the tile of neighbour code c of tile (tx, ty) (bucket_lead_code)
__device__ __forceinline__ int code_tile(int c, int tx, int ty, const RunDesc& rd) {
  int kx = tx + c / 3 - 1, ky = ty + c % 3 - 1;
  kx = kx < 0 ? kx + rd.tiles_x : (kx >= rd.tiles_x ? kx - rd.tiles_x : kx);
  ky = ky < 0 ? ky + rd.tiles_y : (ky >= rd.tiles_y ? ky - rd.tiles_y : ky);
  return kx * rd.tiles_y + ky;
}

// lanes below this one with their bit set in m
__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_tile_hist(const RunDesc* __restrict__ runs,
                                                      const RunState* __restrict__ st,
                                                      const R* __restrict__ x,
                                                      const R* __restrict__ y,
                                                      const R* __restrict__ vx,
                                                      const R* __restrict__ vy,
                                                      int* __restrict__ table,
                                                      const int2* __restrict__ items) {
  extern __shared__ int h[];
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const Geo<R> g = make_geo<R>(rd.nx, rd.ny, rd.lx, rd.ly);
  const int np = st[it.x].np;
  const int nb = rd.nbuckets;
  const int chunk = it.y / rd.schunk;
  for (int b = threadIdx.x; b < nb; b += PIC_WG) h[b] = 0;
  __syncthreads();
  const int p1 = min(it.y + rd.schunk, np);
  // four particles per thread per pass, loads first
  for (int q = it.y + threadIdx.x; q < p1; q += 4 * PIC_WG) {
    R xs[4], ys[4], vxs[4], vys[4];
    const bool lead = rd.sort_lead != 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int p = q + u * PIC_WG;
      xs[u] = p < p1 ? x[rd.pbase + p] : (R)0;
      ys[u] = p < p1 ? y[rd.pbase + p] : (R)0;
      vxs[u] = (lead && p < p1) ? vx[rd.pbase + p] : (R)0;
      vys[u] = (lead && p < p1) ? vy[rd.pbase + p] : (R)0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (q + u * PIC_WG < p1)
        atomicAdd(&h[bucket_lead<R>(xs[u], ys[u], vxs[u], vys[u], g, rd)], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += PIC_WG)
    table[rd.tbase + (long long)b * rd.nchunks + chunk] = h[b];
}

// exclusive scan of one PIC_CELL_CHUNK slice of a run's tile table, in place
__global__ __launch_bounds__(PIC_WG) void k_tscan_local(const RunDesc* __restrict__ runs,
                                                        int* __restrict__ table,
                                                        int* __restrict__ chunk_sums,
                                                        const int2* __restrict__ items) {
  __shared__ int wsum[4];
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const long long len = (long long)rd.nbuckets * rd.nchunks, tb = rd.tbase;
  const long long c0 = it.y + threadIdx.x * 8;
  int v[8], s = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    v[k] = (c0 + k < len) ? table[tb + c0 + k] : 0;
    s += v[k];
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = s;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int wpre = 0;
  for (int k = 0; k < w; ++k) wpre += wsum[k];
  int ex = wpre + inc - s;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (c0 + k < len) table[tb + c0 + k] = ex;
    ex += v[k];
  }
  if (threadIdx.x == PIC_WG - 1) chunk_sums[blockIdx.x] = wpre + inc;
}

__global__ __launch_bounds__(PIC_WG) void k_tscan_chunks(const RunDesc* __restrict__ runs,
                                                         int* __restrict__ chunk_sums) {
  __shared__ int wsum[4];
  const RunDesc rd = runs[blockIdx.x];
  block_exclusive_scan(chunk_sums + rd.tscan_item_begin,
                       rd.tscan_item_end - rd.tscan_item_begin, wsum);
}

__global__ __launch_bounds__(PIC_WG) void k_tscan_add(const RunDesc* __restrict__ runs,
                                                      int* __restrict__ table,
                                                      const int* __restrict__ chunk_sums,
                                                      const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const long long len = (long long)rd.nbuckets * rd.nchunks, tb = rd.tbase;
  const int add = chunk_sums[blockIdx.x];
  for (int k = threadIdx.x; k < PIC_CELL_CHUNK; k += PIC_WG) {
    const long long c = (long long)it.y + k;
    if (c < len) table[tb + c] += add;
  }
}

// ---- scan of the fused sort's count table (the workgroup bodies are in step_tail.h)
__global__ __launch_bounds__(PIC_WG) void k_fscan_part(const RunDesc* __restrict__ runs,
                                                       const int* __restrict__ table,
                                                       int* __restrict__ part, int stride,
                                                       const int2* __restrict__ items) {
  fscan_part(runs, table, part, stride, items, blockIdx.x);
}

__global__ __launch_bounds__(PIC_WG) void k_fscan_base(const RunDesc* __restrict__ runs,
                                                       RunState* __restrict__ st,
                                                       int* __restrict__ part, int stride,
                                                       int* __restrict__ toff) {
  fscan_base(runs, st, part, stride, toff, blockIdx.x);
}

__global__ __launch_bounds__(PIC_WG) void k_fscan_rows(const RunDesc* __restrict__ runs,
                                                       int* __restrict__ table,
                                                       const int* __restrict__ part,
                                                       int stride,
                                                       const int2* __restrict__ items) {
  fscan_rows(runs, table, part, stride, items, blockIdx.x);
}

// A workgroup per chunk of G * TILE_SCAT_NT particles, all of them in registers, an equal part
// per wave in index order, in groups of 64.  Lanes with equal buckets are found by one ballot per
// bucket bit, whatever the order, and the first lane of each bucket counts for all of them, so no
// two lanes meet at a counter.  16,777,216 FP32 particles in no order: 169 us (40 bytes each
// take 132 at the rate of a copy); a ballot per distinct bucket by one wave per chunk 224, the
// state read again for the move 228, moved in the chunk's sorted order 236.  524,288 in order in
// chunks of 1024: 24.6 -> 9.6.
#define TILE_SCAT_NT 512
template <typename R, int G>
__global__ __launch_bounds__(TILE_SCAT_NT) void k_tile_scatter(const RunDesc* __restrict__ runs,
                                                               RunState* __restrict__ st,
                                                               PartBufs<R> src, PartBufs<R> dst,
                                                               const int* __restrict__ table,
                                                               int* __restrict__ toff,
                                                               const int2* __restrict__ items) {
  extern __shared__ int base[];  // [waves][nb]: counts, then the next slots
  constexpr int NT = TILE_SCAT_NT, NW = NT / 64;
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const Geo<R> g = make_geo<R>(rd.nx, rd.ny, rd.lx, rd.ly);
  const int np = st[it.x].np;
  const int nb = rd.nbuckets;
  const int chunk = it.y / (G * NT);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long long pb = rd.pbase;
  const int p1 = min(it.y + G * NT, np);
  const int q0 = it.y + w * 64 * G + lane;  // this lane's particles: q0, q0 + 64, ...
  R x[G], y[G], vx[G], vy[G];
  int id[G];
#pragma unroll
  for (int i = 0; i < G; ++i) {
    // lanes past p1 load the run's first particle
    const int p = q0 + i * 64;
    const long long pl = pb + (p < p1 ? p : 0);
    x[i] = src.x[pl];
    y[i] = src.y[pl];
    vx[i] = src.vx[pl];
    vy[i] = src.vy[pl];
    id[i] = src.id[pl];
  }
  for (int i = threadIdx.x; i < NW * nb; i += NT) base[i] = 0;
  if (chunk == 0 && threadIdx.x == 0) {
    toff[rd.toffbase + nb] = np;
    st[it.x].nsorted = np;
  }
  __syncthreads();
  const int nbits = nb > 1 ? 32 - __builtin_clz((unsigned)(nb - 1)) : 0;
  int* __restrict__ wb = base + w * nb;
  // bucket (bits 0-12), rank among the group's lanes of the bucket (13-18), their number (19-25)
  unsigned at[G];
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const bool act = q0 + i * 64 < p1;
    const unsigned key = (unsigned)bucket_lead<R>(x[i], y[i], vx[i], vy[i], g, rd);
    unsigned long long m = __ballot(act);
    for (int k = 0; k < nbits; ++k) {
      const bool bit = (key >> k) & 1;
      const unsigned long long ones = __ballot(bit);
      m &= bit ? ones : ~ones;
    }
    const unsigned r = (unsigned)lanes_below(m), c = (unsigned)__popcll(m);
    if (act && r == 0) atomicAdd(&wb[key], (int)c);
    at[i] = key | r << 13 | c << 19;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += NT) {
    int v = table[rd.tbase + (long long)b * rd.nchunks + chunk];
    if (chunk == 0) toff[rd.toffbase + b] = v;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      const int c = base[k * nb + b];
      base[k * nb + b] = v;
      v += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (q0 + i * 64 >= p1) continue;
    const unsigned key = at[i] & 8191u, r = (at[i] >> 13) & 63u;
    const int b = wb[key];
    const long long d = pb + b + (int)r;
    // the group's lanes have read their slots before one of them moves the bucket's on, and
    // the next group reads it after (one wave: program order)
    __builtin_amdgcn_wave_barrier();
    if (r == 0) wb[key] = b + (int)(at[i] >> 19);
    __builtin_amdgcn_wave_barrier();
    dst.x[d] = x[i]; dst.y[d] = y[i]; dst.vx[d] = vx[i]; dst.vy[d] = vy[i];
    dst.id[d] = id[i];
  }
}

__global__ void k_fill_i32(int* p, long long n, int v) {
  for (long long i = blockIdx.x * (long long)PIC_WG + threadIdx.x; i < n;
       i += (long long)gridDim.x * PIC_WG)
    p[i] = v;
}
__global__ void k_iota(int* p, long long n) {
  for (long long i = blockIdx.x * (long long)PIC_WG + threadIdx.x; i < n;
       i += (long long)gridDim.x * PIC_WG)
    p[i] = (int)i;
}
__global__ void k_fill_u64(unsigned long long* p, long long n) {
  for (long long i = blockIdx.x * (long long)PIC_WG + threadIdx.x; i < n;
       i += (long long)gridDim.x * PIC_WG)
    p[i] = 0ull;
}

// ===================================================================== push
// One workgroup per (tile, split): the particles of the tile are the T column ranges
// [off[cx*ny + ty*T], off[cx*ny + ty*T + T]) of the cell-sorted arrays.  The new charge
// is accumulated in an LDS window of (T+2H+1)^2 nodes around the tile with int64 atomics
// and flushed once per workgroup; particles that drifted outside the window since the
// last sort deposit straight to HBM.  Gather reads the padded E array (L2-resident).
template <typename R>
struct EWin {
  typedef typename std::conditional<sizeof(R) == 4, float2, double2>::type R2;
};

#include "push_kernel.inc"

// One particle's state as it leaves: (x, y, vx, vy) together.
template <typename R>
struct alignas(4 * sizeof(R)) OutRec {
  R x, y, vx, vy;
};

// Particles of run `run` in id order.  KICK: synchronous velocities, v + 1/2 dt qm E(x) (the
// pending half kick on the copy).  REC: one record per particle to rec[id], for
// k_out_split; else straight to the output arrays (those that are not NULL).
// The particles lie in tile order, so after some steps consecutive ones have unrelated ids and
// every store is a line of its own: bound by those lines.  A record is one line where four
// arrays are four (16,777,216 FP32 particles, the whole output call: 1697 us with the kick in a
// launch of its own, four scattered stores and four copies, 555 with records).
template <typename R, bool KICK, bool REC>
__global__ __launch_bounds__(PIC_WG) void k_out_particles(const RunDesc* __restrict__ runs,
                                                          const RunState* __restrict__ st,
                                                          int run, PartBufs<R> p,
                                                          const R* __restrict__ Eall,
                                                          OutRec<R>* __restrict__ rec,
                                                          R* __restrict__ ox, R* __restrict__ oy,
                                                          R* __restrict__ ovx,
                                                          R* __restrict__ ovy) {
  const RunDesc rd = runs[run];
  const int np = st[run].np;
  const long long q = blockIdx.x * (long long)PIC_WG + threadIdx.x;
  if (q >= np) return;
  const long long i = rd.pbase + q;
  OutRec<R> o;
  o.x = p.x[i]; o.y = p.y[i]; o.vx = p.vx[i]; o.vy = p.vy[i];
  const int k = p.id[i];
  if (KICK) {
    typedef typename EWin<R>::R2 R2;
    const Geo<R> g = make_geo<R>(rd.nx, rd.ny, rd.lx, rd.ly);
    const R hk = (R)(0.5 * rd.dt * rd.qm);
    const R2* E = reinterpret_cast<const R2*>(Eall) + rd.ebase;
    const int ny1 = g.ny + 1;
    int cx, cy;
    R g00, g10, g01, g11, epx, epy;
    gather_weights<R>(o.x, o.y, g, cx, cy, g00, g10, g01, g11);
    const int i00 = cx * ny1 + cy;
    interp<R>(g00, g10, g01, g11, E[i00], E[i00 + ny1], E[i00 + 1], E[i00 + ny1 + 1], epx, epy);
    o.vx = fmar(hk, epx, o.vx);
    o.vy = fmar(hk, epy, o.vy);
  }
  if (k < 0 || k >= np) return;
  if (REC) {
    rec[k] = o;
  } else {
    if (ox) ox[k] = o.x;
    if (oy) oy[k] = o.y;
    if (ovx) ovx[k] = o.vx;
    if (ovy) ovy[k] = o.vy;
  }
}

template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_out_split(const OutRec<R>* __restrict__ rec, int n,
                                                      R* __restrict__ ox, R* __restrict__ oy,
                                                      R* __restrict__ ovx,
                                                      R* __restrict__ ovy) {
  const long long k = blockIdx.x * (long long)PIC_WG + threadIdx.x;
  if (k >= n) return;
  const OutRec<R> o = rec[k];
  if (ox) ox[k] = o.x;
  if (oy) oy[k] = o.y;
  if (ovx) ovx[k] = o.vx;
  if (ovy) ovy[k] = o.vy;
}

template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_check_finite(const RunDesc* __restrict__ runs,
                                                         const RunState* __restrict__ st,
                                                         PartBufs<R> p,
                                                         const int2* __restrict__ items,
                                                         int* flag) {
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const int p1 = min(it.y + PIC_CHUNK, st[it.x].np);
  bool bad = false;
  for (int q = it.y + threadIdx.x; q < p1; q += PIC_WG) {
    const long long i = rd.pbase + q;
    R s = p.x[i] + p.y[i] + p.vx[i] + p.vy[i];
    if (!isfinite(s)) bad = true;
  }
  if (bad) atomicOr(flag, 1);
}

// ===================================================================== ops
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_op_cell_keys(const R* __restrict__ x,
                                                         const R* __restrict__ y, int64_t n,
                                                         int nx, int ny, double dx, double dy,
                                                         int* __restrict__ keys) {
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * PIC_WG) {
    int cx, cy;
    R f;
    locate(x[p], (R)dx, nx, cx, f);
    locate(y[p], (R)dy, ny, cy, f);
    keys[p] = cx * ny + cy;
  }
}

// ---- gather + push of a caller's particles, in place and in any order.  Four sources of the
// field give the same values (each is the node's FP64 field rounded to R):
//   GP_NODES   the caller's two node arrays: eight 8-byte loads per particle
//   GP_PACKED  (Ex, Ey) pairs on the padded (nx + 1) x (ny + 1) nodes, made by k_op_pack_E:
//              a cell's two node rows are two contiguous pieces of two pairs
//   GP_ROWS    the pairs with the two node rows of a cell interleaved, entry (i, j) = nodes
//              (i, j), (i + 1, j): all four corners are one contiguous piece, for twice the
//              memory.  The state is written past the caches, which then hold the pairs
//   GP_LDS     the padded pairs of a small grid, in every workgroup's LDS
// Random positions are bound by the vector L1: 64 lanes of a load meet up to 64 lines, so the
// number of load instructions sets the time (launch_op_gather_push has the measurements).
//   GP_AUTO    nodes, packed or rows by the word that k_op_pack_E leaves
enum { GP_NODES, GP_PACKED, GP_ROWS, GP_LDS, GP_AUTO };

// Form for the order that the positions are in, judged by 64 pairs of neighbours spread over the
// arrays: `ordered` when half of the pairs lie within a row (FP64: four) and 8 columns of each
// other (a wave's gathers meet a few lines), `local` when within a sixteenth of the grid either
// way, else `other`.
// For one whole wave; every workgroup finds the same, as it reads the same particles.
template <typename R>
__device__ __forceinline__ int gp_form(const R* __restrict__ x, const R* __restrict__ y, int64_t n,
                                       const Geo<R>& g, int ordered, int local, int other) {
  const int64_t p = (n - 2) * (threadIdx.x & 63) / 63;
  int cx, cy, dx, dy;
  R f;
  locate_w(x[p], g.idx, g.nx, cx, f);
  locate_w(y[p], g.idy, g.ny, cy, f);
  locate_w(x[p + 1], g.idx, g.nx, dx, f);
  locate_w(y[p + 1], g.idy, g.ny, dy, f);
  auto half_within = [&](int rows, int cols) {
    return __popcll(__ballot(pwrap(dx - cx + rows, g.nx) <= 2 * rows &&
                             pwrap(dy - cy + cols, g.ny) <= 2 * cols)) >= 32;
  };
  if (half_within(sizeof(R) == 8 ? 4 : 1, 8)) return ordered;
  return half_within(g.nx >> 4, g.ny >> 4) ? local : other;
}

// form: GP_PACKED or GP_ROWS (the interleaved form, nx rows of 2 * (ny + 1) entries).  choice (or
// NULL): the form is gp_form's, with `form` as its other, and is written there; GP_NODES packs
// nothing.
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_op_pack_E(const double* __restrict__ ex,
                                                      const double* __restrict__ ey,
                                                      const R* __restrict__ x,
                                                      const R* __restrict__ y, int64_t n,
                                                      int ordered, int local, int form,
                                                      int* choice, int nx, int ny, double lx,
                                                      double ly,
                                                      typename EWin<R>::R2* __restrict__ E) {
  if (choice) {
    __shared__ int chosen;
    if (threadIdx.x < 64) {
      const int c = gp_form<R>(x, y, n, make_geo<R>(nx, ny, lx, ly), ordered, local, form);
      if (threadIdx.x == 0) {
        chosen = c;
        if (blockIdx.x == 0) *choice = c;
      }
    }
    __syncthreads();
    form = chosen;
    if (form == GP_NODES) return;
  }
  const bool rows = form == GP_ROWS;
  const int lny = __builtin_ctz((unsigned)ny);
  const int G = nx * ny;
  for (int q = blockIdx.x * PIC_WG + threadIdx.x; q < G; q += gridDim.x * PIC_WG) {
    const int i = q >> lny, j = q & (ny - 1);
    typename EWin<R>::R2 v;
    v.x = (R)ex[q];
    v.y = (R)ey[q];
    if (rows) {
      // node (i, j): the first of entry (i, j), the second of entry (i - 1, j)
      const long long a = 2ll * i * (ny + 1), b = 2ll * ((i ? i : nx) - 1) * (ny + 1) + 1;
      E[a + 2 * j] = v;
      E[b + 2 * j] = v;
      if (j == 0) E[a + 2 * ny] = E[b + 2 * ny] = v;
      continue;
    }
    typename EWin<R>::R2* row = E + (long long)i * (ny + 1);
    row[j] = v;
    if (j == 0) row[ny] = v;
    if (i == 0) {
      typename EWin<R>::R2* last = E + (long long)nx * (ny + 1);
      last[j] = v;
      if (j == 0) last[ny] = v;
    }
  }
}

// The pushes of a workgroup of NT threads, U particles per thread at a time; returns the thread's
// share of sum |v_n|^2.  el: the padded field in LDS (GP_LDS).
template <typename R, int SRC, int NT, int U>
__device__ __forceinline__ double gp_span(R* x, R* y, R* vx, R* vy, int64_t n,
                                          const double* __restrict__ ex,
                                          const double* __restrict__ ey,
                                          const typename EWin<R>::R2* __restrict__ E,
                                          const typename EWin<R>::R2* el, const Geo<R>& g, R hk,
                                          R dtr, double skc) {
  typedef typename EWin<R>::R2 R2;
  const int nx = g.nx, ny = g.ny, ny1 = ny + 1;
  double ke = 0;
  const int64_t stride = (int64_t)gridDim.x * NT;
  for (int64_t p0 = blockIdx.x * (int64_t)NT + threadIdx.x; p0 < n; p0 += U * stride) {
    // the state of U particles, then their fields, then their pushes (past the end: the last)
    R xr[U], yr[U], vxr[U], vyr[U], g00[U], g10[U], g01[U], g11[U];
    R2 e00[U], e10[U], e01[U], e11[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t p = p0 + u * stride;
      const int64_t pl = p < n ? p : n - 1;
      xr[u] = x[pl]; yr[u] = y[pl]; vxr[u] = vx[pl]; vyr[u] = vy[pl];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int cx, cy;
      R fx, fy;
      locate_w(xr[u], g.idx, nx, cx, fx);
      locate_w(yr[u], g.idy, ny, cy, fy);
      const R qs = (R)(1.0 / (double)(1 << Fix<R>::QB));
      const R gx1 = (R)qweight(fx) * qs, gy1 = (R)qweight(fy) * qs;
      const R gx0 = (R)1 - gx1, gy0 = (R)1 - gy1;
      g00[u] = gx0 * gy0; g10[u] = gx1 * gy0; g01[u] = gx0 * gy1; g11[u] = gx1 * gy1;
      if (SRC == GP_NODES) {
        const int cxp = (cx + 1 == nx) ? 0 : cx + 1, cyp = (cy + 1 == ny) ? 0 : cy + 1;
        const long long n00 = (long long)cx * ny + cy, n10 = (long long)cxp * ny + cy,
                        n01 = (long long)cx * ny + cyp, n11 = (long long)cxp * ny + cyp;
        e00[u].x = (R)ex[n00]; e10[u].x = (R)ex[n10]; e01[u].x = (R)ex[n01]; e11[u].x = (R)ex[n11];
        e00[u].y = (R)ey[n00]; e10[u].y = (R)ey[n10]; e01[u].y = (R)ey[n01]; e11[u].y = (R)ey[n11];
      } else if (SRC == GP_LDS) {
        const int i0 = cx * ny1 + cy;
        e00[u] = el[i0]; e01[u] = el[i0 + 1]; e10[u] = el[i0 + ny1]; e11[u] = el[i0 + ny1 + 1];
      } else if (SRC == GP_ROWS) {
        R2 r[4];
        __builtin_memcpy(r, E + 2 * ((long long)cx * ny1 + cy), sizeof(r));
        e00[u] = r[0]; e10[u] = r[1]; e01[u] = r[2]; e11[u] = r[3];
      } else {
        // two neighbouring pairs as one piece (16 B in FP32, aligned to 8)
        R2 r0[2], r1[2];
        const R2* e = E + (long long)cx * ny1 + cy;
        __builtin_memcpy(r0, e, sizeof(r0));
        __builtin_memcpy(r1, e + ny1, sizeof(r1));
        e00[u] = r0[0]; e01[u] = r0[1]; e10[u] = r1[0]; e11[u] = r1[1];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t p = p0 + u * stride;
      if (p >= n) continue;
      R epx = g00[u] * e00[u].x;
      epx = fmar(g10[u], e10[u].x, epx);
      epx = fmar(g01[u], e01[u].x, epx);
      epx = fmar(g11[u], e11[u].x, epx);
      R epy = g00[u] * e00[u].y;
      epy = fmar(g10[u], e10[u].y, epy);
      epy = fmar(g01[u], e01[u].y, epy);
      epy = fmar(g11[u], e11[u].y, epy);
      const double vsx = (double)vxr[u] + skc * (double)epx;
      const double vsy = (double)vyr[u] + skc * (double)epy;
      ke += vsx * vsx + vsy * vsy;
      const R wx = fmar(hk, epx, vxr[u]), wy = fmar(hk, epy, vyr[u]);
      const R wxp = wrap_pos(fmar(dtr, wx, xr[u]), g.Lx);
      const R wyp = wrap_pos(fmar(dtr, wy, yr[u]), g.Ly);
      if (SRC == GP_ROWS) {
        __builtin_nontemporal_store(wxp, x + p);
        __builtin_nontemporal_store(wyp, y + p);
        __builtin_nontemporal_store(wx, vx + p);
        __builtin_nontemporal_store(wy, vy + p);
      } else {
        x[p] = wxp;
        y[p] = wyp;
        vx[p] = wx;
        vy[p] = wy;
      }
    }
  }
  return ke;
}

template <typename R, int SRC>
__global__ __launch_bounds__(SRC == GP_LDS ? GP_LDS_NT : PIC_WG) void k_op_gather_push(
    R* x, R* y, R* vx, R* vy, int64_t n, const double* __restrict__ ex,
    const double* __restrict__ ey, const typename EWin<R>::R2* __restrict__ E,
    const int* __restrict__ choice, int nx, int ny, double lx, double ly, double dt, double qm,
    double c, double* partials) {
  typedef typename EWin<R>::R2 R2;
  constexpr int NT = SRC == GP_LDS ? GP_LDS_NT : PIC_WG;
  extern __shared__ double2 gp_lds[];
  __shared__ double red[NT / 64];
  const Geo<R> g = make_geo<R>(nx, ny, lx, ly);
  const R hk = (R)(c * dt * qm), dtr = (R)dt;
  const double skc = (c - 0.5) * dt * qm;
  R2* el = reinterpret_cast<R2*>(gp_lds);
  if (SRC == GP_LDS) {
    const int lny = __builtin_ctz((unsigned)ny), ny1 = ny + 1;
#pragma unroll 4
    for (int q = threadIdx.x; q < nx * ny; q += NT) {
      const int i = q >> lny, j = q & (ny - 1);
      R2 v;
      v.x = (R)ex[q];
      v.y = (R)ey[q];
      el[i * ny1 + j] = v;
      if (j == 0) el[i * ny1 + ny] = v;
      if (i == 0) {
        el[nx * ny1 + j] = v;
        if (j == 0) el[nx * ny1 + ny] = v;
      }
    }
    __syncthreads();
  }
  const int form = SRC == GP_AUTO ? *choice : SRC;  // uniform
  auto span = [&](auto src, auto u) {
    return gp_span<R, decltype(src)::value, NT, decltype(u)::value>(x, y, vx, vy, n, ex, ey, E, el,
                                                                   g, hk, dtr, skc);
  };
  using std::integral_constant;
  // the node arrays beside the pairs: as many at a time as the pairs' registers hold
  double ke;
  if (SRC == GP_AUTO && form == GP_NODES)
    ke = span(integral_constant<int, GP_NODES>(), integral_constant<int, sizeof(R) == 4 ? 2 : 4>());
  else if (SRC == GP_AUTO && form == GP_PACKED)
    ke = span(integral_constant<int, GP_PACKED>(), integral_constant<int, 4>());
  else
    ke = span(integral_constant<int, SRC == GP_AUTO ? GP_ROWS : SRC>(),
              integral_constant<int, SRC == GP_NODES ? 1 : 4>());
  if (!partials) return;  // uniform
  ke = wave_sum(ke);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ke;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < NT / 64; ++w) s += red[w];
    partials[blockIdx.x] = s;
  }
}

__global__ __launch_bounds__(PIC_WG) void k_op_fixed_to_double(const unsigned long long* hi,
                                                               const unsigned long long* lo,
                                                               long long G, int fp64,
                                                               double scale, double* out) {
  for (long long q = blockIdx.x * (long long)PIC_WG + threadIdx.x; q < G;
       q += (long long)gridDim.x * PIC_WG) {
    if (fp64)
      out[q] = ((double)(long long)hi[q] * 9.313225746154785e-10 +
                (double)(long long)lo[q] * 8.673617379884035e-19) * scale;
    else
      out[q] = (double)(long long)hi[q] * scale;
  }
}

__global__ void k_reduce_sum(const double* parts, int n, double* out) {
  __shared__ double red[4];
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += PIC_WG) v += parts[i];
  v = block_sum(v, red);
  if (threadIdx.x == 0) *out = v;
}

// Eighth moments of the velocities.  Bound by the read of the velocities; 1024 workgroups, as 256
// leave too few loads in flight: the call that sets 16,777,216 FP32 particles takes 1016 us
// without this kernel, 1108 with 256 workgroups, 1044 with 1024; 10,000 particles 112, 115, 118.
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_speed8(const R* __restrict__ vx,
                                                   const R* __restrict__ vy, int64_t n,
                                                   double* __restrict__ part) {
  __shared__ double red[4];
  double sx = 0.0, sy = 0.0;
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)SPEED_BLOCKS * PIC_WG) {
    const double a = (double)vx[p] * (double)vx[p], b = (double)vy[p] * (double)vy[p];
    sx += (a * a) * (a * a);
    sy += (b * b) * (b * b);
  }
  sx = block_sum(sx, red);
  sy = block_sum(sy, red);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = sx;
    part[2 * blockIdx.x + 1] = sy;
  }
}

inline int grid_for(long long n) {
  long long b = (n + PIC_WG - 1) / PIC_WG;
  return (int)(b < 1 ? 1 : (b > 8192 ? 8192 : b));
}

}  // namespace

// ====================================================================== launchers
void launch_fill_i32(hipStream_t s, int* p, long long n, int v) {
  if (n > 0) k_fill_i32<<<grid_for(n), PIC_WG, 0, s>>>(p, n, v);
}
void launch_iota(hipStream_t s, int* p, long long n) {
  if (n > 0) k_iota<<<grid_for(n), PIC_WG, 0, s>>>(p, n);
}
void launch_fill_u64(hipStream_t s, unsigned long long* p, long long n) {
  if (n > 0) k_fill_u64<<<grid_for(n), PIC_WG, 0, s>>>(p, n);
}
void launch_op_fixed_to_double(hipStream_t s, const unsigned long long* hi,
                               const unsigned long long* lo, long long G, int fp64, double scale,
                               double* out) {
  k_op_fixed_to_double<<<grid_for(G), PIC_WG, 0, s>>>(hi, lo, G, fp64, scale, out);
}
void launch_reduce_sum(hipStream_t s, const double* parts, int n, double* out) {
  k_reduce_sum<<<1, PIC_WG, 0, s>>>(parts, n, out);
}

template <typename R>
void launch_speed8(hipStream_t s, PartBufs<R> p, long long base, int64_t n, double* part) {
  k_speed8<R><<<SPEED_BLOCKS, PIC_WG, 0, s>>>(p.vx + base, p.vy + base, n, part);
}

template <typename R>
void launch_tile_sort(hipStream_t s, const RunDesc* runs, RunState* st, int nruns,
                      PartBufs<R> src, PartBufs<R> dst, SortBufs sb, const int2* pitems,
                      int npitems, int schunk) {
  const size_t lds = sizeof(int) * (size_t)sb.max_buckets;
  k_tile_hist<R><<<npitems, PIC_WG, lds, s>>>(runs, st, src.x, src.y, src.vx, src.vy, sb.table,
                                               pitems);
  k_tscan_local<<<sb.ntscan_items, PIC_WG, 0, s>>>(runs, sb.table, sb.tchunk_sums,
                                                   sb.tscan_items);
  k_tscan_chunks<<<nruns, PIC_WG, 0, s>>>(runs, sb.tchunk_sums);
  k_tscan_add<<<sb.ntscan_items, PIC_WG, 0, s>>>(runs, sb.table, sb.tchunk_sums,
                                                 sb.tscan_items);
  const size_t scat = TILE_SCAT_NT / 64 * lds;
  if (schunk == PIC_CHUNK)
    k_tile_scatter<R, PIC_CHUNK / TILE_SCAT_NT><<<npitems, TILE_SCAT_NT, scat, s>>>(
        runs, st, src, dst, sb.table, sb.toff, pitems);
  else
    k_tile_scatter<R, PIC_CHUNK_SMALL / TILE_SCAT_NT><<<npitems, TILE_SCAT_NT, scat, s>>>(
        runs, st, src, dst, sb.table, sb.toff, pitems);
}

void launch_fused_scan(hipStream_t s, const RunDesc* runs, RunState* st, int nruns,
                       SortBufs sb, int* toff_new) {
  k_fscan_part<<<sb.nfscan_items, PIC_WG, 0, s>>>(runs, sb.ftable, sb.fchunk_sums,
                                                  sb.max_buckets, sb.fscan_items);
  k_fscan_base<<<nruns, PIC_WG, 0, s>>>(runs, st, sb.fchunk_sums, sb.max_buckets, toff_new);
  k_fscan_rows<<<sb.nfscan_items, PIC_WG, 0, s>>>(runs, sb.ftable, sb.fchunk_sums,
                                                  sb.max_buckets, sb.fscan_items);
}

// End of a step, one workgroup per run: the diagnostics row, then the step counter.
// Kernel order makes the partials visible (no grid-wide fences in the producers).
__global__ __launch_bounds__(PIC_WG) void k_step_finish(const RunDesc* __restrict__ runs,
                                                        RunState* __restrict__ st,
                                                        const double* __restrict__ ppush,
                                                        const double* __restrict__ prows,
                                                        double* __restrict__ diag) {
  step_finish_run(runs, st, ppush, prows, diag, blockIdx.x, true);
}

void launch_step_finish(hipStream_t s, const RunDesc* runs, RunState* st, int nruns,
                        const double* ppush, const double* prows, double* diag) {
  k_step_finish<<<nruns, PIC_WG, 0, s>>>(runs, st, ppush, prows, diag);
}

template <typename R>
void launch_push(hipStream_t s, const PushArgs<R>& a) {
  if (a.nitems <= 0) return;
  if (a.by_cell) {
    // FP32 only, and without the fused sort
    if constexpr (sizeof(R) == 4) {
      if (a.mode != 0) k_push<R, 1, 0, 1><<<a.nitems, PUSH_NT, a.lds_bytes, s>>>(a);
      else k_push<R, 0, 0, 1><<<a.nitems, PUSH_NT, a.lds_bytes, s>>>(a);
    }
  } else if (a.mode != 0)
    k_push<R, 1, 0><<<a.nitems, PUSH_NT, a.lds_bytes, s>>>(a);
  else if (a.sort_mode == 1)
    k_push<R, 0, 1><<<a.nitems, PUSH_NT, a.lds_bytes, s>>>(a);
  else if (a.sort_mode == 2)
    k_push<R, 0, 2><<<a.nitems, PUSH_NT, a.lds_bytes, s>>>(a);
  else
    k_push<R, 0, 0><<<a.nitems, PUSH_NT, a.lds_bytes, s>>>(a);
}

// n: the run's particle count (st[run].np).  rec given: records (and nothing else); else the
// output arrays.
template <typename R>
void launch_out_particles(hipStream_t s, const RunDesc* runs, RunState* st, int run, int n,
                          PartBufs<R> p, const R* E, void* rec, R* ox, R* oy, R* ovx, R* ovy) {
  if (n <= 0) return;
  const int blocks = (int)(((long long)n + PIC_WG - 1) / PIC_WG);
  OutRec<R>* r = (OutRec<R>*)rec;
  if (r && E)
    k_out_particles<R, true, true><<<blocks, PIC_WG, 0, s>>>(runs, st, run, p, E, r, ox, oy, ovx,
                                                             ovy);
  else if (r)
    k_out_particles<R, false, true><<<blocks, PIC_WG, 0, s>>>(runs, st, run, p, E, r, ox, oy, ovx,
                                                              ovy);
  else if (E)
    k_out_particles<R, true, false><<<blocks, PIC_WG, 0, s>>>(runs, st, run, p, E, r, ox, oy, ovx,
                                                              ovy);
  else
    k_out_particles<R, false, false><<<blocks, PIC_WG, 0, s>>>(runs, st, run, p, E, r, ox, oy,
                                                               ovx, ovy);
}

template <typename R>
void launch_out_split(hipStream_t s, const void* rec, int n, R* ox, R* oy, R* ovx, R* ovy) {
  if (n > 0)
    k_out_split<R><<<(int)(((long long)n + PIC_WG - 1) / PIC_WG), PIC_WG, 0, s>>>(
        (const OutRec<R>*)rec, n, ox, oy, ovx, ovy);
}

template <typename R>
void launch_check_finite(hipStream_t s, const RunDesc* runs, RunState* st, PartBufs<R> p,
                         const int2* pitems, int npitems, int* flag) {
  k_check_finite<R><<<npitems, PIC_WG, 0, s>>>(runs, st, p, pitems, flag);
}

template <typename R>
void launch_op_cell_keys(hipStream_t s, const R* x, const R* y, int64_t n, int nx, int ny,
                         double lx, double ly, int* keys) {
  k_op_cell_keys<R><<<grid_for(n), PIC_WG, 0, s>>>(x, y, n, nx, ny, lx / nx, ly / ny, keys);
}

// LDS: grids whose padded pairs leave two workgroups per CU.  Packed: enough particles to pay
// for packing (a launch, and 24 or 32 bytes per node).  Whole calls, random order, node arrays
// -> new form, FP32 / FP64 (us):
//   LDS, 64^2: 8,000,009 particles 145 / 155 -> 59 / 97, 1,048,576: 36 / 39 -> 25 / 28
//   (32^2: 20 / 22 -> 20 / 21 at 262,144)
//   packed, 512^2: 8,000,009 particles 281 / 319 -> 112 / 217 (with random velocities 316 ->
//   148; the kernel 269 -> 97 + 5 to pack, FP32), 1,048,576: 56 / 60 -> 35 / 48, 524,288:
//   36 / 38 -> 30 / 36, 262,144: 26 -> 27; 1024^2 at 524,288: 51 / 53 -> 40 / 47, 2048^2 at
//   1,048,577 100 / 106 -> 75 / 91, at 524,289 58 / 63 -> 54 / 65 (66 / 81 from HBM)
// Interleaved rows instead of packed: where they take little of an XCD's 4 MiB L2, where the
// packed pairs do not fit it either, or where the state is a large part of the last-level
// cache, whose lines then come from HBM anyway; enough particles to pay for packing twice the
// memory.  Packed -> rows, the state in the last-level cache / in HBM at the start (us):
//   FP32  128^2: 8,000,009 particles 98 / 155 -> 89 / 135, 1,048,576: 33 / 38 -> 30 / 36
//         512^2: 20,000,003 334 / 376 -> 273 / 301, 8,000,009 114 / 166 -> 126 / 137,
//         but 4,194,304 74 / 95 -> 82 / 88, 1,048,576 36 / 41 -> 41 / 41
//         1024^2: 8,000,009 235 / 238 -> 195 / 199, 1,048,576 54 / 57 -> 52 / 57
//         2048^2: 8,000,009 338 / 350 -> 233 / 251, 4,194,304 201 / 211 -> 146 / 162
//   FP64  128^2: 8,000,009 150 / 235 -> 147 / 209
//         256^2: 8,000,009 146 / 241 -> 163 / 215, but 4,194,304 88 / 133 -> 100 / 132
//         1024^2: 8,000,009 353 / 353 -> 275 / 284, 1,048,576 68 / 73 -> 67 / 77
//         2048^2: 4,194,304 243 / 260 -> 198 / 230, but 1,048,576 88 / 106 -> 84 / 119
// In a step of the operators (deposit, Poisson, E, push: the deposit follows the rows' stores
// past the caches) the large state's line costs 1.6 % at 8,000,009 FP32 on 512^2 (235 -> 239 us
// packed -> rows), gives 11 % at 20,000,003 (567 -> 510), 4 % at 8,000,009 FP64 on 256^2
// (379 -> 362).
// Grids whose pairs outgrow the L2, up to 8 particles per node: random positions want the pairs,
// but those that lie in cell order meet few lines of the node arrays and pay for packing, and
// nearby ones meet few lines of the packed form.  The caller's order is not known here, so the
// packing looks (gp_form: 2 to 4 us).  Sorted / within 10 cells of it / random (us), by node
// arrays; packed; rows; as chosen:
//   FP64 2048^2, 4,194,307: 70 / 112 / 353; 96 / 121 / 241; 134 / 165 / 201; 77 / 125 / 209
//        1024^2, 1,048,579: 35 / 46 / 88; 40 / 50 / 69; 51 / 61 / 69; 39 / 53 / 71
//   FP32 2048^2, 4,194,307: 52 / 106 / 336; 64 / 81 / 198; 72 / 93 / 144; 59 / 82 / 147
//        1024^2, 4,194,307: 47 / 88 / 272; 50 / 64 / 135; 55 / 70 / 118; 53 / 72 / 117
// On smaller grids looking costs what it gives (FP64 512^2, 4,194,307, sorted 80 either way).
GatherPushPlan gather_push_plan(int64_t n, int nx, int ny, int fp64) {
  GatherPushPlan p;
  const long long G = (long long)nx * ny, pad = (long long)(nx + 1) * (ny + 1);
  const long long bytes = pad * (fp64 ? 16 : 8);
  p.pairs = 0;
  p.rows = p.choose = p.ordered = p.local = 0;
  p.lds = 0;
  if (bytes <= 72 * 1024 && n >= std::max(262144ll, 256 * G)) {
    p.lds = (int)bytes;
    // four particles per thread, and at least as many as the fill has nodes
    const long long per = std::max<long long>(4 * GP_LDS_NT, G);
    const long long b = (n + per - 1) / per;
    p.blocks = (int)(b > 512 ? 512 : b);
    return p;
  }
  if (n >= 524288 && n >= G / 4) {
    const long long state = n * (fp64 ? 32 : 16);
    p.rows = n >= std::max(1048576ll, G) &&
             (2 * bytes <= (4 << 20) / 3 || bytes > (6 << 20) || state >= (96ll << 20));
    p.pairs = p.rows ? 2ll * nx * (ny + 1) : pad;
    p.choose = bytes > (6 << 20) && n <= 8 * G;
    p.ordered = fp64 || n <= 2 * G ? GP_NODES : GP_PACKED;
    p.local = fp64 && n < G ? GP_NODES : n <= 4 * G || !p.rows ? GP_PACKED : GP_ROWS;
  }
  const long long per = p.pairs ? 4 * PIC_WG : PIC_WG;
  const long long b = (n + per - 1) / per;
  p.blocks = (int)(b < 1 ? 1 : (b > 4096 ? 4096 : b));
  return p;
}

template <typename R>
void launch_op_gather_push(hipStream_t s, const GatherPushPlan& p, R* x, R* y, R* vx, R* vy,
                           int64_t n, const double* ex, const double* ey, int nx, int ny,
                           double lx, double ly, double dt, double qm, double c,
                           double* ke_partials, void* pairs, int* choice) {
  typedef typename EWin<R>::R2 R2;
  R2* E = (R2*)pairs;
  if (p.lds) {
    k_op_gather_push<R, GP_LDS><<<p.blocks, GP_LDS_NT, p.lds, s>>>(
        x, y, vx, vy, n, ex, ey, nullptr, nullptr, nx, ny, lx, ly, dt, qm, c, ke_partials);
    return;
  }
  auto push = [&](auto kernel) {
    kernel<<<p.blocks, PIC_WG, 0, s>>>(x, y, vx, vy, n, ex, ey, E, choice, nx, ny, lx, ly, dt, qm,
                                       c, ke_partials);
  };
  if (!E) return push(k_op_gather_push<R, GP_NODES>);
  const int other = p.rows ? GP_ROWS : GP_PACKED;
  // workgroups that look at the positions first: no more than fill the chip
  const int blocks = std::min(grid_for((long long)nx * ny), choice ? 2048 : 8192);
  k_op_pack_E<R><<<blocks, PIC_WG, 0, s>>>(ex, ey, x, y, n, p.ordered, p.local, other, choice, nx,
                                           ny, lx, ly, E);
  if (choice) push(k_op_gather_push<R, GP_AUTO>);
  else if (p.rows) push(k_op_gather_push<R, GP_ROWS>);
  else push(k_op_gather_push<R, GP_PACKED>);
}

#define PIC_INST(R)                                                                          \
  template void launch_speed8<R>(hipStream_t, PartBufs<R>, long long, int64_t, double*);     \
  template void launch_tile_sort<R>(hipStream_t, const RunDesc*, RunState*, int, PartBufs<R>,\
                                    PartBufs<R>, SortBufs, const int2*, int, int);            \
  template void launch_push<R>(hipStream_t, const PushArgs<R>&);                            \
  template void launch_out_particles<R>(hipStream_t, const RunDesc*, RunState*, int, int,   \
                                        PartBufs<R>, const R*, void*, R*, R*, R*, R*);      \
  template void launch_out_split<R>(hipStream_t, const void*, int, R*, R*, R*, R*);         \
  template void launch_check_finite<R>(hipStream_t, const RunDesc*, RunState*, PartBufs<R>, \
                                       const int2*, int, int*);                             \
  template void launch_op_cell_keys<R>(hipStream_t, const R*, const R*, int64_t, int, int,  \
                                       double, double, int*);                               \
  template void launch_op_gather_push<R>(hipStream_t, const GatherPushPlan&, R*, R*, R*, R*, \
                                         int64_t, const double*, const double*, int, int,   \
                                         double, double, double, double, double, double*,   \
                                         void*, int*);
PIC_INST(float)
PIC_INST(double)
