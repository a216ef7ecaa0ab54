// k_cellsort.hip -- cell sort of the engine's runs with DSMC collisions: cell lists of
// thesisCode/dsmcCollisions/cellTrackerAdvanced/src/pic.cu:419-445 (particles contiguous per
// cell, ascending id inside a cell), rebuilt every step.
//   k_cell_rank    cell of every particle and its rank among the particles of its cell
//   k_scan_*       exclusive scan of the cell counts; tile offsets
//   k_cell_place   (id, source slot) of every particle to its cell's range, in rank order
//   k_cell_order   each particle's place by id inside its cell, and the particle moved there
//   k_cell_big     the same for cells above CELL_MAX particles, by sorting
// 256^2, 2,097,152 particles, us: a Gaussian blob (183 per cell at its centre) 20 + 10 + 10 +
// 44 + 5, spread out evenly 17 + 10 + 9 + 27 + 5.  With ranks by slices of 1024, a bitonic
// network per cell and the particles moved in a launch of their own the blob's sort took
// 28 + 10 + 7 + 43 + 5 + 29.
#include "launch.h"

namespace {

#define RANK_NT 1024
#define RANK_U (PIC_CHUNK / RANK_NT)  // particles per thread
#define RANK_SLOTS 8192               // LDS table entries: twice the keys a chunk can hold
#define RANK_SHIFT 19                 // 32 - log2 RANK_SLOTS
#define CELL_MAX 512                  // particles of a cell ranked by counting
#define CELL_U 4                      // slots per thread of the ordering kernel
#define CELL_SLICES (PIC_CHUNK / (CELL_U * PIC_WG))
static_assert(CELL_SLICES * CELL_U * PIC_WG == PIC_CHUNK, "whole slices");

// Cell numbering of the engine's own sorts: tile-major (tile t = (cx/T)*tiles_y + cy/T,
// then cx%T, cy%T), so that every tile and every cell is one contiguous range.
// Tile sizes are powers of two and cells are clamped to >= 0: shifts and masks.
__device__ __forceinline__ int engine_cell_key(int cx, int cy, const RunDesc& rd) {
  const int sh = __builtin_ctz((unsigned)rd.tile), m = rd.tile - 1;
  const int t = (cx >> sh) * rd.tiles_y + (cy >> sh);
  return (((t << sh) + (cx & m)) << sh) + (cy & m);
}

__device__ __forceinline__ int cell_of(float x, float y, float dx, float dy, const RunDesc& rd) {
  int cx, cy;
  float f;
  locate(x, dx, rd.nx, cx, f);
  locate(y, dy, rd.ny, cy, f);
  return engine_cell_key(cx, cy, rd);
}

// One chunk per workgroup.  Its particles are counted per cell in an LDS hash table (the cell
// numbers of neighbouring tiles lie far apart, and a window over them all outgrows LDS on
// larger grids), then each cell found costs one returning atomic on the global counts: those
// atomics bound the kernel, so chunks are as large as a workgroup can take.
__global__ __launch_bounds__(RANK_NT) void k_cell_rank(const RunDesc* __restrict__ runs,
                                                       const RunState* __restrict__ st,
                                                       const float* __restrict__ x,
                                                       const float* __restrict__ y,
                                                       int* __restrict__ keys,
                                                       int* __restrict__ rank,
                                                       int* __restrict__ counts,
                                                       const int2* __restrict__ items) {
  __shared__ int tkey[RANK_SLOTS], tcnt[RANK_SLOTS];
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const int np = st[it.x].np;
  const int p0 = it.y, p1 = min(p0 + PIC_CHUNK, np);
  if (p0 >= p1) return;  // uniform across the workgroup
  const long long pb = rd.pbase;
  const float dxr = (float)rd.dx, dyr = (float)rd.dy;
  // the chunk's loads go out together (lanes past p1 load particle p1 - 1)
  float xv[RANK_U], yv[RANK_U];
#pragma unroll
  for (int u = 0; u < RANK_U; ++u) {
    const int pl = min(p0 + (int)threadIdx.x + u * RANK_NT, p1 - 1);
    xv[u] = x[pb + pl];
    yv[u] = y[pb + pl];
  }
  for (int i = threadIdx.x; i < RANK_SLOTS; i += RANK_NT) {
    tkey[i] = -1;
    tcnt[i] = 0;
  }
  __syncthreads();
  int slot[RANK_U], rk[RANK_U];
#pragma unroll
  for (int u = 0; u < RANK_U; ++u) {
    const int p = p0 + threadIdx.x + u * RANK_NT;
    slot[u] = -1;
    if (p >= p1) continue;
    const int key = cell_of(xv[u], yv[u], dxr, dyr, rd);
    keys[pb + p] = key;
    // at most PIC_CHUNK of the RANK_SLOTS entries are ever taken, so the probe ends
    unsigned h = ((unsigned)key * 2654435761u) >> RANK_SHIFT;
    for (;;) {
      int k = tkey[h];
      if (k == -1) k = atomicCAS(&tkey[h], -1, key);
      if (k == -1 || k == key) break;
      h = (h + 1) & (RANK_SLOTS - 1);
    }
    slot[u] = (int)h;
    rk[u] = atomicAdd(&tcnt[h], 1);
  }
  __syncthreads();
  int* cnt = counts + rd.cbase;
  for (int i = threadIdx.x; i < RANK_SLOTS; i += RANK_NT) {
    const int c = tcnt[i];
    if (c) tcnt[i] = atomicAdd(&cnt[tkey[i]], c);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < RANK_U; ++u)
    if (slot[u] >= 0) rank[pb + p0 + threadIdx.x + u * RANK_NT] = rk[u] + tcnt[slot[u]];
}

// exclusive scan of the counts of one chunk of PIC_CELL_CHUNK cells; the counts are zeroed
// once read (they are zero between sorts, so no fill launch precedes the rank kernel)
__global__ __launch_bounds__(PIC_WG) void k_scan_local(const RunDesc* __restrict__ runs,
                                                       int* __restrict__ counts,
                                                       int* __restrict__ offsets,
                                                       int* __restrict__ chunk_sums,
                                                       const int2* __restrict__ items) {
  __shared__ int wsum[4];
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const int G = rd.nx * rd.ny;
  const int c0 = it.y + threadIdx.x * 8;
  int v[8], s = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    int c = c0 + k;
    v[k] = (c < G) ? counts[rd.cbase + c] : 0;
    s += v[k];
  }
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (c0 + k < G) counts[rd.cbase + c0 + k] = 0;
  // inclusive wave scan of per-thread totals
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
    int c = c0 + k;
    if (c < G) offsets[rd.cbase + c] = ex;
    ex += v[k];
  }
  if (threadIdx.x == PIC_WG - 1) chunk_sums[blockIdx.x] = wpre + inc;
}

// The chunk's base added to its offsets: the base is the sum of the run's chunk totals
// before it (integer adds, so any order gives the same base), added up by the workgroup
// itself, which saves a launch that scanned the chunk totals.  Also the tile offsets toff[t] =
// offsets[t T^2] (the cell numbering is tile-major: tile t owns cells [t T^2, (t + 1) T^2)).
// The run's last chunk writes the total: offsets[G], nsorted and the closing tile offset; the
// first workgroup clears the count of cells too large for the within-cell sort's small kernel
// (which appends to it next).
__global__ __launch_bounds__(PIC_WG) void k_scan_add(const RunDesc* __restrict__ runs,
                                                     RunState* __restrict__ st,
                                                     int* __restrict__ offsets,
                                                     const int* __restrict__ chunk_sums,
                                                     const int2* __restrict__ items,
                                                     int* __restrict__ toff,
                                                     int* __restrict__ big_count) {
  __shared__ int wsum[PIC_WG / 64];
  const int2 it = items[blockIdx.x];
  const RunDesc rd = runs[it.x];
  const int G = rd.nx * rd.ny;
  const int TT = rd.tile * rd.tile;
  int part = 0;
  for (int i = rd.cell_item_begin + (int)threadIdx.x; i < (int)blockIdx.x; i += PIC_WG)
    part += chunk_sums[i];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) part += __shfl_xor(part, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = part;
  __syncthreads();
  int add = 0;
#pragma unroll
  for (int w = 0; w < PIC_WG / 64; ++w) add += wsum[w];
  for (int k = threadIdx.x; k < PIC_CELL_CHUNK; k += PIC_WG) {
    int c = it.y + k;
    if (c < G) {
      const int o = offsets[rd.cbase + c] + add;
      offsets[rd.cbase + c] = o;
      if (c % TT == 0) toff[rd.toffbase + c / TT] = o;
    }
  }
  if (threadIdx.x == 0) {
    if ((int)blockIdx.x == rd.cell_item_end - 1) {
      const int total = add + chunk_sums[blockIdx.x];
      offsets[rd.cbase + G] = total;
      st[it.x].nsorted = total;
      toff[rd.toffbase + rd.nbuckets] = total;
    }
    if (blockIdx.x == 0) *big_count = 0;
  }
}

__global__ __launch_bounds__(PIC_WG) void k_cell_place(const RunDesc* __restrict__ runs,
                                                       const RunState* __restrict__ st,
                                                       const int* __restrict__ keys,
                                                       const int* __restrict__ rank,
                                                       const int* __restrict__ id,
                                                       const int* __restrict__ offsets,
                                                       unsigned long long* __restrict__ rec,
                                                       const int2* __restrict__ items) {
  const int2 it = items[blockIdx.x / CELL_SLICES];
  const RunDesc rd = runs[it.x];
  const int np = st[it.x].np;
  const int p0 = it.y + (blockIdx.x % CELL_SLICES) * (CELL_U * PIC_WG);
  const int p1 = min(p0 + CELL_U * PIC_WG, np);
  if (p0 >= p1) return;
  const long long pb = rd.pbase;
  int d[CELL_U], idv[CELL_U];
#pragma unroll
  for (int u = 0; u < CELL_U; ++u) {
    const int pl = min(p0 + (int)threadIdx.x + u * PIC_WG, p1 - 1);
    d[u] = offsets[rd.cbase + keys[pb + pl]] + rank[pb + pl];
    idv[u] = id[pb + pl];
  }
#pragma unroll
  for (int u = 0; u < CELL_U; ++u) {
    const int p = p0 + threadIdx.x + u * PIC_WG;
    if (p < p1)
      rec[pb + d[u]] = ((unsigned long long)(unsigned)idv[u] << 32) | (unsigned)p;
  }
}

// 1024 consecutive slots per workgroup, a thread per slot: its place is the start of its cell
// plus the ids of the cell below its own, counted over the cell's ids in LDS.  n comparisons
// per particle of an n-particle cell, without exchanges between lanes: less than a bitonic
// network's steps up to a few hundred particles (the lanes of a wave hold neighbouring cells,
// which share the LDS reads).  The particle's state is loaded before the counting.
__global__ __launch_bounds__(PIC_WG) void k_cell_order(const RunDesc* __restrict__ runs,
                                                       const RunState* __restrict__ st,
                                                       const unsigned long long* __restrict__ rec,
                                                       const int* __restrict__ offsets,
                                                       PartBufs<float> src, PartBufs<float> dst,
                                                       int* __restrict__ big_list,
                                                       int* __restrict__ big_count,
                                                       const int2* __restrict__ items) {
  // the slots' ids and those of the first and last cell beyond the slots
  __shared__ int ids[CELL_U * PIC_WG + 2 * CELL_MAX];
  __shared__ int range[2];
  const int2 it = items[blockIdx.x / CELL_SLICES];
  const RunDesc rd = runs[it.x];
  const int np = st[it.x].np;
  const int s0 = it.y + (blockIdx.x % CELL_SLICES) * (CELL_U * PIC_WG);
  const int s1 = min(s0 + CELL_U * PIC_WG, np);
  if (s0 >= s1) return;  // uniform across the workgroup
  const long long pb = rd.pbase;
  const float dxr = (float)rd.dx, dyr = (float)rd.dy;
  float x[CELL_U], y[CELL_U], vx[CELL_U], vy[CELL_U];
  int idv[CELL_U], b[CELL_U], n[CELL_U], key[CELL_U];
#pragma unroll
  for (int u = 0; u < CELL_U; ++u) {
    const unsigned long long r = rec[pb + min(s0 + (int)threadIdx.x + u * PIC_WG, s1 - 1)];
    const long long s = pb + (int)(unsigned)(r & 0xffffffffull);
    idv[u] = (int)(r >> 32);
    x[u] = src.x[s]; y[u] = src.y[s]; vx[u] = src.vx[s]; vy[u] = src.vy[s];
  }
#pragma unroll
  for (int u = 0; u < CELL_U; ++u) {
    key[u] = cell_of(x[u], y[u], dxr, dyr, rd);  // as k_cell_rank has it, from the same values
    b[u] = offsets[rd.cbase + key[u]];
    n[u] = offsets[rd.cbase + key[u] + 1] - b[u];
    const int slot = s0 + threadIdx.x + u * PIC_WG;
    if (slot == s0) range[0] = n[u] > CELL_MAX ? s0 : b[u];
    if (slot == s1 - 1) range[1] = n[u] > CELL_MAX ? s1 : b[u] + n[u];
  }
  __syncthreads();
  const int i0 = range[0], i1 = range[1];
  for (int i = i0 + threadIdx.x; i < i1; i += PIC_WG) ids[i - i0] = (int)(rec[pb + i] >> 32);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < CELL_U; ++u) {
    const int slot = s0 + threadIdx.x + u * PIC_WG;
    if (slot >= s1) continue;
    if (n[u] > CELL_MAX) {  // k_cell_big's
      if (slot == b[u]) {
        const int q = atomicAdd(big_count, 1);
        big_list[2 * q] = it.x;
        big_list[2 * q + 1] = key[u];
      }
      continue;
    }
    const int* c = ids + (b[u] - i0);
    int r = 0, k = 0;
    for (; k + 4 <= n[u]; k += 4) {
      const int c0 = c[k], c1 = c[k + 1], c2 = c[k + 2], c3 = c[k + 3];
      r += (c0 < idv[u] ? 1 : 0) + (c1 < idv[u] ? 1 : 0);
      r += (c2 < idv[u] ? 1 : 0) + (c3 < idv[u] ? 1 : 0);
    }
    for (; k < n[u]; ++k) r += c[k] < idv[u] ? 1 : 0;
    const long long d = pb + b[u] + r;
    dst.x[d] = x[u]; dst.y[d] = y[u]; dst.vx[d] = vx[u]; dst.vy[d] = vy[u];
    dst.id[d] = idv[u];
  }
}

// Large cells: bitonic sort of their records by one workgroup, in LDS up to 4096 entries, else
// in a global scratch region [2*(pbase+b), 2*(pbase+b) + m) with m = next pow2 >= n (<= 2n),
// then their particles moved.
__global__ __launch_bounds__(PIC_WG) void k_cell_big(const RunDesc* __restrict__ runs,
                                                     const unsigned long long* __restrict__ rec,
                                                     const int* __restrict__ offsets,
                                                     PartBufs<float> src, PartBufs<float> dst,
                                                     const int* __restrict__ big_list,
                                                     const int* __restrict__ big_count,
                                                     unsigned long long* __restrict__ scratch) {
  __shared__ unsigned long long s[4096];
  const int nbig = *big_count;
  for (int q = blockIdx.x; q < nbig; q += gridDim.x) {
    const int run = big_list[2 * q], c = big_list[2 * q + 1];
    const RunDesc rd = runs[run];
    const long long pb = rd.pbase;
    const int b = offsets[rd.cbase + c], e = offsets[rd.cbase + c + 1];
    const int n = e - b;
    int m = 1;
    while (m < n) m <<= 1;
    unsigned long long* a = (m <= 4096) ? s : scratch + 2 * (pb + b);
    for (int i = threadIdx.x; i < m; i += PIC_WG) a[i] = (i < n) ? rec[pb + b + i] : ~0ull;
    __syncthreads();
    for (int k = 2; k <= m; k <<= 1) {
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int i = threadIdx.x; i < m; i += PIC_WG) {
          int l = i ^ j;
          if (l > i) {
            unsigned long long u = a[i], v = a[l];
            bool up = (i & k) == 0;
            if ((u > v) == up) { a[i] = v; a[l] = u; }
          }
        }
        __syncthreads();
      }
    }
    for (int i = threadIdx.x; i < n; i += PIC_WG) {
      const unsigned long long r = a[i];
      const long long f = pb + (int)(unsigned)(r & 0xffffffffull), d = pb + b + i;
      dst.x[d] = src.x[f]; dst.y[d] = src.y[f]; dst.vx[d] = src.vx[f]; dst.vy[d] = src.vy[f];
      dst.id[d] = (int)(r >> 32);
    }
    __syncthreads();
  }
}

}  // namespace

void launch_cell_sort(hipStream_t s, const RunDesc* runs, RunState* st, PartBufs<float> src,
                      PartBufs<float> dst, SortBufs sb, const int2* pitems, int npitems,
                      const int2* citems, int ncitems) {
  // sb.counts is zero here: zeroed at allocation and by the scan of every sort since
  k_cell_rank<<<npitems, RANK_NT, 0, s>>>(runs, st, src.x, src.y, sb.keys, sb.rank, sb.counts,
                                          pitems);
  k_scan_local<<<ncitems, PIC_WG, 0, s>>>(runs, sb.counts, sb.offsets, sb.chunk_sums, citems);
  k_scan_add<<<ncitems, PIC_WG, 0, s>>>(runs, st, sb.offsets, sb.chunk_sums, citems, sb.toff,
                                        sb.big_count);
  k_cell_place<<<npitems * CELL_SLICES, PIC_WG, 0, s>>>(runs, st, sb.keys, sb.rank, src.id,
                                                        sb.offsets, sb.rec, pitems);
  k_cell_order<<<npitems * CELL_SLICES, PIC_WG, 0, s>>>(runs, st, sb.rec, sb.offsets, src, dst,
                                                        sb.big_list, sb.big_count, pitems);
  k_cell_big<<<256, PIC_WG, 0, s>>>(runs, sb.rec, sb.offsets, src, dst, sb.big_list,
                                    sb.big_count, sb.scratch);
}
