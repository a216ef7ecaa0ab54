// k_radix.hip -- stable sort of integer keys (pic_op_sort): perm, counts and offsets of the
// cell lists of thesisCode/dsmcCollisions/cellTrackerAdvanced/src/pic.cu:419-445.
//
// Least-significant-digit radix sort of (key, index): the keys have ceil(log2 ncells) bits,
// taken in equal digits of at most 8 bits (65,536 cells: two passes).  Every pass is stable,
// so ties keep ascending index without a sort inside the cells.  A pass is three launches:
//   hist     digit counts of each workgroup's tile of items -> table[digit][tile]
//   rows     exclusive scan of each digit's row over the tiles, and the digit totals
//   scatter  ranks inside the tile (below), items grouped by digit in LDS, then written in
//            runs of one digit to slot digit base + row entry + place in the tile's run
// after which offsets[c] is the lower bound of c in the sorted keys.
// Bound: HBM (12 to 20 B moved per item and pass) above about a million items, launch
// latency below.  Ranking by digit costs the same for any distribution of keys: the counting
// sort this replaced took one returning global atomic per particle (127 us for 3,000,017 in
// 65,536 cells, random order) and then ordered each cell by index, a cell above 256
// particles by one workgroup's bitonic network (2.9 ms for the 2-cell sort of 100,003).
// Whole calls, counting sort -> this one: 434 -> 88 us (keys and sort of the 3,000,017); with the
// other steps of it, 7.0 -> 0.21 ms (the reference's DSMC collide of 100,003 particles, which
// sorts twice).
#include "launch.h"

namespace {

#define RADIX_MAX 256            // digits per pass
#define RADIX_NT 512             // threads of the scatter

__device__ __forceinline__ int radix_lanes_below(unsigned long long m) {
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                        __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// Exclusive scan over the threads of a workgroup of NW waves; *total (every thread) the sum.
// The caller synchronises before wsum is used again.
template <int NW>
__device__ __forceinline__ int wg_exclusive(int v, int* wsum, int* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int pre = 0, sum = 0;
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    if (k < w) pre += wsum[k];
    sum += wsum[k];
  }
  *total = sum;
  return pre + inc - v;
}

// FIRST: the caller's keys, checked against [0, ncells) (flag); later kernels do nothing once
// it is set, so a refused call writes none of its outputs.
template <int IT, bool FIRST>
__global__ __launch_bounds__(PIC_WG) void k_radix_hist(const int* __restrict__ keys, int n,
                                                       int shift, int bits, int ncells,
                                                       int ntiles, int* __restrict__ table,
                                                       int* __restrict__ flag) {
  __shared__ int h[RADIX_MAX];
  if (!FIRST && *flag) return;
  const int nd = 1 << bits;
  if (threadIdx.x < nd) h[threadIdx.x] = 0;
  __syncthreads();
  const int p0 = blockIdx.x * (IT * PIC_WG) + threadIdx.x;
  int k[IT];
#pragma unroll
  for (int u = 0; u < IT; ++u) k[u] = keys[min(p0 + u * PIC_WG, n - 1)];
  bool bad = false;
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    if (FIRST && (k[u] < 0 || k[u] >= ncells)) bad = true;
    if (p0 + u * PIC_WG < n) atomicAdd(&h[((unsigned)k[u] >> shift) & (nd - 1)], 1);
  }
  if (FIRST && bad) atomicOr(flag, 1);
  __syncthreads();
  if (threadIdx.x < nd) table[(long long)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// one workgroup per digit: its row of the table scanned in place, four tiles per thread
// (flag may be NULL)
__global__ __launch_bounds__(PIC_WG) void k_radix_rows(int* __restrict__ table, int ntiles,
                                                       int* __restrict__ totals,
                                                       const int* __restrict__ flag) {
  constexpr int NW = PIC_WG / 64;
  __shared__ int wsum[NW];
  if (flag && *flag) return;
  int* row = table + (long long)blockIdx.x * ntiles;
  int carry = 0;
  for (int t0 = 0; t0 < ntiles; t0 += 4 * PIC_WG) {
    const int i = t0 + 4 * threadIdx.x;
    int v[4], s = 0, total;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = (i + k < ntiles) ? row[i + k] : 0;
      s += v[k];
    }
    int ex = carry + wg_exclusive<NW>(s, wsum, &total);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (i + k < ntiles) row[i + k] = ex;
      ex += v[k];
    }
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Items of a tile go by (wave, u, lane), which is their order in the input.  A wave ranks
// its 64 items of one u by their digit with one ballot per digit bit (the lanes that agree
// in every bit), on top of its running count of the digit in LDS: a chain over the wave's items,
// so tiles are spread over eight waves (us per pass with four, eight and sixteen: 3,000,017 items
// in tiles of 4096 20.2, 19.7, 26; 100,003 in tiles of 1024 5.8, 5.0, 5.0).
template <int IT, bool FIRST>
__global__ __launch_bounds__(RADIX_NT) void k_radix_scatter(
    const int* __restrict__ keys, const int* __restrict__ idx, int n, int shift, int bits,
    int ntiles, const int* __restrict__ table, const int* __restrict__ totals,
    int* __restrict__ keys_out, int* __restrict__ idx_out, const int* __restrict__ flag) {
  constexpr int NT = RADIX_NT, NW = NT / 64;
  __shared__ int wh[NW][RADIX_MAX];  // per-wave digit counts, then their prefix
  __shared__ int lstart[RADIX_MAX], gstart[RADIX_MAX];
  __shared__ int wsum[2][NW];
  __shared__ int skey[IT * NT], sidx[IT * NT];
  if (*flag) return;
  const int nd = 1 << bits, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int tile0 = blockIdx.x * (IT * NT);
  const int count = min(IT * NT, n - tile0);
  const int q0 = w * (IT * 64) + lane;
  int k[IT], ix[IT], rk[IT];
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const int p = tile0 + min(q0 + u * 64, count - 1);
    k[u] = keys[p];
    ix[u] = FIRST ? p : idx[p];
  }
#pragma unroll
  for (int q = 0; q < NW; ++q)
    if (threadIdx.x < nd) wh[q][threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const bool ok = q0 + u * 64 < count;
    const int dg = (int)(((unsigned)k[u] >> shift) & (nd - 1));
    unsigned long long m = __ballot(ok);
    for (int b = 0; b < bits; ++b) {
      const bool one = (dg >> b) & 1;
      const unsigned long long s = __ballot(one);
      m &= one ? s : ~s;
    }
    const int below = radix_lanes_below(m);
    const int had = wh[w][dg];
    rk[u] = had + below;
    // the lanes of a wave read had before its first lane of the digit moves the count on
    __builtin_amdgcn_wave_barrier();
    if (ok && below == 0) wh[w][dg] = had + __popcll(m);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  {
    const int d = threadIdx.x;
    int c[NW], mine = 0;
#pragma unroll
    for (int q = 0; q < NW; ++q) {
      c[q] = (d < nd) ? wh[q][d] : 0;
      mine += c[q];
    }
    int sum;
    const int ls = wg_exclusive<NW>(mine, wsum[0], &sum);
    const int gb = wg_exclusive<NW>(d < nd ? totals[d] : 0, wsum[1], &sum);
    if (d < nd) {
      int run = 0;
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        wh[q][d] = run;
        run += c[q];
      }
      lstart[d] = ls;
      gstart[d] = gb + table[(long long)d * ntiles + blockIdx.x] - ls;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    if (q0 + u * 64 >= count) continue;
    const int dg = (int)(((unsigned)k[u] >> shift) & (nd - 1));
    const int lp = lstart[dg] + wh[w][dg] + rk[u];
    skey[lp] = k[u];
    sidx[lp] = ix[u];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < count; i += NT) {
    const int key = skey[i];
    const int dst = gstart[((unsigned)key >> shift) & (nd - 1)] + i;
    keys_out[dst] = key;
    idx_out[dst] = sidx[i];
  }
}

// lower bound of v in a[lo, hi), a quarter of the range per step (three loads at once)
__device__ __forceinline__ int lower_bound_i(const int* __restrict__ a, int lo, int hi, int v) {
  while (lo < hi) {
    const int len = hi - lo;
    const int m1 = lo + len / 4, m2 = lo + len / 2, m3 = m2 + len / 4;  // all below hi
    const bool b1 = a[m1] < v, b2 = a[m2] < v, b3 = a[m3] < v;
    const int l = b3 ? m3 + 1 : b2 ? m2 + 1 : b1 ? m1 + 1 : lo;
    hi = !b1 ? m1 : !b2 ? m2 : !b3 ? m3 : hi;
    lo = l;
  }
  return lo;
}

// A search per cell costs the same for any gaps between the occupied cells; a cell's end is its
// right neighbour's search.  The chain of its loads is the kernel's time, so it starts from the
// range of the cell's last digit (the totals of the last pass; NULL: no items) and takes three
// loads per step (3,000,017 items, 65,536 cells: 9 us; from the whole array, one load per step 12).
__global__ __launch_bounds__(PIC_WG) void k_radix_offsets(const int* __restrict__ sorted, int n,
                                                          int ncells, int shift, int bits,
                                                          const int* __restrict__ totals,
                                                          int* __restrict__ counts,
                                                          int* __restrict__ offsets,
                                                          const int* __restrict__ flag) {
  constexpr int NW = PIC_WG / 64;
  static_assert(RADIX_MAX == PIC_WG, "a digit per thread");
  __shared__ int start[RADIX_MAX + 1];
  __shared__ int wsum[NW];
  if (*flag) return;
  {
    int sum;
    const int d = threadIdx.x;
    start[d] = wg_exclusive<NW>(totals && d < (1 << bits) ? totals[d] : 0, wsum, &sum);
    if (d == 0) start[RADIX_MAX] = sum;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  auto search = [&](long long c) {
    if (c >= ncells || n == 0) return n;
    const int d = (int)c >> shift;
    return lower_bound_i(sorted, start[d], start[d + 1], (int)c);
  };
  for (long long c0 = blockIdx.x * (long long)PIC_WG + threadIdx.x - lane; c0 < ncells;
       c0 += (long long)gridDim.x * PIC_WG) {
    const long long c = c0 + lane;
    const int b = search(c);
    int e = __shfl_down(b, 1, 64);
    if (lane == 63) e = search(c + 1);
    if (c < ncells) {
      offsets[c] = b;
      counts[c] = e - b;
      if (c == ncells - 1) offsets[ncells] = e;
    }
  }
}

template <int IT>
void radix_passes(hipStream_t s, const int* keys, int n, int ncells, const RadixPlan& p,
                  RadixBufs b, int* perm, int* counts, int* offsets) {
  constexpr int SIT = IT * PIC_WG / RADIX_NT;
  const int* kin = keys;
  const int* iin = nullptr;
  for (int q = 0; q < p.passes && n > 0; ++q) {
    const int shift = q * p.bits;
    int* kout = b.keys[q & 1];
    int* iout = (q == p.passes - 1) ? perm : b.idx[q & 1];
    if (q == 0)
      k_radix_hist<IT, true><<<p.tiles, PIC_WG, 0, s>>>(kin, n, shift, p.bits, ncells, p.tiles,
                                                        b.table, b.flag);
    else
      k_radix_hist<IT, false><<<p.tiles, PIC_WG, 0, s>>>(kin, n, shift, p.bits, ncells, p.tiles,
                                                         b.table, b.flag);
    launch_scan_rows(s, b.table, 1 << p.bits, p.tiles, b.totals, b.flag);
    if (q == 0)
      k_radix_scatter<SIT, true><<<p.tiles, RADIX_NT, 0, s>>>(
          kin, iin, n, shift, p.bits, p.tiles, b.table, b.totals, kout, iout, b.flag);
    else
      k_radix_scatter<SIT, false><<<p.tiles, RADIX_NT, 0, s>>>(
          kin, iin, n, shift, p.bits, p.tiles, b.table, b.totals, kout, iout, b.flag);
    kin = kout;
    iin = iout;
  }
  const long long blocks = ((long long)ncells + PIC_WG - 1) / PIC_WG;
  k_radix_offsets<<<(int)(blocks > 16384 ? 16384 : blocks), PIC_WG, 0, s>>>(
      kin, n, ncells, (p.passes - 1) * p.bits, p.bits, n > 0 ? b.totals : nullptr, counts, offsets,
      b.flag);
}

}  // namespace

void launch_scan_rows(hipStream_t s, int* table, int rows, int cols, int* totals,
                      const int* flag) {
  k_radix_rows<<<rows, PIC_WG, 0, s>>>(table, cols, totals, flag);
}

// Tiles of 1024 items until they fill the chip four times over, of 4096 above (a tile's
// digit runs, and so the pieces it writes, are longer).
RadixPlan radix_plan(long long n, int ncells) {
  RadixPlan p;
  int bits = 1;
  while (bits < 31 && (1ll << bits) < ncells) ++bits;
  p.passes = (bits + 7) / 8;
  p.bits = (bits + p.passes - 1) / p.passes;
  p.items = n <= (1ll << 20) ? 4 : 16;
  const long long per = (long long)p.items * PIC_WG;
  p.tiles = (int)((n + per - 1) / per);
  return p;
}

void launch_radix_sort(hipStream_t s, const int* keys, int n, int ncells, const RadixPlan& p,
                       RadixBufs b, int* perm, int* counts, int* offsets) {
  if (p.items == 4) radix_passes<4>(s, keys, n, ncells, p, b, perm, counts, offsets);
  else radix_passes<16>(s, keys, n, ncells, p, b, perm, counts, offsets);
}
