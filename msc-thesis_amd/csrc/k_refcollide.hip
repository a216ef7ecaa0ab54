// k_refcollide.hip -- the reference's own collide arithmetic on an injected uniform stream.
//
// The reference's host collisions draw from one std::mt19937 in particle order:
//   MCC  thesisCode/mccCollisions/src/particle.cc:112-127: r; if prob > r six more draws
//        give v = (2(u1 + u2 + u3 - 1.5), 2(u4 + u5 + u6 - 1.5));
//   DSMC thesisCode/dsmcCollisions/cellTrackerAdvanced/src/main.cc:288-350: the same draws
//        for every particle whose nearest cell partner has a larger index, and the partner
//        gets the opposite velocity.
// Consumer j (a particle that draws) starts at stream position s_j: s_0 = 0 and
// s_{j+1} = s_j + (prob > u[s_j] ? 7 : 1), a sequential chain.  It is resolved in parallel
// as an automaton over the positions: its state is the number of positions still to skip
// (0 .. 6; a consumer starts where it is 0), a stretch of the stream is a map of the 7 states
// at its start to those at its end, and maps compose.
//   k_chain_maps    a chunk of REF_CHAIN_CHUNK positions per workgroup: the map of 16
//                   positions per thread (from their hit bits), scanned over the threads;
//                   per chunk and entry state the exit state and the consumers started
//   k_chain_scan    one workgroup: the chunks' maps scanned, entry state and first consumer
//                   of every chunk
//   k_chain_starts  the thread maps of a chunk again, now from its known entry: the starts
// Bound: launch latency (8 B per position read twice).  On a stream of 700,000 uniforms for
// the DSMC collide of 100,003 particles the three kernels take 8.3 + 5.1 + 8.2 us; they took
// 136 + 489 + 162 us when a thread walked each chunk position by position and one thread
// composed the chunks (the whole call, with the nearest search below: 1107 -> 315 us).
#include "launch.h"

namespace {

#define REF_CHAIN_SEG 16  // positions per thread
static_assert(REF_CHAIN_SEG * PIC_WG == REF_CHAIN_CHUNK, "a chunk is a workgroup's positions");

// Map of the 7 states, three bits each: exit state of state e in bits [3 e, 3 e + 3).
__device__ __forceinline__ unsigned map_then(unsigned f, unsigned g) {  // f, then g
  unsigned h = 0;
#pragma unroll
  for (int e = 0; e < 7; ++e) h |= ((g >> (3 * ((f >> (3 * e)) & 7u))) & 7u) << (3 * e);
  return h;
}
__device__ __forceinline__ unsigned map_identity() {
  unsigned h = 0;
#pragma unroll
  for (int e = 0; e < 7; ++e) h |= (unsigned)e << (3 * e);
  return h;
}

// Consumers started in a segment of len positions (hit bits; none at or past len) entered in
// state e, and the position where the walk leaves it (< len + 7).
__device__ __forceinline__ int seg_walk(unsigned bits, int len, int e, int& pos) {
  int cnt = 0;
  pos = e;
  while (pos < len) {
    const unsigned m = bits >> pos;
    if (!m) {
      cnt += len - pos;
      pos = len;
      break;
    }
    const int q = __builtin_ctz(m);
    cnt += q + 1;
    pos += q + 7;
  }
  return cnt;
}

// Hit bits and length of this thread's segment of chunk j (loads coalesced over the chunk,
// the bits passed through LDS).  words: REF_CHAIN_CHUNK / 64.
__device__ __forceinline__ unsigned chunk_bits(const double* __restrict__ u, long long nu,
                                               double prob, long long j,
                                               unsigned long long* words, int& len) {
  const long long p0 = j * REF_CHAIN_CHUNK;
  double v[REF_CHAIN_SEG];
#pragma unroll
  for (int r = 0; r < REF_CHAIN_SEG; ++r) {
    const long long p = p0 + r * PIC_WG + threadIdx.x;
    v[r] = u[p < nu ? p : nu - 1];
  }
#pragma unroll
  for (int r = 0; r < REF_CHAIN_SEG; ++r) {
    const bool hit = p0 + r * PIC_WG + threadIdx.x < nu && prob > v[r];
    const unsigned long long m = __ballot(hit);
    if ((threadIdx.x & 63) == 0) words[r * (PIC_WG / 64) + (threadIdx.x >> 6)] = m;
  }
  __syncthreads();
  const long long left = nu - (p0 + REF_CHAIN_SEG * threadIdx.x);
  len = left < 0 ? 0 : (left > REF_CHAIN_SEG ? REF_CHAIN_SEG : (int)left);
  return (unsigned)(words[threadIdx.x >> 2] >> ((threadIdx.x & 3) * 16)) & 0xffffu;
}

// map of the segment; cnts: the consumers started per entry state, 5 bits each
__device__ __forceinline__ unsigned seg_map(unsigned bits, int len, unsigned long long& cnts) {
  unsigned f = 0;
  cnts = 0;
#pragma unroll
  for (int e = 0; e < 7; ++e) {
    int pos;
    const int c = seg_walk(bits, len, e, pos);
    cnts |= (unsigned long long)c << (5 * e);
    // the exit of a segment cut by the stream's end is not used (nothing starts after it)
    const int x = pos - REF_CHAIN_SEG;
    f |= (unsigned)(x < 0 ? 0 : x) << (3 * e);
  }
  return f;
}

// Exclusive scan of the threads' maps over the workgroup; *all the map of the whole chunk.
__device__ __forceinline__ unsigned chunk_scan(unsigned f, unsigned* wmap, unsigned* all) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned inc = f;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned t = __shfl_up(inc, o, 64);
    if (lane >= o) inc = map_then(t, inc);
  }
  if (lane == 63) wmap[w] = inc;
  unsigned ex = __shfl_up(inc, 1, 64);
  if (lane == 0) ex = map_identity();
  __syncthreads();
  unsigned pre = map_identity();
#pragma unroll
  for (int k = 0; k < PIC_WG / 64; ++k) {
    if (k == w) ex = map_then(pre, ex);
    pre = map_then(pre, wmap[k]);
  }
  *all = pre;
  return ex;
}

__global__ __launch_bounds__(PIC_WG) void k_chain_maps(const double* __restrict__ u, long long nu,
                                                       double prob, int2* __restrict__ maps) {
  __shared__ unsigned long long words[REF_CHAIN_CHUNK / 64];
  __shared__ unsigned wmap[PIC_WG / 64];
  __shared__ int wcnt[7][PIC_WG / 64];
  int len;
  unsigned long long cnts;
  const unsigned bits = chunk_bits(u, nu, prob, blockIdx.x, words, len);
  unsigned all;
  const unsigned ex = chunk_scan(seg_map(bits, len, cnts), wmap, &all);
#pragma unroll
  for (int e = 0; e < 7; ++e) {
    int c = (int)(cnts >> (5 * ((ex >> (3 * e)) & 7u))) & 31;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) wcnt[e][threadIdx.x >> 6] = c;
  }
  __syncthreads();
  if (threadIdx.x < 7) {
    const int e = threadIdx.x;
    int c = 0;
    for (int k = 0; k < PIC_WG / 64; ++k) c += wcnt[e][k];
    maps[7 * (long long)blockIdx.x + e] = make_int2((int)((all >> (3 * e)) & 7u), c);
  }
}

// One workgroup: entry state and first consumer of every chunk, and the consumers the stream
// starts in total.  A thread composes a run of consecutive chunks, the runs are scanned over
// the threads, and each thread walks its run again from its entry.
__global__ __launch_bounds__(PIC_WG) void k_chain_scan(const int2* __restrict__ maps,
                                                       long long nchunks, int* __restrict__ entry,
                                                       long long* __restrict__ base,
                                                       long long* __restrict__ total) {
  __shared__ unsigned smap[PIC_WG];
  __shared__ long long scnt[7][PIC_WG];
  const long long per = (nchunks + PIC_WG - 1) / PIC_WG;
  const long long j0 = per * threadIdx.x < nchunks ? per * threadIdx.x : nchunks;
  const long long j1 = j0 + per < nchunks ? j0 + per : nchunks;
  unsigned f = map_identity();
  long long c[7] = {0, 0, 0, 0, 0, 0, 0};
  for (long long j = j0; j < j1; ++j) {
    unsigned h = 0;
#pragma unroll
    for (int e = 0; e < 7; ++e) {
      const int2 m = maps[7 * j + ((f >> (3 * e)) & 7u)];
      h |= (unsigned)m.x << (3 * e);
      c[e] += m.y;
    }
    f = h;
  }
  smap[threadIdx.x] = f;
#pragma unroll
  for (int e = 0; e < 7; ++e) scnt[e][threadIdx.x] = c[e];
  __syncthreads();
  for (int o = 1; o < PIC_WG; o <<= 1) {
    const bool has = (int)threadIdx.x >= o;
    const unsigned before = has ? smap[threadIdx.x - o] : 0u;
    long long n[7];
    if (has) {
#pragma unroll
      for (int e = 0; e < 7; ++e)
        n[e] = scnt[e][threadIdx.x - o] + scnt[(before >> (3 * e)) & 7u][threadIdx.x];
    }
    const unsigned mine = smap[threadIdx.x];
    __syncthreads();
    if (has) {
      smap[threadIdx.x] = map_then(before, mine);
#pragma unroll
      for (int e = 0; e < 7; ++e) scnt[e][threadIdx.x] = n[e];
    }
    __syncthreads();
  }
  int e = threadIdx.x ? (int)(smap[threadIdx.x - 1] & 7u) : 0;
  long long b = threadIdx.x ? scnt[0][threadIdx.x - 1] : 0;
  for (long long j = j0; j < j1; ++j) {
    entry[j] = e;
    base[j] = b;
    const int2 m = maps[7 * j + e];
    e = m.x;
    b += m.y;
  }
  if (threadIdx.x == PIC_WG - 1) *total = scnt[0][PIC_WG - 1];
}

__global__ __launch_bounds__(PIC_WG) void k_chain_starts(const double* __restrict__ u,
                                                         long long nu, double prob,
                                                         const int* __restrict__ entry,
                                                         const long long* __restrict__ base,
                                                         long long m,
                                                         long long* __restrict__ start) {
  __shared__ unsigned long long words[REF_CHAIN_CHUNK / 64];
  __shared__ unsigned wmap[PIC_WG / 64];
  __shared__ int wsum[PIC_WG / 64];
  const long long j = blockIdx.x;
  if (base[j] >= m) return;  // uniform: every consumer started before this chunk
  int len;
  unsigned long long cnts;
  const unsigned bits = chunk_bits(u, nu, prob, j, words, len);
  unsigned all;
  const unsigned ex = chunk_scan(seg_map(bits, len, cnts), wmap, &all);
  const int e = (int)((ex >> (3 * entry[j])) & 7u);
  const int c = (int)(cnts >> (5 * e)) & 31;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int inc = c;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  long long idx = base[j] + inc - c;
  for (int k = 0; k < w; ++k) idx += wsum[k];
  const long long p0 = j * REF_CHAIN_CHUNK + REF_CHAIN_SEG * (int)threadIdx.x;
  for (int pos = e; pos < len && idx < m; pos += ((bits >> pos) & 1u) ? 7 : 1)
    start[idx++] = p0 + pos;
}

// uniforms taken by the first m consumers (last start + its draws), or -1 when the stream
// cannot serve them all
__global__ void k_chain_consumed(const double* __restrict__ u, long long nu, double prob,
                                 const long long* __restrict__ start,
                                 const long long* __restrict__ total, long long m,
                                 long long* __restrict__ consumed) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  if (m == 0) { *consumed = 0; return; }
  if (*total < m) { *consumed = -1; return; }
  const long long s = start[m - 1];
  const long long e = s + ((prob > u[s]) ? 7 : 1);
  *consumed = e <= nu ? e : -1;
}

// Bird's approximate unit normal of the reference, 2*(U1 + U2 + U3 - 1.5), left to right
__device__ __forceinline__ double bird_normal(const double* u) {
  return 2.0 * (u[0] + u[1] + u[2] - 1.5);
}

__global__ __launch_bounds__(PIC_WG) void k_mcc_reference(double* __restrict__ vx,
                                                          double* __restrict__ vy, long long n,
                                                          double prob,
                                                          const double* __restrict__ u,
                                                          const long long* __restrict__ start) {
  for (long long i = blockIdx.x * (long long)PIC_WG + threadIdx.x; i < n;
       i += (long long)gridDim.x * PIC_WG) {
    const long long s = start[i];
    if (prob > u[s]) {
      vx[i] = bird_normal(u + s + 1);
      vy[i] = bird_normal(u + s + 4);
    }
  }
}

__global__ __launch_bounds__(PIC_WG) void k_ref_cell_keys(const double* __restrict__ x,
                                                          const double* __restrict__ y,
                                                          long long n, int nx, int ny,
                                                          double dx, double dy,
                                                          int* __restrict__ keys,
                                                          int* __restrict__ bad) {
  for (long long i = blockIdx.x * (long long)PIC_WG + threadIdx.x; i < n;
       i += (long long)gridDim.x * PIC_WG) {
    const double tx = x[i] / dx, ty = y[i] / dy;
    // (int)(x/dx) as the reference's Particle keeps it; outside the grid is an input error
    if (!(tx >= 0.0 && tx < (double)nx && ty >= 0.0 && ty < (double)ny)) {
      atomicOr(bad, 1);
      keys[i] = 0;
      continue;
    }
    keys[i] = (int)tx * ny + (int)ty;
  }
}

// Nearest other particle of the cell (cell lists in ascending particle index), strictly
// smaller distance wins (the first found on ties), initial bound 1e8; kept only when its
// index is larger, else -1.  valid[i] = 0 for a drawing particle, 1 otherwise (sort key).
// A thread per slot of the cell lists, so that the lanes of a wave share their cells' loads
// (100,003 particles, 24 per cell: 41 -> 24 us).
// The square root is taken only of a square below that of the nearest so far: rounding keeps
// its order, so no other can be strictly nearer.
__global__ __launch_bounds__(PIC_WG) void k_ref_nearest(const double* __restrict__ x,
                                                        const double* __restrict__ y,
                                                        long long n,
                                                        const int* __restrict__ keys,
                                                        const int* __restrict__ perm,
                                                        const int* __restrict__ offsets,
                                                        int* __restrict__ target,
                                                        int* __restrict__ drawkey) {
  for (long long slot = blockIdx.x * (long long)PIC_WG + threadIdx.x; slot < n;
       slot += (long long)gridDim.x * PIC_WG) {
    const int i = perm[slot];
    const int c = keys[i];
    const double xi = x[i], yi = y[i];
    double nearest = 1e8, nearest2 = 1e16;  // sqrt(1e16) is 1e8 exactly
    int t = -1;
    for (int s = offsets[c]; s < offsets[c + 1]; ++s) {
      const int q = perm[s];
      if (q == i) continue;
      const double ddx = xi - x[q], ddy = yi - y[q];
      const double d2 = ddx * ddx + ddy * ddy;
      if (d2 < nearest2) {
        const double d = sqrt(d2);
        if (d < nearest) {
          nearest = d;
          nearest2 = d2;
          t = q;
        }
      }
    }
    if (t < i) t = -1;
    target[i] = t;
    drawkey[i] = t >= 0 ? 0 : 1;
  }
}

// consumer j = the j-th drawing particle: draw, and record the pair's reset velocity
__global__ __launch_bounds__(PIC_WG) void k_dsmc_reference_draw(
    long long m, double prob, const double* __restrict__ u, const long long* __restrict__ start,
    const int* __restrict__ consumers, const int* __restrict__ target, double* __restrict__ m1,
    double* __restrict__ m2, int* __restrict__ self, int* __restrict__ lastw,
    unsigned long long* __restrict__ ncoll) {
  unsigned int acc = 0;
  for (long long j = blockIdx.x * (long long)PIC_WG + threadIdx.x; j < m;
       j += (long long)gridDim.x * PIC_WG) {
    const long long s = start[j];
    if (prob > u[s]) {
      const int i = consumers[j];
      m1[j] = bird_normal(u + s + 1);
      m2[j] = bird_normal(u + s + 4);
      self[i] = (int)j;
      atomicMax(&lastw[target[i]], (int)j);
      ++acc;
    }
  }
  // one atomic per wave (one per thread serialised thousands on the single address)
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0 && acc) atomicAdd(ncoll, (unsigned long long)acc);
}

// The reference writes v_i and then v_target for i = 0, 1, ...: a particle's last write is
// its own draw when it has one (its partners all have smaller indices), else the draw of
// the largest index that chose it as partner (opposite velocity).
__global__ __launch_bounds__(PIC_WG) void k_dsmc_reference_apply(
    double* __restrict__ vx, double* __restrict__ vy, long long n, const double* __restrict__ m1,
    const double* __restrict__ m2, const int* __restrict__ self, const int* __restrict__ lastw) {
  for (long long p = blockIdx.x * (long long)PIC_WG + threadIdx.x; p < n;
       p += (long long)gridDim.x * PIC_WG) {
    const int j = self[p];
    if (j >= 0) {
      vx[p] = m1[j];
      vy[p] = m2[j];
    } else if (lastw[p] >= 0) {
      vx[p] = -m1[lastw[p]];
      vy[p] = -m2[lastw[p]];
    }
  }
}

inline int grid_of(long long n) {
  long long b = (n + PIC_WG - 1) / PIC_WG;
  return (int)(b < 1 ? 1 : (b > 16384 ? 16384 : b));
}

}  // namespace

void launch_ref_chain(hipStream_t s, const double* u, long long nu, double prob, long long m,
                      RefChainBufs b) {
  const long long nv = ref_chain_stream(nu, m);
  const long long nchunks = (nv + REF_CHAIN_CHUNK - 1) / REF_CHAIN_CHUNK;
  if (nchunks > 0) k_chain_maps<<<(unsigned)nchunks, PIC_WG, 0, s>>>(u, nv, prob, b.maps);
  k_chain_scan<<<1, PIC_WG, 0, s>>>(b.maps, nchunks, b.entry, b.base, b.total);
  if (nchunks > 0)
    k_chain_starts<<<(unsigned)nchunks, PIC_WG, 0, s>>>(u, nv, prob, b.entry, b.base, m, b.start);
  k_chain_consumed<<<1, 64, 0, s>>>(u, nu, prob, b.start, b.total, m, b.consumed);
}

void launch_mcc_reference(hipStream_t s, double* vx, double* vy, long long n, double prob,
                          const double* u, const long long* start) {
  if (n > 0) k_mcc_reference<<<grid_of(n), PIC_WG, 0, s>>>(vx, vy, n, prob, u, start);
}

void launch_ref_cell_keys(hipStream_t s, const double* x, const double* y, long long n, int nx,
                          int ny, double dx, double dy, int* keys, int* bad) {
  if (n > 0) k_ref_cell_keys<<<grid_of(n), PIC_WG, 0, s>>>(x, y, n, nx, ny, dx, dy, keys, bad);
}

void launch_ref_nearest(hipStream_t s, const double* x, const double* y, long long n,
                        const int* keys, const int* perm, const int* offsets, int* target,
                        int* drawkey) {
  if (n > 0)
    k_ref_nearest<<<grid_of(n), PIC_WG, 0, s>>>(x, y, n, keys, perm, offsets, target, drawkey);
}

void launch_dsmc_reference(hipStream_t s, double* vx, double* vy, long long n, long long m,
                           double prob, const double* u, const long long* start,
                           const int* consumers, const int* target, double* m1, double* m2,
                           int* self, int* lastw, unsigned long long* ncoll) {
  if (m > 0)
    k_dsmc_reference_draw<<<grid_of(m), PIC_WG, 0, s>>>(m, prob, u, start, consumers, target, m1,
                                                        m2, self, lastw, ncoll);
  if (n > 0) k_dsmc_reference_apply<<<grid_of(n), PIC_WG, 0, s>>>(vx, vy, n, m1, m2, self, lastw);
}
