// k_adjoint.hip -- reverse-mode (adjoint) kernels of the collisionless step.
//
// Forward step k (no reference counterpart; it is the reference step of
// thesisCode/collisionless/double/src/main.cc:137-172 written as a map):
//   rho_k = D(x_k)                         CIC deposit, charge qp per particle
//   E_k   = M rho_k                        spectral Poisson + central-difference symbol
//   v_{k+1/2} = v_{k-1/2} + c_k dt qm G(x_k) E_k      (c_0 = 1/2 from synchronous v_0)
//   x_{k+1}   = x_k + dt v_{k+1/2}
// Loss L = sum |E_N|^2 dx dy.  Reverse step k (lambda_x, lambda_v = dL/dx, dL/dv):
//   lv' = lv + dt lx                                   (drift)
//   lE  = c_k dt qm sum_p W(x_p) lv'_p                 (gather is the transpose of deposit)
//   lrho = M^T lE                                      (conjugate Fourier symbols)
//   lx += c_k dt qm (grad W . E_k) lv' + (qp/dA) grad W . lrho
// The CIC weights are piecewise bilinear; their derivatives are taken on the continuous
// fractions (the fixed-point quantisation of the forward weights is below 2^-18 of a cell).
#include <type_traits>
#include "fft_lds.h"
#include "deposit.h"
#include "launch.h"
#include "adjoint_launch.h"

namespace {

#define ADJ_NT 1024  // threads per workgroup of the windowed kernels

template <typename R>
using R2T = typename std::conditional<sizeof(R) == 4, float2, double2>::type;

template <typename R>
__device__ __forceinline__ Geo<R> geo_of(const AdjGrid& g) {
  return make_geo<R>(g.nx, g.ny, g.lx, g.ly);
}

// two neighbouring nodes (j, j + 1) of a padded field as one piece
template <typename R>
__device__ __forceinline__ void load_pair(const R2T<R>* e, R2T<R> r[2]) {
  __builtin_memcpy(r, e, 2 * sizeof(R2T<R>));
}

// x0 = xl + sum_m a_m cos(kx_m xl + ky_m yl) (wrapped), y0 = yl; deposits x0's charge
// unless hi is NULL
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_adj_init(AdjGrid g, const double* __restrict__ xl,
                                                     const double* __restrict__ yl, int64_t n,
                                                     const double* __restrict__ amps,
                                                     const double* __restrict__ mkx,
                                                     const double* __restrict__ mky, int nm,
                                                     R* __restrict__ x, R* __restrict__ y,
                                                     unsigned long long* hi,
                                                     unsigned long long* lo) {
  const Geo<R> q = geo_of<R>(g);
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * PIC_WG) {
    const double a = xl[p], b = yl[p];
    double d = 0.0;
    for (int m = 0; m < nm; ++m) d += amps[m] * cos(mkx[m] * a + mky[m] * b);
    const R xr = wrap_pos((R)wrap_pos(a + d, g.lx), (R)g.lx);
    const R yr = (R)b;
    x[p] = xr;
    y[p] = yr;
    if (hi) {
      int cx, cy;
      long long w[4];
      deposit_weights<R>(xr, yr, q, cx, cy, w);
      deposit_global<R>(hi, lo, cx, cy, w, q);
    }
  }
}

// The pushes of a segment from its checkpoint, for the reverse sweep: the fields of its steps
// are stored, so a particle's steps need nothing of the others and one thread takes them all
// in a row, its state in registers.  Writes the positions after step k0 + 1, ..., k0 + nst
// (xs, ys: n per step); per step the arithmetic is that of k_adj_push_win.  Bound: the latency
// of the steps' dependent gathers.  128^2, 524,288 particles, 10 steps: one launch of 19 us
// where a restore and ten launches of a push took 62.
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_adj_segment(AdjGrid g, const R* __restrict__ ck,
                                                        const R* __restrict__ Eseg,
                                                        long long estride, int k0, int nst,
                                                        R* __restrict__ xs, R* __restrict__ ys,
                                                        int64_t n) {
  const Geo<R> q = geo_of<R>(g);
  const R Lx = (R)g.lx, Ly = (R)g.ly, dtr = (R)g.dt;
  const R qs = (R)(1.0 / (double)(1 << Fix<R>::QB));
  const int ny1 = g.ny + 1;
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * PIC_WG) {
    R xr = ck[p], yr = ck[n + p], vxr = ck[2 * n + p], vyr = ck[3 * n + p];
    for (int k = 0; k < nst; ++k) {
      const R2T<R>* E = reinterpret_cast<const R2T<R>*>(Eseg + k * estride);
      const R hk = (R)((k0 + k == 0 ? 0.5 : 1.0) * g.dt * g.qm);
      int cx, cy;
      R fx, fy;
      locate_w(xr, q.idx, g.nx, cx, fx);
      locate_w(yr, q.idy, g.ny, cy, fy);
      const R gx1 = (R)qweight(fx) * qs, gy1 = (R)qweight(fy) * qs;
      const R gx0 = (R)1 - gx1, gy0 = (R)1 - gy1;
      R2T<R> r0[2], r1[2];
      load_pair<R>(E + cx * ny1 + cy, r0);
      load_pair<R>(E + (cx + 1) * ny1 + cy, r1);
      R epx = (gx0 * gy0) * r0[0].x;
      epx = epx + (gx1 * gy0) * r1[0].x;
      epx = epx + (gx0 * gy1) * r0[1].x;
      epx = epx + (gx1 * gy1) * r1[1].x;
      R epy = (gx0 * gy0) * r0[0].y;
      epy = epy + (gx1 * gy0) * r1[0].y;
      epy = epy + (gx0 * gy1) * r0[1].y;
      epy = epy + (gx1 * gy1) * r1[1].y;
      vxr = vxr + hk * epx;
      vyr = vyr + hk * epy;
      xr = wrap_pos((R)(xr + dtr * vxr), Lx);
      yr = wrap_pos((R)(yr + dtr * vyr), Ly);
      xs[k * n + p] = xr;
      ys[k * n + p] = yr;
    }
  }
}

__global__ __launch_bounds__(PIC_WG) void k_adj_zero(double* __restrict__ a, long long n) {
  for (long long q = blockIdx.x * (long long)PIC_WG + threadIdx.x; q < n;
       q += (long long)gridDim.x * PIC_WG)
    a[q] = 0.0;
}

// Constants of the reverse passes, the reciprocals rounded once.
template <typename R>
struct CicGeo {
  R dxr, dyr, rdx, rdy;              // cell sides in R and their reciprocals
  double ix, iy;                     // 1 / dx, 1 / dy
};
template <typename R>
__device__ __forceinline__ CicGeo<R> cic_geo(const AdjGrid& g) {
  CicGeo<R> c;
  c.dxr = (R)g.dx; c.dyr = (R)g.dy;
  c.rdx = (R)1 / c.dxr; c.rdy = (R)1 / c.dyr;
  c.ix = 1.0 / g.dx; c.iy = 1.0 / g.dy;
  return c;
}

// x / d with inv = 1 / d correctly rounded: one Newton step on the quotient (Markstein's
// division) gives the correctly rounded quotient in three operations instead of a division
// sequence per coordinate.
template <typename R>
__device__ __forceinline__ R div_by(R x, R d, R inv) {
  const R q = x * inv;
  return fmar(fmar(-q, d, x), inv, q);
}

// Continuous CIC fractions at x in double arithmetic; the cell is (int)(x / dx) in R, clamped.
struct CicD {
  int cx, cy;
  double fx, fy;
};

template <typename R>
__device__ __forceinline__ CicD cic_d(R xr, R yr, const AdjGrid& g, const CicGeo<R>& q) {
  CicD r;
  int cx = (int)div_by<R>(xr, q.dxr, q.rdx), cy = (int)div_by<R>(yr, q.dyr, q.rdy);
  cx = cx > g.nx - 1 ? g.nx - 1 : cx;
  cy = cy > g.ny - 1 ? g.ny - 1 : cy;
  r.cx = cx < 0 ? 0 : cx;
  r.cy = cy < 0 ? 0 : cy;
  const double fx = div_by<double>((double)xr, g.dx, q.ix) - r.cx;
  const double fy = div_by<double>((double)yr, g.dy, q.iy) - r.cy;
  r.fx = fx < 0 ? 0 : (fx > 1 ? 1 : fx);
  r.fy = fy < 0 ? 0 : (fy > 1 ? 1 : fy);
  return r;
}

// gradient of the CIC interpolation of node values f00, f10, f01, f11
__device__ __forceinline__ void cic_grad(const CicD& c, double ix, double iy, double f00,
                                         double f10, double f01, double f11, double& gx,
                                         double& gy) {
  gx = (-(1 - c.fy) * ix) * f00;
  gx += ((1 - c.fy) * ix) * f10;
  gx += (-c.fy * ix) * f01;
  gx += (c.fy * ix) * f11;
  gy = (-(1 - c.fx) * iy) * f00;
  gy += (-c.fx * iy) * f10;
  gy += ((1 - c.fx) * iy) * f01;
  gy += (c.fx * iy) * f11;
}

// gradient of the padded sensitivity lrho at a position
template <typename R>
__device__ __forceinline__ void lrho_grad(const double* __restrict__ lrho, R xr, R yr,
                                          const AdjGrid& g, const CicGeo<R>& q, double& sx,
                                          double& sy) {
  const CicD c = cic_d<R>(xr, yr, g, q);
  double r0[2], r1[2];
  const double* l = lrho + c.cx * (g.ny + 1) + c.cy;
  __builtin_memcpy(r0, l, sizeof(r0));
  __builtin_memcpy(r1, l + g.ny + 1, sizeof(r1));
  cic_grad(c, q.ix, q.iy, r0[0], r1[0], r0[1], r1[1], sx, sy);
}

// Deposit Jacobian of step 0 at x_0, which ends the reverse sweep.
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_adj_pass_end(AdjGrid g, const R* __restrict__ xk,
                                                         const R* __restrict__ yk,
                                                         const double* __restrict__ lrho,
                                                         double cq, double* __restrict__ lx,
                                                         double* __restrict__ ly, int64_t n) {
  const CicGeo<R> q = cic_geo<R>(g);
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * PIC_WG) {
    double sx, sy;
    lrho_grad<R>(lrho, xk[p], yk[p], g, q, sx, sy);
    lx[p] = lx[p] + cq * sx;
    ly[p] = ly[p] + cq * sy;
  }
}

// ---- windowed forms.  The particles are counting-sorted by tile at every checkpoint
// (stable, with their original indices), so within a segment the particles of a push item
// stay near its tile: the field is read from an LDS window of the tile + halo, and the
// deposits (int64 charge forward, FP64 E sensitivity in reverse) are summed in an LDS
// window and flushed with one global atomic per touched node.  Particles that drifted out
// of the window since the checkpoint use the global arrays directly.  The flush costs a global
// atomic per touched node and item, so an item keeps about 2048 particles and gets ADJ_NT
// threads for them: at 128^2 and 524,288 particles there is one item per CU, and 256 threads
// of eight particles each left its latencies exposed (push 15.7 -> 9.8 us; the reverse pass,
// with its divisions and index arithmetic cut as well, 21.7 -> 12.3).

// item {tile x, tile y, split} -> particle range [f0, f1) and window origin
__device__ __forceinline__ void adj_item(const AdjGrid& g, const int4 it,
                                         const int* __restrict__ toff, int& f0, int& f1,
                                         int& x0, int& y0) {
  const int tb = it.x * g.tiles_y + it.y;
  const long long s0 = toff[tb], F = toff[tb + 1] - s0;
  f0 = (int)(s0 + F * it.z / g.splits);
  f1 = (int)(s0 + F * (it.z + 1) / g.splits);
  x0 = it.x * g.tile - g.halo;
  y0 = it.y * g.tile - g.halo;
}

// The state is read from (xi, yi, vxi, vyi) and written to (xo, yo, vxo, vyo), which may be the
// same arrays.  PUSH = false: deposit the charge of the positions as they are (no field, no
// motion).
template <typename R, bool PUSH>
__global__ __launch_bounds__(ADJ_NT) void k_adj_push_win(AdjGrid g,
                                                         const int4* __restrict__ items,
                                                         const int* __restrict__ toff,
                                                         const R* xi, const R* yi,
                                                         const R* vxi, const R* vyi, R* xo,
                                                         R* yo, R* vxo, R* vyo,
                                                         const R* __restrict__ Epad, double c,
                                                         unsigned long long* hi,
                                                         unsigned long long* lo) {
  extern __shared__ unsigned long long wsh[];
  const int W = g.win, nw = W * W;
  constexpr int NQ = (sizeof(R) == 8) ? 2 : 1;  // int64 words per node (hi, lo)
  unsigned long long* whi = wsh;
  unsigned long long* wlo = wsh + nw;            // FP64 particles only
  R2T<R>* ew = reinterpret_cast<R2T<R>*>(wsh + NQ * nw);
  int f0, f1, x0, y0;
  adj_item(g, items[blockIdx.x], toff, f0, f1, x0, y0);
  const int ny1 = g.ny + 1;
  const R2T<R>* E = reinterpret_cast<const R2T<R>*>(Epad);
  for (int i = threadIdx.x; i < NQ * nw; i += ADJ_NT) wsh[i] = 0ull;
  if (PUSH)
    for (int i = threadIdx.x; i < nw; i += ADJ_NT) {
      const int r = i / W, cc = i - r * W;
      ew[i] = E[(long long)pwrap(x0 + r, g.nx) * ny1 + pwrap(y0 + cc, g.ny)];
    }
  __syncthreads();
  const Geo<R> q = geo_of<R>(g);
  const R Lx = (R)g.lx, Ly = (R)g.ly;
  const R hk = (R)(c * g.dt * g.qm), dtr = (R)g.dt;
  const R qs = (R)(1.0 / (double)(1 << Fix<R>::QB));
  for (int p = f0 + threadIdx.x; p < f1; p += ADJ_NT) {
    R xr = xi[p], yr = yi[p];
    int cx, cy, rx, ry;
    if (PUSH) {
      R vxr = vxi[p], vyr = vyi[p];
      R fx, fy;
      locate_w(xr, q.idx, g.nx, cx, fx);
      locate_w(yr, q.idy, g.ny, cy, fy);
      const R gx1 = (R)qweight(fx) * qs, gy1 = (R)qweight(fy) * qs;
      const R gx0 = (R)1 - gx1, gy0 = (R)1 - gy1;
      R2T<R> e00, e01, e10, e11;
      rx = pwrap(cx - x0, g.nx);
      ry = pwrap(cy - y0, g.ny);
      if (rx < W - 1 && ry < W - 1) {
        const int i0 = rx * W + ry;
        e00 = ew[i0]; e01 = ew[i0 + 1]; e10 = ew[i0 + W]; e11 = ew[i0 + W + 1];
      } else {
        const long long i00 = (long long)cx * ny1 + cy;
        e00 = E[i00]; e01 = E[i00 + 1]; e10 = E[i00 + ny1]; e11 = E[i00 + ny1 + 1];
      }
      R epx = (gx0 * gy0) * e00.x;
      epx = epx + (gx1 * gy0) * e10.x;
      epx = epx + (gx0 * gy1) * e01.x;
      epx = epx + (gx1 * gy1) * e11.x;
      R epy = (gx0 * gy0) * e00.y;
      epy = epy + (gx1 * gy0) * e10.y;
      epy = epy + (gx0 * gy1) * e01.y;
      epy = epy + (gx1 * gy1) * e11.y;
      vxr = vxr + hk * epx;
      vyr = vyr + hk * epy;
      xr = wrap_pos((R)(xr + dtr * vxr), Lx);
      yr = wrap_pos((R)(yr + dtr * vyr), Ly);
      xo[p] = xr;
      yo[p] = yr;
      vxo[p] = vxr;
      vyo[p] = vyr;
    }
    long long w[4];
    deposit_weights<R>(xr, yr, q, cx, cy, w);
    rx = pwrap(cx - x0, g.nx);
    ry = pwrap(cy - y0, g.ny);
    if (rx < W - 1 && ry < W - 1) {
      const int i0 = rx * W + ry;
      const int off[4] = {0, W, 1, W + 1};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (sizeof(R) == 8) {
          atomicAdd(&whi[i0 + off[k]], (unsigned long long)(w[k] >> 30));
          atomicAdd(&wlo[i0 + off[k]], (unsigned long long)(w[k] & ((1ll << 30) - 1)));
        } else {
          atomicAdd(&whi[i0 + off[k]], (unsigned long long)w[k]);
        }
      }
    } else {
      deposit_global<R>(hi, lo, cx, cy, w, q);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nw; i += ADJ_NT) {
    const unsigned long long v = whi[i];
    const unsigned long long vl = (sizeof(R) == 8) ? wlo[i] : 0ull;
    if (v | vl) {
      const int r = i / W, cc = i - r * W;
      const long long nd = (long long)pwrap(x0 + r, g.nx) * g.ny + pwrap(y0 + cc, g.ny);
      if (v) atomicAdd(&hi[nd], v);
      if (sizeof(R) == 8 && vl) atomicAdd(&lo[nd], vl);
    }
  }
}

// Fused reverse pass: finish step k (deposit Jacobian at x_k with lrho_k), then start step
// k-1: drift, deposit of lv' into lE (scaled by ck1), kick Jacobian at x_{k-1} with the field
// E_{k-1}.
template <typename R>
__global__ __launch_bounds__(ADJ_NT) void k_adj_pass_win(AdjGrid g,
                                                         const int4* __restrict__ items,
                                                         const int* __restrict__ toff,
                                                         const R* __restrict__ xk,
                                                         const R* __restrict__ yk,
                                                         const double* __restrict__ lrho,
                                                         double cq, const R* __restrict__ xp,
                                                         const R* __restrict__ yp,
                                                         const R* __restrict__ Eprev,
                                                         double ck1, double* __restrict__ lx,
                                                         double* __restrict__ ly,
                                                         double* __restrict__ lvx,
                                                         double* __restrict__ lvy,
                                                         double* __restrict__ lE) {
  extern __shared__ double wl[];  // E sensitivity window: x components, then y
  const int W = g.win, nw = W * W;
  const int G = g.nx * g.ny;
  int f0, f1, x0, y0;
  adj_item(g, items[blockIdx.x], toff, f0, f1, x0, y0);
  const CicGeo<R> q = cic_geo<R>(g);
  for (int i = threadIdx.x; i < 2 * nw; i += ADJ_NT) wl[i] = 0.0;
  __syncthreads();
  const R2T<R>* E = reinterpret_cast<const R2T<R>*>(Eprev);
  const int ny1 = g.ny + 1;
  for (int p = f0 + threadIdx.x; p < f1; p += ADJ_NT) {
    double ax = lx[p], ay = ly[p], bx = lvx[p], by = lvy[p];
    const R xpr = xp[p], ypr = yp[p];
    // the field at x_{k-1} does not wait for the sensitivity at x_k
    const CicD c = cic_d<R>(xpr, ypr, g, q);
    R2T<R> r0[2], r1[2];
    load_pair<R>(E + c.cx * ny1 + c.cy, r0);
    load_pair<R>(E + (c.cx + 1) * ny1 + c.cy, r1);
    double sx, sy;
    lrho_grad<R>(lrho, xk[p], yk[p], g, q, sx, sy);
    ax += cq * sx;
    ay += cq * sy;
    bx = bx + g.dt * ax;
    by = by + g.dt * ay;
    double exx, exy, eyx, eyy;
    cic_grad(c, q.ix, q.iy, (double)r0[0].x, (double)r1[0].x, (double)r0[1].x, (double)r1[1].x,
             exx, exy);
    cic_grad(c, q.ix, q.iy, (double)r0[0].y, (double)r1[0].y, (double)r0[1].y, (double)r1[1].y,
             eyx, eyy);
    const double w[4] = {(1 - c.fx) * (1 - c.fy), c.fx * (1 - c.fy), (1 - c.fx) * c.fy,
                         c.fx * c.fy};
    const int rx = pwrap(c.cx - x0, g.nx), ry = pwrap(c.cy - y0, g.ny);
    if (rx < W - 1 && ry < W - 1) {
      const int i0 = rx * W + ry;
      const int off[4] = {0, W, 1, W + 1};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        atomicAdd(&wl[i0 + off[k]], ck1 * w[k] * bx);
        atomicAdd(&wl[nw + i0 + off[k]], ck1 * w[k] * by);
      }
    } else {
      const int cxp = pwrap(c.cx + 1, g.nx), cyp = pwrap(c.cy + 1, g.ny);
      const int nd[4] = {c.cx * g.ny + c.cy, cxp * g.ny + c.cy, c.cx * g.ny + cyp,
                         cxp * g.ny + cyp};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        atomicAdd(&lE[nd[k]], ck1 * w[k] * bx);
        atomicAdd(&lE[G + nd[k]], ck1 * w[k] * by);
      }
    }
    ax += ck1 * (bx * exx + by * eyx);
    ay += ck1 * (bx * exy + by * eyy);
    lvx[p] = bx;
    lvy[p] = by;
    lx[p] = ax;
    ly[p] = ay;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nw; i += ADJ_NT) {
    const double sx = wl[i], sy = wl[nw + i];
    if (sx != 0.0 || sy != 0.0) {
      const int r = i / W, cc = i - r * W;
      const int nd = pwrap(x0 + r, g.nx) * g.ny + pwrap(y0 + cc, g.ny);
      if (sx != 0.0) atomicAdd(&lE[nd], sx);
      if (sy != 0.0) atomicAdd(&lE[G + nd], sy);
    }
  }
}

// four particle arrays into the order before a sort: b[k][from[d]] = a[k][d]
__global__ __launch_bounds__(PIC_WG) void k_adj_reorder(const int* __restrict__ from,
                                                        const double* __restrict__ a,
                                                        double* __restrict__ b, int64_t n) {
  for (int64_t d = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; d < n;
       d += (int64_t)gridDim.x * PIC_WG) {
    const int64_t o = from[d];
#pragma unroll
    for (int k = 0; k < 4; ++k) b[k * n + o] = a[k * n + d];
  }
}

// lE = s * E (unpadded FP64 two-component array from the padded field)
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_adj_seed(AdjGrid g, const R* __restrict__ Epad,
                                                     double s, double* __restrict__ lE) {
  const int G = g.nx * g.ny;
  const R2T<R>* E = reinterpret_cast<const R2T<R>*>(Epad);
  for (int q = blockIdx.x * PIC_WG + threadIdx.x; q < G; q += gridDim.x * PIC_WG) {
    const int i = q / g.ny, j = q % g.ny;
    const R2T<R> e = E[(long long)i * (g.ny + 1) + j];
    lE[q] = s * (double)e.x;
    lE[G + q] = s * (double)e.y;
  }
}

// sum over nodes of Ex^2 + Ey^2 (block partials; the host adds them in order)
template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_adj_energy(AdjGrid g, const R* __restrict__ Epad,
                                                       double* __restrict__ part) {
  __shared__ double red[4];
  const int G = g.nx * g.ny;
  const R2T<R>* E = reinterpret_cast<const R2T<R>*>(Epad);
  double s = 0.0;
  for (int q = blockIdx.x * PIC_WG + threadIdx.x; q < G; q += gridDim.x * PIC_WG) {
    const int i = q / g.ny, j = q % g.ny;
    const R2T<R> e = E[(long long)i * (g.ny + 1) + j];
    s += (double)e.x * (double)e.x + (double)e.y * (double)e.y;
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// ---- M^T by a complex 2D FFT of the packed pair z = lEx + i lEy
// rows: z[i][j] -> A[k][i] = FFT_y(z[i])[k]  (transposed, all k)
// (lE is zeroed as it is read, ready for the next reverse deposit)
__global__ __launch_bounds__(PIC_WG) void k_adj_rows_fwd(AdjGrid g, double* __restrict__ lE,
                                                         double2* __restrict__ A,
                                                         const double2* __restrict__ tw) {
  extern __shared__ double2 s[];
  const int i = xcd_item(blockIdx.x, gridDim.x), ny = g.ny, G = g.nx * g.ny;
  for (int j = threadIdx.x; j < ny; j += PIC_WG) {
    s[bitrev(j, g.logny)] = make_double2(lE[i * ny + j], lE[G + i * ny + j]);
    lE[i * ny + j] = 0.0;
    lE[G + i * ny + j] = 0.0;
  }
  __syncthreads();
  fft_lds(s, ny, g.logny, -1, tw);
  for (int k = threadIdx.x; k < ny; k += PIC_WG) A[(long long)k * g.nx + i] = s[k];
}

// columns k and k' = -k: FFT_x, unpack lEx_hat / lEy_hat, apply the conjugate symbols,
// inverse FFT_x; writes R_hat columns back into A.
__global__ __launch_bounds__(PIC_WG) void k_adj_cols(AdjGrid g, double2* __restrict__ A,
                                                     const double2* __restrict__ tw) {
  extern __shared__ double2 s[];
  const int nx = g.nx, ny = g.ny;
  const int k = blockIdx.x;            // 0 .. ny/2
  const int k2 = (ny - k) & (ny - 1);  // partner column
  double2* a = s;                      // column k
  double2* b = s + nx;                 // column k2
  double2* ra = s + 2 * nx;
  double2* rb = s + 3 * nx;
  double2* twl = s + 4 * nx;           // the transform's nx/2 twiddles
  fft_stage_twiddles(twl, nx, tw);
  for (int i = threadIdx.x; i < nx; i += PIC_WG) {
    a[bitrev(i, g.lognx)] = A[(long long)k * nx + i];
    b[bitrev(i, g.lognx)] = A[(long long)k2 * nx + i];
  }
  __syncthreads();
  fft_lds_rows(a, 2, nx, g.lognx, -1, twl, g.lognx);  // a, b consecutive
  const double twopi = 6.283185307179586476925;
  for (int m = threadIdx.x; m < nx; m += PIC_WG) {
    const int m2 = (nx - m) & (nx - 1);
    const int mm = (2 * m < nx) ? m : m - nx;
    const double kxv = twopi * mm / g.lx;
    const double sx = sin2pi_frac(m, nx, twl, g.lognx) / g.dx;
    for (int side = 0; side < 2; ++side) {
      const int kk = side ? k2 : k;
      const double2 zk = side ? b[m] : a[m];      // Z(m, kk)
      const double2 zc = side ? a[m2] : b[m2];    // Z(-m, -kk)
      const double2 hx = make_double2(0.5 * (zk.x + zc.x), 0.5 * (zk.y - zc.y));
      const double2 hy = make_double2(0.5 * (zk.y + zc.y), -0.5 * (zk.x - zc.x));
      const int kw = (2 * kk < ny) ? kk : kk - ny;
      const double kyv = twopi * kw / g.ly;
      const double sy = sin2pi_frac(kk, ny, tw) / g.dy;
      const double k2v = kxv * kxv + kyv * kyv;
      const double gr = (m == 0 && kk == 0) ? 0.0 : 1.0 / k2v;
      // R = i gr (sx hx + sy hy)
      const double re = sx * hx.x + sy * hy.x, im = sx * hx.y + sy * hy.y;
      const double2 r = make_double2(-gr * im, gr * re);
      (side ? rb : ra)[bitrev(m, g.lognx)] = r;
    }
  }
  __syncthreads();
  fft_lds_rows(ra, 2, nx, g.lognx, +1, twl, g.lognx);  // ra, rb consecutive
  for (int i = threadIdx.x; i < nx; i += PIC_WG) {
    A[(long long)k * nx + i] = ra[i];
    if (k2 != k) A[(long long)k2 * nx + i] = rb[i];
  }
}

// rows: inverse FFT_y of R_hat row i -> padded lrho[i][j] = Re / (nx ny)
__global__ __launch_bounds__(PIC_WG) void k_adj_rows_inv(AdjGrid g, const double2* __restrict__ A,
                                                         double* __restrict__ lrho,
                                                         const double2* __restrict__ tw) {
  extern __shared__ double2 s[];
  const int i = xcd_item(blockIdx.x, gridDim.x), ny = g.ny;
  for (int k = threadIdx.x; k < ny; k += PIC_WG) s[bitrev(k, g.logny)] = A[(long long)k * g.nx + i];
  __syncthreads();
  fft_lds(s, ny, g.logny, +1, tw);
  const double norm = 1.0 / ((double)g.nx * ny);
  // padded like E: row nx repeats row 0, column ny repeats column 0
  for (int j = threadIdx.x; j <= ny; j += PIC_WG) {
    const double v = s[j & (ny - 1)].x * norm;
    lrho[i * (ny + 1) + j] = v;
    if (i == 0) lrho[g.nx * (ny + 1) + j] = v;
  }
}

// dL/da_m = sum_p lx_p cos(kx_m xl_p + ky_m yl_p): block partials [block][m]
__global__ __launch_bounds__(PIC_WG) void k_adj_amp_grad(const double* __restrict__ lx,
                                                         const double* __restrict__ xl,
                                                         const double* __restrict__ yl,
                                                         int64_t n, const double* __restrict__ mkx,
                                                         const double* __restrict__ mky, int nm,
                                                         double* __restrict__ part) {
  __shared__ double red[4];
  for (int m = 0; m < nm; ++m) {
    double s = 0.0;
    for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
         p += (int64_t)gridDim.x * PIC_WG)
      s += lx[p] * cos(mkx[m] * xl[p] + mky[m] * yl[p]);
    s = block_sum(s, red);
    if (threadIdx.x == 0) part[(long long)blockIdx.x * nm + m] = s;
  }
}

__global__ __launch_bounds__(PIC_WG) void k_adj_amp_reduce(const double* __restrict__ part,
                                                           int nblocks, int nm, double scale,
                                                           double* __restrict__ out) {
  if (threadIdx.x < nm) {
    // in block order; the loads of eight blocks are issued before their adds
    double s = 0.0;
    int b = 0;
    for (; b + 8 <= nblocks; b += 8) {
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = part[(long long)(b + k) * nm + threadIdx.x];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
    for (; b < nblocks; ++b) s += part[(long long)b * nm + threadIdx.x];
    out[threadIdx.x] = scale * s;
  }
}

template <typename R>
__global__ __launch_bounds__(PIC_WG) void k_adj_to_r(const double* __restrict__ a, double s,
                                                     R* __restrict__ out, int64_t n) {
  for (int64_t p = blockIdx.x * (int64_t)PIC_WG + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * PIC_WG)
    out[p] = (R)(s * a[p]);
}

inline int gridn(long long n) {
  long long b = (n + PIC_WG - 1) / PIC_WG;
  return (int)(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

}  // namespace

template <typename R>
void adj_init(hipStream_t s, const AdjGrid& g, const double* xl, const double* yl, int64_t n,
              const double* amps, const double* mkx, const double* mky, int nm, R* x, R* y,
              unsigned long long* hi, unsigned long long* lo) {
  k_adj_init<R><<<gridn(n), PIC_WG, 0, s>>>(g, xl, yl, n, amps, mkx, mky, nm, x, y, hi, lo);
}
template <typename R>
void adj_segment(hipStream_t s, const AdjGrid& g, const R* ck, const R* Eseg, long long estride,
                 int k0, int nst, R* xs, R* ys, int64_t n) {
  k_adj_segment<R><<<gridn(n), PIC_WG, 0, s>>>(g, ck, Eseg, estride, k0, nst, xs, ys, n);
}
void adj_zero(hipStream_t s, double* a, long long n) {
  k_adj_zero<<<gridn(n), PIC_WG, 0, s>>>(a, n);
}
template <typename R>
void adj_pass_end(hipStream_t s, const AdjGrid& g, const R* xk, const R* yk, const double* lrho,
                  double cq, double* lx, double* ly, int64_t n) {
  k_adj_pass_end<R><<<gridn(n), PIC_WG, 0, s>>>(g, xk, yk, lrho, cq, lx, ly, n);
}
template <typename R>
void adj_push_win(hipStream_t s, const AdjGrid& g, const int4* items, const int* toff,
                  const R* const in[4], R* const out[4], const R* E, double c,
                  unsigned long long* hi, unsigned long long* lo) {
  const size_t nw = (size_t)g.win * g.win;
  const size_t lds = nw * ((sizeof(R) == 8 ? 2 : 1) * sizeof(unsigned long long) +
                           2 * sizeof(R));
  if (E)
    k_adj_push_win<R, true><<<g.nitems, ADJ_NT, lds, s>>>(g, items, toff, in[0], in[1], in[2],
                                                          in[3], out[0], out[1], out[2], out[3],
                                                          E, c, hi, lo);
  else
    k_adj_push_win<R, false><<<g.nitems, ADJ_NT, lds, s>>>(g, items, toff, in[0], in[1], nullptr,
                                                           nullptr, nullptr, nullptr, nullptr,
                                                           nullptr, nullptr, c, hi, lo);
}
template <typename R>
void adj_pass_win(hipStream_t s, const AdjGrid& g, const int4* items, const int* toff,
                  const R* xk, const R* yk, const double* lrho, double cq, const R* xp,
                  const R* yp, const R* Eprev, double ck1, double* lx, double* ly,
                  double* lvx, double* lvy, double* lE) {
  const size_t lds = 2 * sizeof(double) * (size_t)g.win * g.win;
  k_adj_pass_win<R><<<g.nitems, ADJ_NT, lds, s>>>(g, items, toff, xk, yk, lrho, cq, xp, yp,
                                                  Eprev, ck1, lx, ly, lvx, lvy, lE);
}
void adj_reorder(hipStream_t s, const int* from, const double* a, double* b, int64_t n) {
  k_adj_reorder<<<gridn(n), PIC_WG, 0, s>>>(from, a, b, n);
}
template <typename R>
void adj_seed(hipStream_t s, const AdjGrid& g, const R* E, double sc, double* lE) {
  k_adj_seed<R><<<gridn((long long)g.nx * g.ny), PIC_WG, 0, s>>>(g, E, sc, lE);
}
template <typename R>
void adj_energy(hipStream_t s, const AdjGrid& g, const R* E, double* part, int nblocks) {
  k_adj_energy<R><<<nblocks, PIC_WG, 0, s>>>(g, E, part);
}
void adj_mt(hipStream_t s, const AdjGrid& g, double* lE, double2* A, double* lrho,
            const double2* tw) {
  k_adj_rows_fwd<<<g.nx, PIC_WG, sizeof(double2) * g.ny, s>>>(g, lE, A, tw);
  k_adj_cols<<<g.ny / 2 + 1, PIC_WG, sizeof(double2) * (4 * g.nx + g.nx / 2), s>>>(g, A, tw);
  k_adj_rows_inv<<<g.nx, PIC_WG, sizeof(double2) * g.ny, s>>>(g, A, lrho, tw);
}
void adj_amp_grad(hipStream_t s, const double* lx, const double* xl, const double* yl, int64_t n,
                  const double* mkx, const double* mky, int nm, double* part, int nblocks,
                  double scale, double* out) {
  if (nm <= 0) return;
  k_adj_amp_grad<<<nblocks, PIC_WG, 0, s>>>(lx, xl, yl, n, mkx, mky, nm, part);
  k_adj_amp_reduce<<<1, PIC_WG, 0, s>>>(part, nblocks, nm, scale, out);
}
template <typename R>
void adj_to_r(hipStream_t s, const double* a, double sc, R* out, int64_t n) {
  k_adj_to_r<R><<<gridn(n), PIC_WG, 0, s>>>(a, sc, out, n);
}

#define ADJ_INST(R)                                                                           \
  template void adj_init<R>(hipStream_t, const AdjGrid&, const double*, const double*,       \
                            int64_t, const double*, const double*, const double*, int, R*,   \
                            R*, unsigned long long*, unsigned long long*);                   \
  template void adj_segment<R>(hipStream_t, const AdjGrid&, const R*, const R*, long long,    \
                               int, int, R*, R*, int64_t);                                   \
  template void adj_pass_end<R>(hipStream_t, const AdjGrid&, const R*, const R*,              \
                                const double*, double, double*, double*, int64_t);           \
  template void adj_push_win<R>(hipStream_t, const AdjGrid&, const int4*, const int*,        \
                                const R* const[4], R* const[4], const R*, double,            \
                                unsigned long long*, unsigned long long*);                   \
  template void adj_pass_win<R>(hipStream_t, const AdjGrid&, const int4*, const int*,         \
                                const R*, const R*, const double*, double, const R*,         \
                                const R*, const R*, double, double*, double*, double*,       \
                                double*, double*);                                           \
  template void adj_seed<R>(hipStream_t, const AdjGrid&, const R*, double, double*);          \
  template void adj_energy<R>(hipStream_t, const AdjGrid&, const R*, double*, int);           \
  template void adj_to_r<R>(hipStream_t, const double*, double, R*, int64_t);
ADJ_INST(float)
ADJ_INST(double)
