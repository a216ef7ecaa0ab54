// ops.cpp -- per-stage operators of the C ABI on caller-owned device arrays.
//
// The reference keeps each stage as a file-static kernel configured through
// __constant__ symbols (thesisCode/collisionless/double/src/pic.cu:13-26, 69-420); these
// entry points expose the same stages with explicit arguments so each can be dropped into
// another driver or tested alone.  Temporaries come from blocks kept between calls
// (workspace.cpp), except in pic_op_deposit_noalloc (a static device array).
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "engine.h"

using namespace pic;

namespace {

int check_grid(const pic_grid* g) {
  if (!g) return fail(PIC_ERR_ARG, "NULL grid");
  pic_config c;
  pic_config_default(&c);
  c.nx = g->nx; c.ny = g->ny; c.lx = g->lx; c.ly = g->ly;
  return validate_config(c);
}

// single-run descriptor for the operator kernels (all bases zero)
RunDesc op_desc(int nx, int ny, double lx, double ly, long long pcap) {
  RunDesc d;
  std::memset(&d, 0, sizeof(d));
  d.schunk = PIC_CHUNK;
  d.nx = nx; d.ny = ny;
  int l = 0;
  while ((1 << l) < nx) ++l;
  d.lognx = l;
  l = 0;
  while ((1 << l) < ny) ++l;
  d.logny = l;
  d.lx = lx; d.ly = ly; d.dx = lx / nx; d.dy = ly / ny;
  d.pcap = (int)pcap;
  fft_groups(nx, nx, ny, &d.fft_pp, &d.fft_rf);
  return d;
}

}  // namespace

extern "C" {

int pic_op_cell_keys(const void* x, const void* y, int64_t n, int precision, const pic_grid* g,
                     int32_t* keys, void* stream) {
  int rc = check_grid(g);
  if (rc) return rc;
  if (n < 0 || (n > 0 && (!x || !y || !keys))) return fail(PIC_ERR_ARG, "bad arrays");
  if (n == 0) return PIC_OK;
  hipStream_t s = (hipStream_t)stream;
  if (precision == PIC_FP64)
    launch_op_cell_keys<double>(s, (const double*)x, (const double*)y, n, g->nx, g->ny, g->lx,
                                g->ly, keys);
  else if (precision == PIC_FP32)
    launch_op_cell_keys<float>(s, (const float*)x, (const float*)y, n, g->nx, g->ny, g->lx, g->ly,
                               keys);
  else
    return fail(PIC_ERR_ARG, "precision must be PIC_FP32 or PIC_FP64");
  PIC_HIP(hipGetLastError());
  return PIC_OK;
}

int pic_op_sort(const int32_t* keys, int64_t n, int ncells, int32_t* perm, int32_t* counts,
                int32_t* offsets, void* stream) {
  if (n < 0 || ncells < 1 || n > 0x7fff0000) return fail(PIC_ERR_ARG, "bad sizes");
  if (!perm || !counts || !offsets || (n > 0 && !keys)) return fail(PIC_ERR_ARG, "NULL array");
  hipStream_t s = (hipStream_t)stream;
  const RadixPlan p = radix_plan(n, ncells);
  const size_t nn = (size_t)std::max<int64_t>(n, 1), nd = (size_t)1 << p.bits;
  Workspace m;
  RadixBufs b;
  std::memset(&b, 0, sizeof(b));
  PIC_HIP(m.get(&b.flag, 1));
  PIC_HIP(m.get(&b.totals, nd));
  PIC_HIP(m.get(&b.table, nd * std::max(p.tiles, 1)));
  for (int k = 0; k < 2; ++k) {
    if (p.passes > k) PIC_HIP(m.get(&b.keys[k], nn));
    if (p.passes > k + 1) PIC_HIP(m.get(&b.idx[k], nn));
  }
  launch_fill_i32(s, b.flag, 1, 0);
  launch_radix_sort(s, keys, (int)n, ncells, p, b, perm, counts, offsets);
  PIC_HIP(hipGetLastError());
  int* h;
  PIC_HIP(m.pinned(&h, 1));
  PIC_HIP(hipMemcpyAsync(h, b.flag, sizeof(int), hipMemcpyDeviceToHost, s));
  PIC_HIP(hipStreamSynchronize(s));
  m.done();
  if (*h) return fail(PIC_ERR_ARG, "key outside [0, ncells)");
  return PIC_OK;
}

int pic_op_deposit(const void* x, const void* y, int64_t n, int precision, const pic_grid* g,
                   double qp, double* rho, void* stream) {
  int rc = check_grid(g);
  if (rc) return rc;
  if (n < 0 || !rho || (n > 0 && (!x || !y))) return fail(PIC_ERR_ARG, "bad arrays");
  if (precision != PIC_FP32 && precision != PIC_FP64) return fail(PIC_ERR_ARG, "bad precision");
  hipStream_t s = (hipStream_t)stream;
  const long long G = (long long)g->nx * g->ny;
  const bool fp64 = precision == PIC_FP64;
  DepositPlan p = deposit_plan(n, g->nx, g->ny, fp64, true);
  Workspace m;
  unsigned long long *hi, *lo = nullptr;
  PIC_HIP(m.get(&hi, G));
  if (fp64) PIC_HIP(m.get(&lo, G));
  DepositBufs b;
  std::memset(&b, 0, sizeof(b));
  if (p.form == DEPOSIT_BINNED) {
    char* pos = nullptr;
    const size_t table = (size_t)p.tiles * p.groups;
    if (m.get(&b.table, table + 2 * (size_t)p.tiles + 1) == hipSuccess &&
        m.get(&pos, (fp64 ? 16 : 8) * (size_t)n) == hipSuccess) {
      b.totals = b.table + table;
      b.offs = b.totals + p.tiles;
      b.pos = pos;
    } else {  // no memory for the moved positions: a form that needs none
      (void)hipGetLastError();
      p = deposit_plan(n, g->nx, g->ny, fp64, false);
    }
  }
  launch_fill_u64(s, hi, G);
  if (fp64) launch_fill_u64(s, lo, G);
  if (n > 0) {
    if (fp64)
      launch_op_deposit<double>(s, p, (const double*)x, (const double*)y, n, g->nx, g->ny, g->lx,
                                g->ly, hi, lo, b);
    else
      launch_op_deposit<float>(s, p, (const float*)x, (const float*)y, n, g->nx, g->ny, g->lx,
                               g->ly, hi, lo, b);
  }
  const double dx = g->lx / g->nx, dy = g->ly / g->ny;
  const double scale = qp / (dx * dy) * (precision == PIC_FP64 ? 1.0 : std::ldexp(1.0, -36));
  launch_op_fixed_to_double(s, hi, lo, G, precision == PIC_FP64, scale, rho);
  PIC_HIP(hipGetLastError());
  PIC_HIP(hipStreamSynchronize(s));
  m.done();
  return PIC_OK;
}

}  // extern "C"

// ---- allocation-free deposit: the fixed-point accumulators live in a file-scope device
// array instead of per-call hipMalloc.  Every device that runs the library holds its own
// copy (16 MiB) until the process ends.  In host code the array's name is only a
// stand-in symbol: its device address comes from hipGetSymbolAddress, once per device.
static __device__ __align__(256) unsigned long long scratch[2 * PIC_DEPOSIT_NOALLOC_MAX_NODES];
// Twiddles of the field solve, exp(-2 pi i j / PIC_FFT_MAX): 16 KiB per device, filled on the
// first call there.
static __device__ double2 op_tw[PIC_FFT_MAX / 2];

namespace {
std::mutex g_scratch_mu;
unsigned long long* g_scratch_ptr[64];  // device address of `scratch` per device ordinal
double2* g_tw_ptr[64];                  // device address of `op_tw`, once filled

int op_twiddles(double2** out) {
  int dev = 0;
  PIC_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return fail(PIC_ERR_UNSUPPORTED, "device ordinal above 63");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_tw_ptr[dev]) {
    std::vector<double2> h(PIC_FFT_MAX / 2);
    for (int j = 0; j < PIC_FFT_MAX / 2; ++j) {
      const long double a = 2.0L * 3.141592653589793238462643383279L * j / PIC_FFT_MAX;
      h[j] = make_double2((double)cosl(a), (double)-sinl(a));
    }
    void* p = nullptr;
    PIC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(op_tw)));
    // synchronous: in place before any stream's kernel reads it
    PIC_HIP(hipMemcpy(p, h.data(), sizeof(double2) * h.size(), hipMemcpyHostToDevice));
    g_tw_ptr[dev] = (double2*)p;
  }
  *out = g_tw_ptr[dev];
  return PIC_OK;
}

// Device address of `scratch` on the current device, looked up on the first call there.
int noalloc_scratch(unsigned long long** out) {
  int dev = 0;
  PIC_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return fail(PIC_ERR_UNSUPPORTED, "device ordinal above 63");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(PIC_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch_ptr[dev] = (unsigned long long*)p;
  }
  *out = g_scratch_ptr[dev];
  return PIC_OK;
}
}  // namespace

extern "C" {

int pic_op_deposit_noalloc(const void* x, const void* y, int64_t n, int precision,
                           const pic_grid* g, double qp, double* rho, void* stream) {
  int rc = check_grid(g);
  if (rc) return rc;
  if (n < 0 || !rho || (n > 0 && (!x || !y))) return fail(PIC_ERR_ARG, "bad arrays");
  if (precision != PIC_FP32 && precision != PIC_FP64) return fail(PIC_ERR_ARG, "bad precision");
  const long long G = (long long)g->nx * g->ny;
  if (G > PIC_DEPOSIT_NOALLOC_MAX_NODES)
    return fail(PIC_ERR_UNSUPPORTED, "pic_op_deposit_noalloc: nx*ny = " + std::to_string(G) +
                                         " exceeds its static scratch of " +
                                         std::to_string(PIC_DEPOSIT_NOALLOC_MAX_NODES) + " nodes");
  unsigned long long* hi = nullptr;
  if ((rc = noalloc_scratch(&hi))) return rc;
  unsigned long long* lo = hi + PIC_DEPOSIT_NOALLOC_MAX_NODES;
  hipStream_t s = (hipStream_t)stream;
  // cleared by a fill kernel (the previous call's sums are still there)
  launch_fill_u64(s, hi, G);
  if (precision == PIC_FP64) launch_fill_u64(s, lo, G);
  if (n > 0) {
    // the forms that need no memory of their own
    const DepositPlan p = deposit_plan(n, g->nx, g->ny, precision == PIC_FP64, false);
    const DepositBufs none = {nullptr, nullptr, nullptr, nullptr};
    if (precision == PIC_FP64)
      launch_op_deposit<double>(s, p, (const double*)x, (const double*)y, n, g->nx, g->ny, g->lx,
                                g->ly, hi, lo, none);
    else
      launch_op_deposit<float>(s, p, (const float*)x, (const float*)y, n, g->nx, g->ny, g->lx,
                               g->ly, hi, nullptr, none);
  }
  const double dx = g->lx / g->nx, dy = g->ly / g->ny;
  const double scale = qp / (dx * dy) * (precision == PIC_FP64 ? 1.0 : std::ldexp(1.0, -36));
  launch_op_fixed_to_double(s, hi, precision == PIC_FP64 ? lo : nullptr, G,
                            precision == PIC_FP64, scale, rho);
  PIC_HIP(hipGetLastError());
  PIC_HIP(hipStreamSynchronize(s));
  return PIC_OK;
}

int pic_op_poisson(const double* rho, double* phi, const pic_grid* g, void* stream) {
  int rc = check_grid(g);
  if (rc) return rc;
  if (!rho || !phi) return fail(PIC_ERR_ARG, "NULL array");
  hipStream_t s = (hipStream_t)stream;
  const int nx = g->nx, ny = g->ny;
  double2* tw = nullptr;
  if ((rc = op_twiddles(&tw))) return rc;
  RunDesc d = op_desc(nx, ny, g->lx, g->ly, 0);
  if (launch_phi_one(s, d, rho, phi, tw)) {
    PIC_HIP(hipGetLastError());
    PIC_HIP(hipStreamSynchronize(s));
    return PIC_OK;
  }
  const int nrp = nx / (2 * d.fft_pp), ncl = ny / 2 + 1;
  const size_t ss = (size_t)ncl * nx;
  Workspace m;
  double2* S;
  RunDesc* dd;
  RunState* st;
  int2* items;
  PIC_HIP(m.get(&S, ss));
  PIC_HIP(m.get(&dd, 1));
  PIC_HIP(m.get(&st, 1));
  PIC_HIP(m.get(&items, (size_t)nrp + ncl));
  launch_op_setup(s, d, dd, st, items, nrp, items + nrp, ncl);
  FieldArgs a;
  std::memset(&a, 0, sizeof(a));
  a.runs = dd; a.st = st;
  a.S = S; a.phi = phi; a.tw = tw;
  a.row_pair_items = items; a.n_row_pair_items = nrp;
  a.col_items = items + nrp; a.n_col_items = ncl;
  a.nruns = 1; a.fp64 = 0; a.want_phi = 1; a.max_nx = nx; a.max_ny = ny;
  a.row_lds = d.fft_pp * ny;
  a.rho_in = rho;
  launch_field(s, a, nullptr);
  PIC_HIP(hipGetLastError());
  PIC_HIP(hipStreamSynchronize(s));
  m.done();
  return PIC_OK;
}

int pic_op_efield(const double* phi, double* ex, double* ey, const pic_grid* g, void* stream) {
  int rc = check_grid(g);
  if (rc) return rc;
  if (!phi || !ex || !ey) return fail(PIC_ERR_ARG, "NULL array");
  launch_op_efield((hipStream_t)stream, phi, ex, ey, g->nx, g->ny, g->lx, g->ly);
  PIC_HIP(hipGetLastError());
  return PIC_OK;
}

int pic_op_gather_push(void* x, void* y, void* vx, void* vy, int64_t n, int precision,
                       const double* ex, const double* ey, const pic_grid* g, double dt,
                       double qm, double c, double* ke, void* stream) {
  int rc = check_grid(g);
  if (rc) return rc;
  if (n < 0 || !ex || !ey || (n > 0 && (!x || !y || !vx || !vy))) return fail(PIC_ERR_ARG, "bad arrays");
  if (precision != PIC_FP32 && precision != PIC_FP64) return fail(PIC_ERR_ARG, "bad precision");
  hipStream_t s = (hipStream_t)stream;
  const bool fp64 = precision == PIC_FP64;
  const GatherPushPlan p = gather_push_plan(n, g->nx, g->ny, fp64);
  Workspace m;
  double* parts = nullptr;
  if (ke) PIC_HIP(m.get(&parts, p.blocks));
  char* pairs = nullptr;
  if (p.pairs && m.get(&pairs, (fp64 ? 16 : 8) * (size_t)p.pairs) != hipSuccess) {
    (void)hipGetLastError();  // no memory for the packed field: the node arrays are read
    pairs = nullptr;
  }
  int* choice = nullptr;
  if (pairs && p.choose) PIC_HIP(m.get(&choice, 1));
  if (fp64)
    launch_op_gather_push<double>(s, p, (double*)x, (double*)y, (double*)vx, (double*)vy, n, ex,
                                  ey, g->nx, g->ny, g->lx, g->ly, dt, qm, c, parts, pairs, choice);
  else
    launch_op_gather_push<float>(s, p, (float*)x, (float*)y, (float*)vx, (float*)vy, n, ex, ey,
                                 g->nx, g->ny, g->lx, g->ly, dt, qm, c, parts, pairs, choice);
  if (ke) launch_reduce_sum(s, parts, p.blocks, ke);
  PIC_HIP(hipGetLastError());
  PIC_HIP(hipStreamSynchronize(s));
  m.done();
  return PIC_OK;
}

int pic_op_mcc(float* x, float* y, float* vx, float* vy, int32_t* id, int64_t* n_io, int64_t cap,
               const pic_config* cfg, int64_t step, int64_t* counts, void* stream) {
  if (!x || !y || !vx || !vy || !id || !n_io || !cfg) return fail(PIC_ERR_ARG, "NULL argument");
  if (*n_io < 0 || cap < *n_io || cap > 0x7fff0000) return fail(PIC_ERR_ARG, "bad sizes");
  pic_config c = *cfg;
  c.collide = PIC_COLLIDE_MCC;
  c.precision = PIC_FP32;
  int rc = validate_config(c);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  Workspace m;
  RunState* st;
  RunDesc* dd;
  int *bc, *bp, *cl, *cp;
  float* bb;
  unsigned long long *scratch, *rho;
  PIC_HIP(m.get(&st, 1));
  PIC_HIP(m.get(&dd, 1));
  PIC_HIP(m.get(&bc, 1));
  PIC_HIP(m.get(&bp, std::max<int64_t>(cap, 1)));
  PIC_HIP(m.get(&bb, 4 * std::max<int64_t>(cap, 1)));
  int lb, lp;
  mcc_list_layout(std::max<int64_t>(*n_io, 1), &lb, &lp);
  PIC_HIP(m.get(&cl, (size_t)lb * lp));
  PIC_HIP(m.get(&cp, 4 * PIC_MCC_BLOCKS));
  PIC_HIP(m.get(&scratch, 2 * std::max<int64_t>(cap, 1)));
  PIC_HIP(m.get(&rho, 2 * (size_t)c.nx * c.ny));
  RunState hs;
  std::memset(&hs, 0, sizeof(hs));
  hs.np = (int)*n_io;
  // next_id = largest id + 1 is the caller's contract: ids are 0..n-1 here
  hs.next_id = *n_io;
  hs.step = step;
  RunDesc d = op_desc(c.nx, c.ny, c.lx, c.ly, cap);
  PIC_HIP(hipMemcpyAsync(st, &hs, sizeof(hs), hipMemcpyHostToDevice, s));
  PIC_HIP(hipMemcpyAsync(dd, &d, sizeof(d), hipMemcpyHostToDevice, s));
  PIC_HIP(hipMemsetAsync(bc, 0, sizeof(int), s));
  PIC_HIP(hipMemsetAsync(rho, 0, sizeof(unsigned long long) * 2 * c.nx * c.ny, s));
  MccArgs a;
  std::memset(&a, 0, sizeof(a));
  a.x = x; a.y = y; a.vx = vx; a.vy = vy; a.id = id;
  a.st = st; a.pbase = 0; a.cap = (int)cap;
  const double kE = 1.602176634e-19, kMe = 9.1093837015e-31;
  a.v_unit2_half_me_over_e = 0.5 * kMe * c.mcc_v_unit * c.mcc_v_unit / kE;
  a.ng_vunit_dtphys = c.mcc_ng * c.mcc_v_unit * c.mcc_dt_phys * c.dt;
  const double numax_dt = mcc_nu_max(c) * c.mcc_dt_phys * c.dt;
  a.nu_max_dt = numax_dt;
  mcc_null_range(1.0 - std::exp(-numax_dt), &a.null_any, &a.null_last);
  a.mass_ratio2 = 2.0 * kMe / c.mcc_neutral_mass;
  a.seed = c.seed;
  a.counts = (long long*)counts;
  a.birth_count = bc; a.birth_parent = bp; a.birth_buf = bb;
  a.coll_list = cl; a.coll_partials = cp;
  a.from_state_step = 0;
  a.step = step;
  launch_mcc(s, a, (int)*n_io);
  launch_mcc_births(s, a, scratch, rho, (long long)c.nx * c.ny, dd, 0, (int)*n_io);
  PIC_HIP(hipGetLastError());
  PIC_HIP(hipMemcpyAsync(&hs, st, sizeof(hs), hipMemcpyDeviceToHost, s));
  PIC_HIP(hipStreamSynchronize(s));
  m.done();
  *n_io = hs.np;
  if (hs.err & 1) return fail(PIC_ERR_OVERFLOW, "births exceeded capacity");
  return PIC_OK;
}

int pic_op_dsmc(float* vx, float* vy, const int32_t* id, const int32_t* offsets, int ncells,
                float* gmax, double coeff, uint64_t seed, int64_t step, int64_t* ncoll,
                void* stream) {
  if (!vx || !vy || !id || !offsets || !gmax || ncells < 1 || !(coeff >= 0))
    return fail(PIC_ERR_ARG, "bad argument");
  DsmcArgs a;
  std::memset(&a, 0, sizeof(a));
  (void)id;  // cells hold their particles in the caller's (canonical) order
  a.vx = vx; a.vy = vy; a.offsets = offsets; a.gmax = gmax;
  a.ncells = ncells; a.tile_shift = -1; a.tiles_y = 1; a.ny = 1; a.coeff = coeff; a.seed = seed; a.step = step; a.st = nullptr;
  a.ncoll = (long long*)ncoll;
  launch_dsmc((hipStream_t)stream, a);
  PIC_HIP(hipGetLastError());
  return PIC_OK;
}

}  // extern "C"
