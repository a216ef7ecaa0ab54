// launch.h -- host-side launchers of the HIP kernels (internal to libpicamd.so).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "pic_device.h"

// Item lists (device, built once per context):
//   chunk items  int2 {run, start}: PIC_CHUNK particles or PIC_CELL_CHUNK cells
//   tile items   int4 {run, tx, ty, split}; tx < 0 marks a tail chunk (start in .z)
//   row items    int2 {run, row}
#define PIC_CELL_CHUNK 2048

struct SortBufs {
  // cell sort (runs with DSMC)
  int* keys;        // [ptotal]
  int* rank;        // [ptotal]
  unsigned long long* rec;      // [ptotal] (id << 32 | run-local source slot) by cell
  int* counts;      // [ctotal]
  int* offsets;     // [ctotal]
  int* chunk_sums;  // [n cell chunk items]
  int* big_list;    // [2*ctotal] cells that one workgroup sorts, (run, cell) pairs
  int* big_count;   // [1]
  unsigned long long* scratch;  // [2*ptotal] power-of-two padded segments (also MCC births)
  // tile sort of the step
  int* table;                   // [sum nbuckets*nchunks] bucket-major count table
  int* tchunk_sums;             // [n table-scan items]
  const int2* tscan_items;      // {run, first entry} items of PIC_CELL_CHUNK table entries
  int ntscan_items;
  int* toff;                    // [sum (nbuckets+1)] tile offsets written by the sort
  int max_buckets;
  // sort fused into the push
  int* ftable;                  // [sum fchunks*nbuckets] row-major counts, then slots
  int* fchunk_sums;             // [n fused table-scan items][max_buckets] group sums
  const int2* fscan_items;      // {run, row group} items of FSCAN_ROWS table rows
  int nfscan_items;
};

template <typename R>
struct PartBufs {
  R *x, *y, *vx, *vy;
  int* id;
};

// ---- cell sort (k_cellsort.hip): src in cell order, ascending id inside a cell, to dst; writes
// sb.offsets, sb.toff and RunState::nsorted
void launch_cell_sort(hipStream_t s, const RunDesc* runs, RunState* st, PartBufs<float> src,
                      PartBufs<float> dst, SortBufs sb, const int2* pitems, int npitems,
                      const int2* citems, int ncitems);

// ---- particle kernels (k_particles.hip)
// stable tile (bucket) sort of the step; writes sb.toff and RunState::nsorted
// scan of the fused sort's count table and the new tile offsets (toff_new, nsorted)
void launch_fused_scan(hipStream_t s, const RunDesc* runs, RunState* st, int nruns,
                       SortBufs sb, int* toff_new);
template <typename R>
void launch_tile_sort(hipStream_t s, const RunDesc* runs, RunState* st, int nruns,
                      PartBufs<R> src, PartBufs<R> dst, SortBufs sb, const int2* pitems,
                      int npitems, int schunk);

// ---- deposit of particles in any order (k_deposit.hip)
enum { DEPOSIT_DIRECT, DEPOSIT_GRID, DEPOSIT_BINNED };
struct DepositPlan {
  int form;            // DEPOSIT_*
  int ltx, lty;        // binned: log2 of the tile sides
  int tiles, tiles_y;
  int items, groups;   // positions per thread and workgroups of the moving pass
  int slice;           // positions per workgroup of the summing pass
};
struct DepositBufs {   // binned form only
  int* table;          // [tiles][groups]
  int* totals;         // [tiles]
  int* offs;           // [tiles + 1]
  void* pos;           // [n] (x, y) pairs
};
// scratch: DepositBufs can be had (the binned form may be chosen)
DepositPlan deposit_plan(int64_t n, int nx, int ny, int fp64, bool scratch);
template <typename R>
void launch_op_deposit(hipStream_t s, const DepositPlan& p, const R* x, const R* y, int64_t n,
                       int nx, int ny, double lx, double ly, unsigned long long* hi,
                       unsigned long long* lo, DepositBufs b);

// ---- stable sort of given keys (k_radix.hip)
struct RadixPlan {
  int bits, passes;    // digit width and number of digits
  int items, tiles;    // items per thread, tiles of items * PIC_WG
};
struct RadixBufs {
  int* table;          // [2^bits][tiles]
  int* totals;         // [2^bits]
  int* keys[2];        // [n]: pass q writes keys[q & 1]
  int* idx[2];         // [n]: pass q writes idx[q & 1]; the last writes perm (so one pass
                       // needs none of them, two need idx[0])
  int* flag;           // [1], zero: set when a key lies outside [0, ncells)
};
RadixPlan radix_plan(long long n, int ncells);
// exclusive scan of every row of table[rows][cols] in place, and the rows' sums; does nothing
// when flag is given and set
void launch_scan_rows(hipStream_t s, int* table, int rows, int cols, int* totals,
                      const int* flag);
void launch_radix_sort(hipStream_t s, const int* keys, int n, int ncells, const RadixPlan& p,
                       RadixBufs b, int* perm, int* counts, int* offsets);

#define FSCAN_ROWS 64  // rows (push items) per fused count-table scan item
#define PUSH_NT 512            // threads per push workgroup
#define PUSH_NW (PUSH_NT / 64)  // waves per push workgroup

template <typename R>
struct PushArgs {
  const RunDesc* runs;
  RunState* st;
  R *x, *y, *vx, *vy;
  const R* E;
  unsigned long long* rho;      // [2][gsum] (hi word for FP64)
  unsigned long long* rho_lo;   // [2][gsum] (FP64 only)
  long long gsum;
  const int* off;
  const int4* items;
  int nitems;
  int nruns;
  double* partials;             // [nitems*3] per-workgroup kinetic energy, px, py
  int mode;                     // 0: gather+push+deposit, 1: deposit only
  int by_cell;                  // the particles are in cell order, many per cell (DSMC); items
                                // may be shares
  int lds_bytes;
  // sort fused into the push (mode 0, tile items): 0 off; 1 count the tiles of the new
  // positions per item into its row of ftable; 2 scatter the particles tile-major (by their
  // positions at the start of this step) into dst, with their ids
  int sort_mode;
  int* ftable;
  PartBufs<R> dst;
  const int* id;                // ids of the source buffer
};
template <typename R>
void launch_push(hipStream_t s, const PushArgs<R>& a);
// per run: diagnostics row of the step from the field and push partials, then step + 1
void launch_step_finish(hipStream_t s, const RunDesc* runs, RunState* st, int nruns,
                        const double* ppush, const double* prows, double* diag);

// The n particles of a run in id order.  E: the run context's padded field, to add the pending
// half kick, or NULL.  rec: n records {x, y, vx, vy} by id are written there, for
// launch_out_split; NULL: the output arrays (those not NULL) are written.
template <typename R>
void launch_out_particles(hipStream_t s, const RunDesc* runs, RunState* st, int run, int n,
                          PartBufs<R> p, const R* E, void* rec, R* ox, R* oy, R* ovx, R* ovy);
template <typename R>
void launch_out_split(hipStream_t s, const void* rec, int n, R* ox, R* oy, R* ovx, R* ovy);
// sums of vx^8 and vy^8 over n particles from slot base on: part[SPEED_BLOCKS][2]
// (device or pinned memory)
#define SPEED_BLOCKS 1024
template <typename R>
void launch_speed8(hipStream_t s, PartBufs<R> p, long long base, int64_t n, double* part);
template <typename R>
void launch_check_finite(hipStream_t s, const RunDesc* runs, RunState* st, PartBufs<R> p,
                         const int2* pitems, int npitems, int* flag);

// ops on plain device arrays (run 0 descriptor)
template <typename R>
void launch_op_cell_keys(hipStream_t s, const R* x, const R* y, int64_t n, int nx, int ny,
                         double lx, double ly, int* keys);
#define GP_LDS_NT 512   // threads per workgroup of the gather + push with the field in LDS
struct GatherPushPlan {
  int blocks;           // workgroups (and kinetic-energy partials)
  int lds;              // bytes of the padded field in LDS, 0: not there
  long long pairs;      // (Ex, Ey) pairs of the packed field, 0: not used
  int rows;             // packed with the two node rows of a cell interleaved
  int choose;           // 1: the form goes by the order of the positions (gp_form)
  int ordered, local;   // then those for ordered and for local positions
};
GatherPushPlan gather_push_plan(int64_t n, int nx, int ny, int fp64);
// pairs: memory for the plan's packed field, or NULL (then the node arrays are read); choice: a word
// for a plan that chooses, else NULL
template <typename R>
void launch_op_gather_push(hipStream_t s, const GatherPushPlan& p, R* x, R* y, R* vx, R* vy,
                           int64_t n, const double* ex, const double* ey, int nx, int ny,
                           double lx, double ly, double dt, double qm, double c,
                           double* ke_partials, void* pairs, int* choice);
void launch_op_fixed_to_double(hipStream_t s, const unsigned long long* hi,
                               const unsigned long long* lo, long long G, int fp64,
                               double scale, double* out);
void launch_fill_i32(hipStream_t s, int* p, long long n, int v);
void launch_iota(hipStream_t s, int* p, long long n);  // p[i] = i
void launch_fill_u64(hipStream_t s, unsigned long long* p, long long n);
void launch_reduce_sum(hipStream_t s, const double* parts, int n, double* out);

// ---- field kernels (k_field.hip)
// Row passes work on groups of consecutive rows (at most about 2048 complex values of LDS),
// so the transposed spectra S[k][x] are read and written in contiguous runs along x.
// Forward rows are packed in pairs (two real rows = one complex FFT).
__host__ __device__ inline int fft_row_pairs_per_block(int nx, int ny) {
  int p = 2048 / ny;
  p = p < 1 ? 1 : (p > 8 ? 8 : p);
  return p > nx / 2 ? nx / 2 : p;
}
__host__ __device__ inline int fft_rows_per_block(int nx, int ny) {
  int r = 2048 / ny;
  r = r < 1 ? 1 : (r > 16 ? 16 : r);
  return r > nx ? nx : r;
}
// Group sizes used by a launch: from about one workgroup per CU (256) of rows, two of pairs, over
// all runs' rows, never above the per-grid limits.  A single grid of 512 rows keeps one pair and
// two rows per workgroup (one row: the field pass 9.0 -> 9.4 us); many small grids get grouped
// rows.  Groups of half the values as before hold less LDS, so more of a CU's workgroups hide
// each other's latency: 48 runs of 64^2 to 256^2 rows 12.3 -> 9.2 us, field 16.3 -> 12.9 (groups
// of 1024 12.1, but the step of 1024^2 69.4 -> 73.4), the step of 2048^2 with few particles 248
// -> 232 us (FP64 369 -> 341).
inline int pow2_floor(long long v) {
  int p = 1;
  while ((long long)p * 2 <= v) p *= 2;
  return p;
}
inline void fft_groups(long long rows_total, int nx, int ny, int* pp, int* rf) {
  const long long t = rows_total / 256, tp = rows_total / 1024;
  const int gr = t >= 1 ? pow2_floor(t) : 1, gp = tp >= 1 ? pow2_floor(tp) : 1;
  *rf = fft_rows_per_block(nx, ny) < gr ? fft_rows_per_block(nx, ny) : gr;
  *pp = fft_row_pairs_per_block(nx, ny) < gp ? fft_row_pairs_per_block(nx, ny) : gp;
}

struct FieldArgs {
  const RunDesc* runs;
  RunState* st;
  const unsigned long long* rho;     // [2][gsum]
  unsigned long long* rho_w;         // same buffer, written (zeroing of the next parity)
  const unsigned long long* rho_lo;  // FP64 only
  unsigned long long* rho_lo_w;
  long long gsum;
  double2* S;    // rho_hat, then phi_hat
  double2* Sx;   // Ex_hat
  double2* Sy;   // Ey_hat
  void* E;       // padded (Ex,Ey) pairs, float or double
  double* phi;   // optional node potential (may be NULL)
  const double2* tw;
  const int2* row_pair_items; int n_row_pair_items;
  const int2* col_items; int n_col_items;
  const int2* row_items; int n_row_items;
  double* partials;                  // [n_row_items] per-row-group field energy (may be NULL)
  double* diag;
  int nruns;
  int fp64;                          // particle precision (E type, rho words)
  int want_phi;                      // 1: phi instead of E (which stays as it was)
  int max_nx, max_ny;                // largest grid of the context (LDS sizing)
  int row_lds;                       // complex values per row-pass workgroup: the largest
                                     // max(fft_pp, fft_rf) * ny over the runs
  const double* rho_in;              // op mode: FP64 density input instead of rho (may be NULL)
  int clear_read;                    // 1: zero the charge words that are read (one buffer);
                                     // 0: zero the other parity's (the next push's target)
  // End-of-step work of the previous step run by extra workgroups of these kernels
  // (step_tail.h).  fold_finish: the rows pass writes the previous step's diagnostics row
  // (nruns workgroups after its row items), and the column pass advances the step counter
  // (so every kernel of this solve reads the counter one behind and adds fold_finish).
  // fold_scan: the rows, column and field passes run the fused sort's count-table scan
  // (fscan_part, fscan_base, fscan_rows) after their own items.
  int fold_finish;
  const double* ppush;               // push partials of the previous step (fold_finish)
  int fold_scan;
  int* ftable;
  int* fchunk_sums;
  int fstride;
  const int2* fscan_items; int nfscan_items;
  int* ftoff;                        // tile offsets of the order the next push writes
};
void launch_field(hipStream_t s, const FieldArgs& a, hipEvent_t* ev /* 4 events or NULL */);
// one-grid descriptor, state and items into device memory (all of them read by launch_field)
void launch_op_setup(hipStream_t s, const RunDesc& d, RunDesc* dd, RunState* st, int2* rp,
                     int nrp, int2* cl, int ncl);
// phi of a small grid in one launch; false (and nothing launched) when the grid is too large
bool launch_phi_one(hipStream_t s, const RunDesc& d, const double* rho, double* phi,
                    const double2* tw);
void launch_op_efield(hipStream_t s, const double* phi, double* ex, double* ey, int nx, int ny,
                      double lx, double ly);
// copy padded E (float/double pairs) of one run out to two FP64 node arrays
void launch_unpad_E(hipStream_t s, const void* E, int fp64, int nx, int ny, double* ex, double* ey);
// rho (fixed point, parity of current step) of one run to FP64 density incl. background
void launch_rho_to_double(hipStream_t s, const RunDesc* runs, RunState* st, int run,
                          const unsigned long long* rho, const unsigned long long* rho_lo,
                          long long gsum, int fp64, double background, double* out);

// ---- collision kernels (k_collide.hip)
struct MccArgs {
  float *x, *y, *vx, *vy;
  int* id;
  RunState* st;       // np / next_id / err of the run (device)
  long long pbase;    // particle base of the run
  int cap;
  double v_unit2_half_me_over_e;  // E[eV] = this * |v|^2
  double ng_vunit_dtphys;         // nu*dt = this * sigma(E) * |v|
  int null_any;                   // random words 0 .. null_last pass the null-collision test
  unsigned null_last;             // (mcc_null_range)
  double nu_max_dt;               // nu_max * dt_phys
  double mass_ratio2;             // 2 m_e / M
  uint64_t seed;
  long long* counts;              // [4]
  int* birth_count;
  int* birth_parent;              // [cap]
  float* birth_buf;               // [4*cap]
  int from_state_step;            // 1: take the step index from st->step
  int finish_after;               // 1: the step's end (counter advance) runs after this
                                  // stage, so st->step is this step's index (else its + 1)
  long long step;
  double* diag;                   // the run's diagnostics rows (may be NULL): the step's
                                  // collisions are added to column PIC_DIAG_NCOLL
  int* coll_list;                 // slots that pass the null-collision test, a region of
                                  // per_block entries per workgroup (mcc_list_layout)
  int* coll_partials;             // [blocks][4] collision counts of each k_mcc workgroup
  int* count_table;               // sort fused into the push, after its count step: the
                                  // count table, to which the births add their tiles (in
                                  // the row of the tail item that will push them); else NULL
};
// the random words that pass a null-collision test of probability p_coll
void mcc_null_range(double p_coll, int* any, unsigned* last);
// MCC collision list layout for n_upper particles: the grid of k_mcc and the list region
// of each workgroup (its grid-stride share); the list needs blocks * per_block entries
#define PIC_MCC_BLOCKS 2048
void mcc_list_layout(long long n_upper, int* blocks, int* per_block);
void launch_mcc(hipStream_t s, const MccArgs& a, int n_upper);
void launch_mcc_births(hipStream_t s, const MccArgs& a, unsigned long long* scratch,
                       unsigned long long* rho, long long gsum, const RunDesc* runs, int run,
                       int n_upper);
#define DSMC_SLOTS 32         // counters of accepted pairs
#define DSMC_SLOT_STRIDE 16   // a cache line apart
struct DsmcArgs {
  float *vx, *vy;
  const int* offsets;             // [ncells + 1] cell ranges in the sort's numbering
  float* gmax;                    // [ncells] per-cell maximum relative speed, row-major cell
  int ncells;
  int tile_shift;                 // offsets in the engine's tile-major numbering with tiles of
                                  // 1 << tile_shift cells a side; < 0: row-major already
  int tiles_y, ny;
  double coeff;
  uint64_t seed;
  long long step;
  const RunState* st;             // may be NULL (op mode uses `step`)
  int finish_after;               // 1: the step's end runs after this stage (st->step is this
                                  // step's index; else its + 1)
  long long* ncoll;
  unsigned long long* slots;      // [DSMC_SLOTS * DSMC_SLOT_STRIDE] zero between launches, or NULL
  double* diag;                   // the run's diagnostics rows (may be NULL)
};
void launch_dsmc(hipStream_t s, const DsmcArgs& a);

// ---- the reference's own collide arithmetic on an injected uniform stream (k_refcollide.hip)
#define REF_CHAIN_CHUNK 4096  // stream positions per chunk of the consumer-start resolution
// positions that m consumers can reach (at most 7 uniforms each): the part of a stream of nu
// that has to be resolved
inline long long ref_chain_stream(long long nu, long long m) { return nu / 7 < m ? nu : 7 * m; }
struct RefChainBufs {
  int2* maps;            // [7 * nchunks] (exit offset, consumers) per chunk and entry offset
  int* entry;            // [nchunks]
  long long* base;       // [nchunks] first consumer starting in the chunk
  long long* total;      // [1] consumers the stream starts
  long long* start;      // [m] stream position of each consumer
  long long* consumed;   // [1] uniforms taken by the m consumers, -1 if the stream is short
};
void launch_ref_chain(hipStream_t s, const double* u, long long nu, double prob, long long m,
                      RefChainBufs b);
void launch_mcc_reference(hipStream_t s, double* vx, double* vy, long long n, double prob,
                          const double* u, const long long* start);
void launch_ref_cell_keys(hipStream_t s, const double* x, const double* y, long long n, int nx,
                          int ny, double dx, double dy, int* keys, int* bad);
void launch_ref_nearest(hipStream_t s, const double* x, const double* y, long long n,
                        const int* keys, const int* perm, const int* offsets, int* target,
                        int* drawkey);
void launch_dsmc_reference(hipStream_t s, double* vx, double* vy, long long n, long long m,
                           double prob, const double* u, const long long* start,
                           const int* consumers, const int* target, double* m1, double* m2,
                           int* self, int* lastw, unsigned long long* ncoll);
