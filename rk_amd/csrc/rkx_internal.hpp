// Internal declarations shared by the rkx host runtime and the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <string>
#include <thread>
#include <vector>

#include "../../include/rkx.h"

namespace rkx {

int fail(int code, const std::string &msg);

#define RKX_HIP(call)                                                              \
  do {                                                                             \
    hipError_t e_ = (call);                                                        \
    if (e_ != hipSuccess)                                                          \
      return ::rkx::fail(RKX_EDEVICE, std::string(#call " failed: ") +             \
                                          hipGetErrorString(e_));                 \
  } while (0)

// Problem descriptor as the kernels see it (by value in kernel arguments).
struct dev_ode {
  int kind;
  int n;        // components
  int cells;    // n / 2: grid points (BRUSS2D), pairs (LV), cells (chain)
  int N;        // BRUSS2D grid size
  double coef;  // BRUSS2D (alpha*(N-1))*(N-1), the reference's alpha*N1*N1
  double c0, d0, d1, c1;
  double diff;
};

dev_ode make_dev_ode(const rkx_ode &p);

// Method coefficients in device memory: A row-major [RKX_MAX_STAGES^2], then
// b, e = b - b_hat (src/impl/seq/D.c:40-41), c.
struct dev_method {
  double A[RKX_MAX_STAGES * RKX_MAX_STAGES];
  double b[RKX_MAX_STAGES];
  double e[RKX_MAX_STAGES];
  double c[RKX_MAX_STAGES];
  // grouped by the stage that scatters with them, as dev_coef::col but not
  // multiplied by h: col[i] = {A[i+1][i], ..., A[s-1][i], b[i], e[i]}.  The
  // fused kernels form h * col themselves at their start (the same products
  // as premult), so their steps need no premultiplication in the control.
  double col[RKX_MAX_STAGES][RKX_MAX_STAGES + 2];
};

// Premultiplied coefficients of the current step (premult, src/methods.c:43-58):
// hA = h*A (j < i), hb = h*b, he = h*e.  Written by the step control together
// with the new h; read as uniform values by every kernel of the next step.
struct dev_coef {
  double hA[RKX_MAX_STAGES * RKX_MAX_STAGES];
  double hb[RKX_MAX_STAGES];
  double he[RKX_MAX_STAGES];
  // the same values grouped by the stage that consumes them: stage i scatters
  // with col[i] = {hA[i+1][i], ..., hA[s-1][i], hb[i], he[i]} (contiguous, so
  // a fused kernel loads one stage's coefficients with one scalar load)
  double col[RKX_MAX_STAGES][RKX_MAX_STAGES + 2];
};

// What the step control reads and updates: the loop variables of one solve.
struct step_vars {
  double t, h, te, tol;
  int acc, rej;
  int cur;                           // which of the two y buffers holds y
  int done;                          // the step loop has ended
  int step_limit;
  int ord;
};

// The step ring of an instance with a fused kernel (one launch per attempted
// step).  Launch number k of an instance reads slot k & 3, runs the step
// control of the attempt before it (pending) in every workgroup from the
// error maxima in err[k & 3], makes its own attempt, folds its error into
// err[(k+1) & 3] and leaves the loop variables it worked with in slot
// (k+1) & 3.  Every workgroup computes the same control from the same values,
// so a step ends with one atomic maximum per workgroup and no workgroup waits
// for another: counting the workgroups that finished and running the control
// in the last of them cost two atomics in a row, a device-wide fence and the
// control itself at the end of every step, with nothing to overlap them (one
// pair of LV: 7.1 us per step).
constexpr int kRing = 4;
// Accumulators of one step: workgroups fold into accumulator (tile & 7), each
// on a cache line of its own, and the next launch reads all of them with one
// load.  256 workgroups' atomics on one word queue for 2.4 us (a kernel of
// nothing else: 4.0 us a launch against 1.66 us).
constexpr int kErrLines = 8;
struct alignas(64) step_slot {
  step_vars v;
  int pending;                       // the attempt from v awaits its control
  int traced;                        // state::trace is set
};
struct alignas(128) err_line {
  unsigned long long bits;           // atomic maximum: bits of a double >= 0
};
struct step_ring {
  step_slot slot[kRing];
  err_line err[kRing][kErrLines];
};
// The error norm of a step: the maximum of its accumulators (doubles >= 0, so
// their bits compare as the values do).
__host__ __device__ inline double ring_err(const err_line (&err)[kErrLines])
{
  unsigned long long b = 0ull;
  for (int k = 0; k < kErrLines; ++k)
    b = err[k].bits > b ? err[k].bits : b;
  return __builtin_bit_cast(double, b);
}

struct state;

// A solve's loop variables in pinned host memory, where its thread watches
// them while it keeps the GPU supplied with steps: written by the step
// control of every step (a posted write, no copy and no wait on the GPU's
// side; a copy of the state after every chunk of steps left the GPU idle for
// 18 us).  done is written last, after the others are visible.
struct host_view {
  double t, h;
  int acc, rej, cur, done;
};

// Integration state of one solve, resident in device memory.  Written only by
// the step control (the last workgroup of a full-storage step, the first
// workgroup of a fused one, or the host).
struct alignas(64) state {
  step_vars v;
  double err;                        // error norm of the last attempt
  unsigned long long err_bits;       // atomicMax accumulator (bits of a double >= 0)
  unsigned int zero_div;             // some divisor max(|y|,|y_old|) was 0
  unsigned int blocks_done;          // last-workgroup detection
  int ctrl;                          // RKX_CTRL_*
  int trace_cap;
  int s;                             // stages
  double *trace;                     // device buffer, 3 doubles per attempt
  const dev_method *meth;            // raw coefficients for the premultiplication
  dev_coef *coef;                    // premultiplied coefficients of the next step
  step_ring *ring;                   // fused kernels (nullptr: full storage)
  host_view *view;                   // full-storage forms: as step_refs::view
};

// premult of the raw table by h (identical on host and device)
__host__ __device__ inline void premult(const dev_method &m, int s, double h, dev_coef &c)
{
  for (int i = 0; i < s; ++i) {
    for (int j = 0; j < i; ++j)
      c.hA[i * RKX_MAX_STAGES + j] = h * m.A[i * RKX_MAX_STAGES + j];
    c.hb[i] = h * m.b[i];
    c.he[i] = h * m.e[i];
  }
  for (int i = 0; i < s; ++i) {
    for (int l = i + 1; l < s; ++l)
      c.col[i][l - i - 1] = c.hA[l * RKX_MAX_STAGES + i];
    c.col[i][s - i - 1] = c.hb[i];
    c.col[i][s - i] = c.he[i];
  }
}

// Step control of include/tools.h:235-278, split at the one libm call.
// ctrl_decide: accept/reject with err, advance t and the counters, and give
// pow's arguments x = tol/err, y = 1/(ord+1).  Returns true when the new h
// needs p = pow(x, y) (variable step size).
__host__ __device__ inline bool ctrl_decide(step_vars &v, double err, double &x, double &y)
{
  if (v.tol <= 0.0) {                  // fixed step size (tools.h:258-263)
    v.t += v.h;
    v.acc += 1;
    v.cur ^= 1;
    return false;
  }
  if (err <= v.tol) {                  // accept (tools.h:264-270)
    v.t += v.h;
    v.acc += 1;
    v.cur ^= 1;
  } else {                             // reject: y stays in the other buffer
    v.rej += 1;
  }
  x = v.tol / err;
  y = 1.0 / (v.ord + 1.0);
  return true;
}

// ctrl_finish: h_new_acc/h_new_rej with p (tools.h:221-233), then the
// for-increment h = fmin(h, te - t) and the loop test of FOR_ALL_GRIDPOINTS
// (tools.h:191-198).
__host__ __device__ inline void ctrl_finish(step_vars &v, bool used_pow, double p)
{
  if (used_pow)
    v.h = v.h * fmin(2.0, fmax(0.5, 0.9 * p));
  v.h = fmin(v.h, v.te - v.t);
  const int attempts = v.acc + v.rej;
  v.done = !((v.t < v.te) && (v.step_limit <= 0 || attempts < v.step_limit));
}

// ---- host runtime helpers (rkx_host.cpp) ------------------------------------
int check_ode(const rkx_ode *p);
int check_method(const rkx_method *m);
void fill_dev_method(const rkx_method &m, dev_method &d);
double initial_h(double H, double tol, int limit, double h0);   // src/tools.c:25-36
int default_stream(hipStream_t *out);
// the step control on the host: ctrl_decide/ctrl_finish with the C library's pow
void host_finish(step_vars &v, double err);

// Device blocks kept between solves (rkx_pool.cpp): take a block of
// `bytes` (to the page: *got), give it back once no stream uses it.
int pool_take(void **out, size_t bytes, size_t *got);
void pool_give(void *p, size_t bytes);
void pool_release();
// hipMalloc, again without the device's kept blocks if it fails
int device_alloc(void **out, size_t bytes);

// What a fused kernel is given of an instance's device-side step state.
struct step_refs {
  state *st;             // published loop variables, trace buffer
  step_ring *ring;
  const dev_method *meth;
  host_view *view;       // nullptr: nobody watches
};
// Rings of instances about to run their first step (nothing pending).
step_ring make_ring(const step_vars &v, bool traced);

// Kernel launchers (rkx_kernels_*.hip).  All return hipError_t of the launch.
hipError_t launch_eval_rng(const dev_ode &p, int i, int j, const double *y, double *f,
                           hipStream_t s);
hipError_t launch_d_step(const dev_ode &p, const dev_coef *cf, int s, state *st,
                         double *y0, double *y1, double *w, double *dy, double *err,
                         bool report, hipStream_t stream);
// Stage-fused step of independent LV pairs (rkx_kernels_lvpairs.hip): every
// table with 2, 3, 4, 7, 8 or 13 stages
bool pairs_supported(const dev_ode &p, const rkx_method &m);
// cf: room for the step's products, used by tables of 13 stages
hipError_t launch_lv_step(const dev_ode &p, int s, const step_refs &R, dev_coef *cf, double *y0,
                          double *y1, int r, hipStream_t stream);
// Runs the pending step control of n states (those without a ring, and those
// that have ended, are left alone), publishes it, and moves each ring on to
// slot 0 (rkx_kernels_step.hip): after launches that ended on ring slot r,
// before the host reads the states for good or starts again at slot 0.
hipError_t launch_step_flush(state *st, int n, int r, hipStream_t stream);

// Gather forms A, E, F (src/impl/seq/A.c, E.c, F.c): non-zero patterns of the
// raw table (zero_pattern, src/methods.c:24-39) as bit masks, bit i of rowA[l]
// for A[l][i], of b for b[i], of e for b[i] - b_hat[i]
struct gather_masks {
  unsigned rowA[RKX_MAX_STAGES];
  unsigned b, e;
};
gather_masks make_gather_masks(const rkx_method &m);
// one attempted step of form RKX_IMPL_A/E/F: v holds s vectors of n, w0 (and
// w1 for F) one each
hipError_t launch_gather_step(int form, const dev_ode &p, const dev_coef *cf, int s,
                              const gather_masks &nz, state *st, double *y0, double *y1,
                              double *v, double *w0, double *w1, bool report, hipStream_t stream);

struct sweep_cfg {
  int waves;     // wavefronts per workgroup (strip width 64*waves lanes)
  int rows;      // band height in grid rows
};
// One BRUSS2D instance as the fused kernel sees it (device memory).  A launch
// covers a table of (instance, tile) pairs, so one kernel steps many
// instances, each with its own state, coefficients and step control.
//
// Columns: nwide strips of OC output columns, each band of a strip one
// workgroup.  When the columns left over after the widest strips fit a strip
// of half the lanes (split), they form a narrow last strip whose bands are
// paired: one workgroup carries two bands of it, each on half of its waves,
// so the narrow strip costs half a strip of workgroups.
struct sweep_inst {
  int N;                 // grid size
  int R;                 // band height (rows)
  int OC;                // output columns per wide strip
  int nstrips, nbands;   // strips (wide + narrow), bands per strip
  int nwide;             // wide strips: tiles 0 .. nwide*nbands-1
  int split;             // 1: a narrow last strip, (nbands+1)/2 paired tiles
  int ntiles;            // workgroups that share this state per step
  double coef;           // (alpha*(N-1))*(N-1)
  double *y0, *y1;       // the two y buffers
  step_refs ref;         // the kernel forms h*A etc. from ref.meth
};

bool sweep_supported(const dev_ode &p, const rkx_method &m);
int sweep_pattern(const rkx_method &m);   // compiled zero pattern (0: none)
sweep_cfg sweep_default_cfg(const dev_ode &p, const rkx_method &m);
// Band height a tile gets for `rows` requested rows: unchanged, or for tables
// whose fused kernel runs whole trips of its s+1-row ring, rounded up so that
// the band's rows + 2(s-1) row iterations, less the peeled ones
// (peeled_iters), fill whole trips, the last up to an exit (trip_iters).
int sweep_band_rows(int pattern, int s, int rows);
// Whether every ghost row a band of an N-row grid loads lies within a single
// reflection about row 0 / N-1 (the kernel's fast form); false for grids
// shorter than the halo, prefetch and ring: those launch the general form.
bool sweep_single_reflect(int pattern, int s, int N);
// The same for one instance's tiles: the paired bands of a narrow strip both
// run the full band height, so the last of them may load rows further past
// N-1 than a band of its own height.
bool sweep_inst_single_reflect(int pattern, int s, const sweep_inst &I);
// Row iterations of tile t of an instance (its band, or the shorter last
// band, plus the 2(s-1) halo rows; paired bands run the full band height).
int sweep_tile_iters(int pattern, int s, const sweep_inst &I, int t);
sweep_inst make_sweep_inst(const dev_ode &p, const rkx_method &m, const sweep_cfg &c,
                           const step_refs &ref, double *y0, double *y1);
// A launch of a fused kernel over many instances (device tables) or, with
// tiles == nullptr, over the one instance it is given by value (its fields
// then come with the kernel's arguments, which saves a step of its chain of
// dependent loads).  r: the ring slot every instance of the launch reads.
template <class INST>
struct fused_launch {
  INST one;
  const INST *insts;
  const int2 *tiles;
  int ntiles;
  int r;
};
// gen: the general reflection form (some instance fails sweep_single_reflect)
hipError_t launch_sweep(int pattern, int K, bool gen, const fused_launch<sweep_inst> &a,
                        hipStream_t stream);
// the VERNER65 and DOPRI87 kernels (translation units of their own: many stages
// take long to build)
hipError_t launch_sweep_verner65(int K, bool gen, const fused_launch<sweep_inst> &a,
                                 hipStream_t stream);
int resident_blocks_verner65(int K);
hipError_t launch_sweep_dopri87(int K, bool gen, const fused_launch<sweep_inst> &a,
                                hipStream_t stream);
int resident_blocks_dopri87(int K);
// workgroups of the fused kernel resident per CU for a pattern and strip
// width; 0: the strip is too wide for that table's kernel
int sweep_resident_blocks(int pattern, int K);

// One BRUSS2D instance as the tile kernel sees it.  Strips of 64 columns and
// bands of W*C rows that overlap by their halos; the last ones end at the
// grid's edge, so the grid's own edges cost no halo.
struct tile_inst {
  int N;
  int nstrips, nbands;
  int ntiles;            // nstrips * nbands workgroups
  double coef;
  double *y0, *y1;
  step_refs ref;
};
// Tile shapes of the kernel: C rows in each of 8 waves of 64 columns.
constexpr int kTileWaves = 8;
constexpr int kTileRows[] = {2, 3, 4, 6};
constexpr int kNumTileShapes = sizeof(kTileRows) / sizeof(kTileRows[0]);
bool tile_supported(int pattern);            // tables of up to 8 stages
tile_inst make_tile_inst(const dev_ode &p, const rkx_method &m, int shape, const step_refs &ref,
                         double *y0, double *y1);
// The shape a single grid runs in, or -1: the row sweep is the faster form.
int tile_default_shape(const dev_ode &p, const rkx_method &m);
hipError_t launch_tile_step(int pattern, int shape, const tile_inst &I, int r, hipStream_t stream);
// Grids of one workgroup (rkx_kernels_run.hip): up to `steps` attempts in one
// launch, each with its control; I: N, coef, the buffers and ref.
bool run_supported(int pattern, int N);
hipError_t launch_run(int pattern, const tile_inst &I, int r, int steps, hipStream_t stream);

// Pieces of n rows or columns in tiles of `full` of them with a halo on either
// inner side: the first and the last piece lose one halo, those between two.
inline int tile_pieces(int n, int full, int halo)
{
  const int rest = n - 2 * (full - halo);
  return n <= full ? 1 : 2 + (rest > 0 ? (rest + full - 2 * halo - 1) / (full - 2 * halo) : 0);
}

// A full-storage form of a BRUSS2D step, stages in groups
// (rkx_kernels_groups.hip).
struct stage_group {
  int N, s;
  int i0;                // the launch's first stage
  int nstrips, nbands, ntiles;
  int r;                 // ring slot, the same for every kernel of a step
  double coef;
  double *y0, *y1;
  double *w, *dy, *err;  // D: w_1..w_{s-1} one after another; A, E, F: w holds v_0..
  step_refs ref;
};
constexpr int kGroupBlocks = 512;   // two workgroups on a compute unit
// all of a step's kernels, form RKX_IMPL_D, A, E or F; a: without i0 and the
// tile counts
hipError_t launch_groups(int form, const stage_group &a, const gather_masks &nz,
                         hipStream_t stream);

// One LV chain instance as the fused chain kernel sees it (device memory).
struct chain_inst {
  int cells;             // M
  int tile_out;          // output cells per segment
  int ntiles;            // segments (a wavefront each) per step
  int nwg;               // workgroups per step (their waves loop over segments)
  double c0, d0, d1, c1, diff;
  double *y0, *y1;
  step_refs ref;         // the kernel forms h*A etc. from ref.meth
};

bool chain_supported(const dev_ode &p, const rkx_method &m);
// C: cells per lane, 2..4 (the kernel's instance)
chain_inst make_chain_inst(const dev_ode &p, const rkx_method &m, int C, const step_refs &ref,
                           double *y0, double *y1);
int chain_default_cells(const dev_ode &p, const rkx_method &m);
// many chains in one launch fill the chip whatever C is: the least halo
constexpr int kChainBatchCells = 4;
hipError_t launch_chain(int pattern, int C, const fused_launch<chain_inst> &a, hipStream_t stream);

// The step of one instance with a step ring: which kernel (kernels, for the
// full-storage forms in groups of stages), and its launch.
struct fused_plan {
  enum kind_t { kPairs, kChain, kTile, kSweep, kGroups } kind = kSweep;
  dev_ode dp{};
  step_refs ref{};
  dev_coef *coef = nullptr;
  double *y0 = nullptr, *y1 = nullptr;
  int s = 0, pattern = 0;
  int shape = 0;           // tile; chain: cells per lane
  bool general = false;    // sweep: general ghost rows
  int waves = 0;           // sweep
  fused_launch<chain_inst> chain{};
  tile_inst tile{};
  fused_launch<sweep_inst> sweep{};
  int form = 0;            // groups: RKX_IMPL_D, A, E, F on BRUSS2D
  stage_group groups{};
  gather_masks nz{};
  // one attempted step; r: the ring slot the kernel reads
  hipError_t launch(int r, hipStream_t stream);
  // > 0: launch_many makes up to this many, each with its control
  int many = 0;
  tile_inst run{};
  hipError_t launch_many(int r, hipStream_t stream);
};
// The plan of a problem and table with a fused kernel.  rows, waves: the
// caller's row-sweep tile (0: chosen); y0, y1: the two y buffers.
int make_fused_plan(const rkx_ode &p, const rkx_method &m, int rows, int waves,
                    const step_refs &ref, dev_coef *coef, double *y0, double *y1, fused_plan *out);

}  // namespace rkx
