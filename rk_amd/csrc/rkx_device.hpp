// Device-side building blocks: right-hand sides, step control, reductions.
//
// Every floating-point expression keeps the reference's operand order and is
// compiled with -ffp-contract=off, so results equal the reference bitwise.
// A fused multiply-add is written explicitly only where the product is exact
// (a power-of-two scale: 2*y, 4*y), where fma(a, b, c) == c + a*b bitwise.
#pragma once

#include "rkx_internal.hpp"
#include "rkx_pow.hpp"

namespace rkx {

// Tables of libm_pow in constant memory (one copy per kernel translation unit).
static __constant__ pow_tables dev_pow_tables =
#include "rkx_pow_tables.inc"
    ;

// Vectors reached through an instance table are generic pointers to the
// compiler, which then emits FLAT memory instructions; those count against
// the LDS counter too, so every wait for LDS (before each barrier) would also
// wait for the global loads in flight.  Kernels that prefetch through such
// pointers view them in the global address space instead.
using gconst = const __attribute__((address_space(1))) double;
using gbyte = const __attribute__((address_space(1))) char;
using gmut = __attribute__((address_space(1))) double;
__device__ __forceinline__ gconst *as_global(const double *p) { return (gconst *) p; }
__device__ __forceinline__ gmut *as_global(double *p) { return (gmut *) p; }

using gmethod = const __attribute__((address_space(1))) dev_method;
__device__ __forceinline__ gmethod *as_global(const dev_method *m) { return (gmethod *) m; }

// Stores v to row[idx] in the lanes where keep holds, without a branch: the
// store goes through a buffer resource of the row (len doubles); the other
// lanes address past its end, and the hardware drops out-of-range buffer
// stores.  row must be wave-uniform (the resource lives in scalar registers).
// A branch around the store would split the surrounding straight-line code
// into scheduling regions the compiler cannot interleave.
using u32x2 = unsigned int __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void store_row_masked(gmut *row, int len, int idx, bool keep, double v)
{
  constexpr int kGfx9RawBuffer = 0x00020000;   // dword 3 of a raw gfx9 buffer resource
  // the row base in scalar registers (it is wave-uniform; said explicitly,
  // the resource needs no per-lane loop)
  const unsigned long long a = reinterpret_cast<unsigned long long>(row);
  const unsigned int lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(a));
  const unsigned int hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned int>(a >> 32));
  void *base = reinterpret_cast<void *>((static_cast<unsigned long long>(hi) << 32) | lo);
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
      base, 0, len * static_cast<int>(sizeof(double)), kGfx9RawBuffer);
  const int off = keep ? idx * static_cast<int>(sizeof(double)) : 0x7ffffff0;
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, 0);
}

// A value that is the same in every lane (a step coefficient), moved to
// scalar registers: loaded through a generic pointer it would otherwise
// occupy a vector register pair in every lane for the whole kernel.
__device__ __forceinline__ double wave_uniform(double x)
{
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readfirstlane(static_cast<int>(b));
  const int hi = __builtin_amdgcn_readfirstlane(static_cast<int>(b >> 32));
  return __longlong_as_double((static_cast<long long>(hi) << 32) |
                              static_cast<unsigned int>(lo));
}

// ---- BRUSS2D-MIX (src/problems/bruss2d-mix.c:66-206) ------------------------
// Laplacian numerator of one component at grid point (k, j) given its
// neighbours.  vN/vS already carry the Neumann mirror on the top/bottom rows
// (the reference's 2.0*y[i+-N2] equals y[i+N2] + y[i+N2] exactly), so only
// the column boundaries need their own operand order:
//   interior column:  ((vN + vS) + vW) + vE - 4 v
//   j == 0:           (vN + vS) + 2 vE - 4 v
//   j == N-1:         (vN + vS) + 2 vW - 4 v
__device__ __forceinline__ double bruss_lap_col(double vN, double vS, double vW, double vE,
                                                double v, int j, int N)
{
  const double t1 = vN + vS;
  double t2;
  if (j == 0)
    t2 = __builtin_fma(2.0, vE, t1);
  else if (j == N - 1)
    t2 = __builtin_fma(2.0, vW, t1);
  else
    t2 = (t1 + vW) + vE;
  return __builtin_fma(-4.0, v, t2);
}

// f_u = ((1 + u*u*v) - 4.4 u) + coef*lap_u ;  f_v = (3.4 u - u*u*v) + coef*lap_v
__device__ __forceinline__ void bruss_react(double u, double v, double lu, double lv,
                                            double coef, double &fu, double &fv)
{
  const double uuv = (u * u) * v;
  fu = ((1.0 + uuv) - 4.4 * u) + coef * lu;
  fv = (3.4 * u - uuv) + coef * lv;
}

// RHS of grid point cell = k*N + j reading a full state vector y (D form).
__device__ __forceinline__ void bruss_cell(const dev_ode &p, const double *__restrict__ y,
                                           int cell, double &fu, double &fv)
{
  const int N = p.N;
  const int N2 = N + N;
  const int k = cell / N;
  const int j = cell - k * N;
  const int i = k * N2 + 2 * j;
  const int iN = (k == 0) ? i + N2 : i - N2;
  const int iS = (k == N - 1) ? i - N2 : i + N2;
  const double2 c = *reinterpret_cast<const double2 *>(y + i);
  const double2 nN = *reinterpret_cast<const double2 *>(y + iN);
  const double2 nS = *reinterpret_cast<const double2 *>(y + iS);
  const double2 nW = (j > 0) ? *reinterpret_cast<const double2 *>(y + i - 2) : c;
  const double2 nE = (j < N - 1) ? *reinterpret_cast<const double2 *>(y + i + 2) : c;
  const double lu = bruss_lap_col(nN.x, nS.x, nW.x, nE.x, c.x, j, N);
  const double lv = bruss_lap_col(nN.y, nS.y, nW.y, nE.y, c.y, j, N);
  bruss_react(c.x, c.y, lu, lv, p.coef, fu, fv);
}

// ---- LV pair (src/problems/lv.c:69-77) ---------------------------------------
__device__ __forceinline__ void lv_pair(const dev_ode &p, double x, double y, double &fx,
                                        double &fy)
{
  fx = p.c0 * x - p.d0 * x * y;
  fy = p.d1 * x * y - p.c1 * y;
}

// ---- LV chain (periodic, d = 2; no reference counterpart) -------------------
//   x' = (c0 x - d0 x y) + D ((x_l + x_r) - 2x), likewise y.
__device__ __forceinline__ void chain_cell(const dev_ode &p, const double *__restrict__ y,
                                           int cell, double &fx, double &fy)
{
  const int l = (cell == 0) ? p.cells - 1 : cell - 1;
  const int r = (cell == p.cells - 1) ? 0 : cell + 1;
  const double2 c = *reinterpret_cast<const double2 *>(y + 2 * cell);
  const double2 a = *reinterpret_cast<const double2 *>(y + 2 * l);
  const double2 b = *reinterpret_cast<const double2 *>(y + 2 * r);
  double gx, gy;
  lv_pair(p, c.x, c.y, gx, gy);
  fx = gx + p.diff * __builtin_fma(-2.0, c.x, a.x + b.x);
  fy = gy + p.diff * __builtin_fma(-2.0, c.y, a.y + b.y);
}

__device__ __forceinline__ void rhs_cell(const dev_ode &p, const double *__restrict__ y,
                                         int cell, double &f0, double &f1)
{
  if (p.kind == RKX_BRUSS2D) {
    bruss_cell(p, y, cell, f0, f1);
  } else if (p.kind == RKX_LV) {
    const double2 c = *reinterpret_cast<const double2 *>(y + 2 * cell);
    lv_pair(p, c.x, c.y, f0, f1);
  } else {
    chain_cell(p, y, cell, f0, f1);
  }
}

// ---- error norm (include/tools.h:280-288) ------------------------------------
// Per component q = |e| / max(|y_new|, |y_old|); a zero divisor raises the
// 1.7e308 sentinel, a NaN quotient is skipped (fmax semantics).
__device__ __forceinline__ void err_term(double e, double yn, double yo, double &qmax,
                                         unsigned int &zero)
{
  const double d = fmax(fabs(yn), fabs(yo));
  if (d == 0.0)
    zero = 1u;
  else
    qmax = fmax(qmax, fabs(e) / d);
}

// ---- step control (include/tools.h:217-278, 191-198) ------------------------

// Every workgroup thread t of nt computes its share of the premultiplied
// coefficients of the next step from the raw table: the same products h*A,
// h*b, h*(b - b_hat) as premult, each written to both places it is read from.
__device__ inline void premult_block(const dev_method &m, int s, double h, dev_coef &c, int t,
                                     int nt)
{
  const int total = s * s + 2 * s;
  for (int idx = t; idx < total; idx += nt) {
    if (idx < s * s) {
      const int i = idx / s, j = idx - (idx / s) * s;
      if (j < i) {
        const double v = h * m.A[i * RKX_MAX_STAGES + j];
        c.hA[i * RKX_MAX_STAGES + j] = v;
        c.col[j][i - j - 1] = v;
      }
    } else if (idx < s * s + s) {
      const int i = idx - s * s;
      const double v = h * m.b[i];
      c.hb[i] = v;
      c.col[i][s - i - 1] = v;
    } else {
      const int i = idx - s * s - s;
      const double v = h * m.e[i];
      c.he[i] = v;
      c.col[i][s - i] = v;
    }
  }
}

// The loop variables for the host's thread (one thread; see host_view).
__device__ inline void show(host_view *w, const step_vars &v)
{
  __hip_atomic_store(&w->t, v.t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&w->h, v.h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&w->acc, v.acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&w->rej, v.rej, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(&w->cur, v.cur, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (v.done)
    __hip_atomic_store(&w->done, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Full-storage forms: the first kernel of a step that reports (and of every
// step past the end) shows what the control at the end of the step before
// left.  A kernel ends when its stores to the host's memory have arrived: in
// the control itself, on every step, they made 1000 LV pairs' steps 9 %
// longer (HEUN2 in D's form).
__device__ __forceinline__ void show_last(const state *st, bool report)
{
  if ((report || st->v.done) && st->view && blockIdx.x == 0 && threadIdx.x == 0)
    show(st->view, st->v);
}

// The trace of an attempt made from v (one thread).
__device__ inline void trace_attempt(state *st, const step_vars &v, double err)
{
  const int attempt = v.acc + v.rej;
  if (st->trace && attempt < st->trace_cap) {
    st->trace[3 * attempt + 0] = v.t;
    st->trace[3 * attempt + 1] = v.h;
    st->trace[3 * attempt + 2] = err;
  }
}

// Full-storage forms: runs in exactly one thread after every workgroup has
// folded its maximum into st->err_bits / st->zero_div.  Resets the
// accumulators for the next step.  The new h uses libm_pow, the C library's pow restated bitwise, so the
// device reproduces the reference's step sizes without a host round trip.
// Returns whether the next step's coefficients need premultiplying (device
// control), which the caller's workgroup does with premult_block.
__device__ inline bool dev_control(state *st)
{
  const unsigned long long bits = atomicOr(&st->err_bits, 0ull);
  const unsigned int zero = atomicOr(&st->zero_div, 0u);
  const double q = __longlong_as_double(static_cast<long long>(bits));
  st->err_bits = 0ull;
  st->zero_div = 0u;
  st->blocks_done = 0u;
  st->err = zero ? fmax(1.7E308, q) : q;
  if (st->ctrl == RKX_CTRL_HOST)
    return false;
  trace_attempt(st, st->v, st->err);
  double px = 0.0, py = 0.0;
  const bool need = ctrl_decide(st->v, st->err, px, py);
  ctrl_finish(st->v, need, need ? libm_pow(px, py, dev_pow_tables) : 0.0);
  return true;
}

// ---- reductions -----------------------------------------------------------------
// A lane's double moved by a DPP control (lanes without a source keep v).
template <int CTRL>
__device__ __forceinline__ double dpp_keep(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = static_cast<int>(b), hi = static_cast<int>(b >> 32);
  const int ml = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
  const int mh = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
  return __longlong_as_double((static_cast<long long>(mh) << 32) | static_cast<unsigned int>(ml));
}
// Maximum over the wavefront, valid in lane 63: shifts within rows of 16
// lanes, then each row's last lane broadcast to the next row(s).  All in
// registers; six exchanges through LDS (shuffles) took 0.3 us at the end of
// every step.
__device__ __forceinline__ double wave_max63(double v)
{
  v = fmax(v, dpp_keep<0x111>(v));   // row_shr:1
  v = fmax(v, dpp_keep<0x112>(v));   // row_shr:2
  v = fmax(v, dpp_keep<0x114>(v));   // row_shr:4
  v = fmax(v, dpp_keep<0x118>(v));   // row_shr:8
  v = fmax(v, dpp_keep<0x142>(v));   // row_bcast:15
  v = fmax(v, dpp_keep<0x143>(v));   // row_bcast:31
  return v;
}

// ---- step control of the fused kernels --------------------------------------
// The tables of libm_pow spread over a wavefront: lane l holds entries l and
// l + 64, loaded once at the start of a kernel beside its other first loads,
// so the two lookups are lane reads instead of two dependent trips to memory.
// For arguments that are the same in every lane.
struct lane_pow_tables {
  double lg[2][3];
  unsigned long long ex[2][2];
  __device__ void load()
  {
    const int lane = threadIdx.x & 63;
    for (int q = 0; q < 2; ++q) {
      for (int c = 0; c < 3; ++c)
        lg[q][c] = dev_pow_tables.logt[lane + 64 * q][c];
      for (int c = 0; c < 2; ++c)
        ex[q][c] = dev_pow_tables.expt[2 * (lane + 64 * q) + c];
    }
  }
  static __device__ unsigned long long lane_of(unsigned long long b, int src)
  {
    const unsigned int lo = __builtin_amdgcn_readlane(static_cast<unsigned int>(b), src);
    const unsigned int hi = __builtin_amdgcn_readlane(static_cast<unsigned int>(b >> 32), src);
    return (static_cast<unsigned long long>(hi) << 32) | lo;
  }
  __device__ double log_at(int i, int c) const
  {
    const int u = __builtin_amdgcn_readfirstlane(i);
    const unsigned long long b =
        __builtin_bit_cast(unsigned long long, u >= 64 ? lg[1][c] : lg[0][c]);
    return __builtin_bit_cast(double, lane_of(b, u & 63));
  }
  __device__ unsigned long long exp_at(int k, int c) const
  {
    const int u = __builtin_amdgcn_readfirstlane(k);
    return lane_of(u >= 64 ? ex[1][c] : ex[0][c], u & 63);
  }
};

// The (instance, tile within it) a workgroup works on: entry `tile` of the
// launch's table, or tile `tile` of its one instance.
template <class INST>
__device__ __forceinline__ int2 launch_tile(const fused_launch<INST> &a, int tile)
{
  if (!a.tiles)
    return make_int2(0, tile);
  const int2 t = a.tiles[tile];
  return make_int2(__builtin_amdgcn_readfirstlane(t.x), __builtin_amdgcn_readfirstlane(t.y));
}
// That instance, in scalar registers (said explicitly: merged from two
// sources, its fields would otherwise occupy vector registers throughout the
// kernel, 40 of them in the row sweep).
template <class INST>
__device__ __forceinline__ INST launch_inst(const fused_launch<INST> &a, int i)
{
  if (!a.tiles)
    return a.one;
  static_assert(sizeof(INST) % 4 == 0, "whole words");
  using gword = const __attribute__((address_space(1))) int;
  gword *src = (gword *) (a.insts + i);
  int w[sizeof(INST) / 4];
  for (unsigned k = 0; k < sizeof(INST) / 4; ++k)
    w[k] = __builtin_amdgcn_readfirstlane(src[k]);
  INST r;
  __builtin_memcpy(&r, w, sizeof(INST));
  return r;
}

using gslot = const __attribute__((address_space(1))) step_slot;

// The loop variables of a slot, through the global address space (scalar loads).
__device__ __forceinline__ step_vars slot_vars(gslot *s)
{
  step_vars v;
  v.t = s->v.t;
  v.h = s->v.h;
  v.te = s->v.te;
  v.tol = s->v.tol;
  v.acc = s->v.acc;
  v.rej = s->v.rej;
  v.cur = s->v.cur;
  v.done = s->v.done;
  v.step_limit = s->v.step_limit;
  v.ord = s->v.ord;
  return v;
}

// The loop variables as the host sees them (one thread).
__device__ inline void publish(state *st, const step_vars &v, double err)
{
  st->v.t = v.t;
  st->v.h = v.h;
  st->v.acc = v.acc;
  st->v.rej = v.rej;
  st->v.cur = v.cur;
  st->v.done = v.done;
  st->err = err;
}

struct step_now {
  double h;
  int cur, done;
};
struct step_lds {
  double h;
  int cur, done;
  unsigned long long *err;   // this step's error accumulator, for step_fold: kept
                             // here, it occupies no scalar registers meanwhile
};

// The start of a fused step, called by every thread of every workgroup: the
// pending control of the attempt before, in the first wavefront, handed to
// the others through LDS (one barrier).  tile: the workgroup's tile within
// the instance; tile 0 writes the next slot and clears the accumulators of
// the launch after next.
__device__ inline step_now step_begin(const step_refs &R, int r, int tile, step_lds &x)
{
  const bool leader = tile == 0;
  if (threadIdx.x < 64) {
    gslot *s = (gslot *) &R.ring->slot[r];
    using gerr = const __attribute__((address_space(1))) double;
    static_assert(kErrLines == 8, "half a row of lanes");
    double err = *(gerr *) &R.ring->err[r][threadIdx.x & 7].bits;
    step_vars v = slot_vars(s);
    const int pending = s->pending, traced = s->traced;
    lane_pow_tables T;
    T.load();
    if (pending) {
      err = fmax(err, dpp_keep<0x111>(err));
      err = fmax(err, dpp_keep<0x112>(err));
      err = fmax(err, dpp_keep<0x114>(err));     // lane 7: all eight
      err = __builtin_bit_cast(
          double, lane_pow_tables::lane_of(__builtin_bit_cast(unsigned long long, err), 7));
      if (traced && leader && threadIdx.x == 0)
        trace_attempt(R.st, v, err);
      double px = 0.0, py = 0.0;
      const bool need = ctrl_decide(v, err, px, py);
      ctrl_finish(v, need, need ? libm_pow(px, py, T) : 0.0);
      if (leader && threadIdx.x == 0) {
        publish(R.st, v, err);
        if (R.view)
          show(R.view, v);
      }
    }
    if (threadIdx.x == 0) {
      x.h = v.h;
      x.cur = v.cur;
      x.done = v.done;
      x.err = &R.ring->err[(r + 1) & (kRing - 1)][tile & (kErrLines - 1)].bits;
      if (leader) {
        step_slot &o = R.ring->slot[(r + 1) & (kRing - 1)];
        o.v = v;
        o.pending = !v.done;
        o.traced = traced;
      }
    }
    if (leader && threadIdx.x < kErrLines)
      __hip_atomic_store(&R.ring->err[(r + 2) & (kRing - 1)][threadIdx.x].bits, 0ull,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  step_now n;
  n.h = wave_uniform(x.h);
  n.cur = __builtin_amdgcn_readfirstlane(x.cur);
  n.done = __builtin_amdgcn_readfirstlane(x.done);
  return n;
}

// The end of a fused step, called by every thread of a workgroup of NW (at
// most 16) wavefronts: folds the error maximum (zero: some divisor was 0, the
// 1.7e308 sentinel) into the accumulator the next launch reads.  red holds NW
// doubles of LDS.  The waves' maxima are read side by side by the lanes of
// one row and folded there: a loop over them in one thread, its count read
// from the dispatch packet, took 0.6 us at the end of every step.
template <int NW>
__device__ __forceinline__ void step_fold(const step_lds &x, double qmax, unsigned int zero,
                                          double *red)
{
  static_assert(NW >= 1 && NW <= 16, "one row of lanes");
  if (zero)
    qmax = fmax(qmax, 1.7E308);
  qmax = wave_max63(qmax);
  if ((threadIdx.x & 63) == 63)
    red[threadIdx.x >> 6] = qmax;
  __syncthreads();
  if (threadIdx.x < 64) {
    double m = red[threadIdx.x % NW];
    m = fmax(m, dpp_keep<0x111>(m));
    m = fmax(m, dpp_keep<0x112>(m));
    m = fmax(m, dpp_keep<0x114>(m));
    m = fmax(m, dpp_keep<0x118>(m));
    using gacc = __attribute__((address_space(1))) unsigned long long;
    if (threadIdx.x == 15)
      __hip_atomic_fetch_max((gacc *) x.err,
                             static_cast<unsigned long long>(__double_as_longlong(m)),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// ---- end of a full-storage step ----------------------------------------------
// Folds each thread's (qmax, zero) into the step accumulators and runs the
// control in the last workgroup of the grid to finish.  Must be called by all
// threads of the block.  red must hold blockDim.x/64 doubles of LDS.
__device__ inline void block_finish(state *st, double qmax, unsigned int zero, double *red,
                                    unsigned int *zred)
{
  const unsigned int nblocks = gridDim.x * gridDim.y * gridDim.z;
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + 63) >> 6;
  qmax = wave_max63(qmax);
  const unsigned long long zb = __ballot(zero != 0u);
  if (lane == 63) {
    red[wid] = qmax;
    zred[wid] = zb ? 1u : 0u;
  }
  __syncthreads();
  __shared__ int is_last;
  if (threadIdx.x == 0) {
    double m = red[0];
    unsigned int z = zred[0];
    for (int w = 1; w < nw; ++w) {
      m = fmax(m, red[w]);
      z |= zred[w];
    }
    atomicMax(&st->err_bits, static_cast<unsigned long long>(__double_as_longlong(m)));
    if (z)
      atomicOr(&st->zero_div, 1u);
    __threadfence();
    const unsigned int prev = atomicAdd(&st->blocks_done, 1u);
    is_last = (prev == nblocks - 1u);
  }
  __syncthreads();
  if (is_last) {                       // uniform over the workgroup
    __shared__ int pm;
    __shared__ double hn;
    if (threadIdx.x == 0) {
      __threadfence();
      pm = dev_control(st) ? 1 : 0;
      hn = st->v.h;
    }
    __syncthreads();
    if (pm)
      premult_block(*st->meth, st->s, hn, *st->coef, static_cast<int>(threadIdx.x),
                    static_cast<int>(blockDim.x));
  }
}

}  // namespace rkx
