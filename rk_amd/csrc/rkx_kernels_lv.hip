// Ensemble of independent Lotka-Volterra pairs: a lane integrates one
// 2-component system at a time x' = c0 x - d0 x y, y' = d1 x y - c1 y (src/problems/lv.c
// with per-system constants) over [t0, te] with its own step size and
// accept/reject.  The arithmetic of every attempted step is that of the
// reference's seq D (block-inline.h:253-320, tools.h:191-288) on a system of
// size 2, so each system's result equals a plain single solve of that system
// (identical accepted/rejected sequences and bitwise the same y).  The step
// control runs in the thread, with libm_pow: the C library's pow restated, so
// every new h equals the reference's (thousands of systems step at once; no
// host round trip).
#include "rkx_device.hpp"

#include <algorithm>

namespace rkx {
namespace {

constexpr int kLvBlock = 256;
constexpr int kLvMaxAttempts = 1 << 24;   // every thread stops after this many

// method table in constant memory: A row-major, b, e = b - b_hat
struct lv_method {
  double A[RKX_MAX_STAGES * RKX_MAX_STAGES];
  double b[RKX_MAX_STAGES];
  double e[RKX_MAX_STAGES];
  int s, ord;
};

// A wavefront runs as long as its slowest system, and the systems' step
// counts differ widely (the benchmark's 262144: 148 on average, up to 567), so
// with one system per thread more than half of all lane-steps were idle.
// Here a wave owns every gridDim-th block of 64 systems and hands the next of
// them to its lanes as those finish, kRefill at a time: a refill costs the
// wave a trip to memory (about one step), idle lanes cost their share of every
// step, and the two balance at about 7 lanes.  No counter is shared: the sum
// over a wave's few hundred systems varies little.
constexpr int kRefill = 8;

// A wave takes its systems in windows of kWindow, the ones that promise the
// most steps first, so that no lane starts a long one when the others are
// nearly done (the benchmark's ensemble: a wave takes 700 steps instead of
// 1050, 590 if no lane ever idled).  Only the order depends on the estimate,
// never a result.
constexpr int kWindow = 256;

// Grows with a system's number of steps: the rates of its linear part and how
// far its orbit is from the fixed point (the conserved quantity
// d1 x - c1 log x + d0 y - c0 log y above its minimum); correlation with the
// steps taken 0.94 over the benchmark's ensemble.
__device__ inline float lv_length(const double *__restrict__ prm, const double *__restrict__ y0)
{
  const float a = static_cast<float>(prm[0]), b = static_cast<float>(prm[1]),
              c = static_cast<float>(prm[2]), d = static_cast<float>(prm[3]),
              x = static_cast<float>(y0[0]), y = static_cast<float>(y0[1]);
  const float v = (c * x - d * __logf(x)) + (b * y - a * __logf(y));
  const float v0 = (d - d * __logf(d / c)) + (a - a * __logf(a / b));
  const float k = a + d + (v - v0);
  return k > 0.0f && k < 1e30f ? k : 0.0f;       // also for constants out of its domain
}

// Keeps a uniform value in a vector register.
__device__ __forceinline__ void in_vector(double &x) { __asm__("" : "+v"(x)); }

template <int S>
__global__ __launch_bounds__(kLvBlock) __attribute__((amdgpu_waves_per_eu(2))) void
k_lv_ensemble(int count, lv_method m, const double *__restrict__ prm,
              const double *__restrict__ y0, double *__restrict__ yout, double t0, double te,
              double tol, double h0, int step_limit, int *__restrict__ acc_out,
              int *__restrict__ rej_out)
{
  __shared__ pow_tables tab;                     // lanes look up different entries
  __shared__ float keys[kLvBlock / 64][kWindow];
  __shared__ unsigned char turn[kLvBlock / 64][kWindow];
  for (unsigned k = threadIdx.x; k < sizeof(pow_tables) / 8; k += kLvBlock)
    reinterpret_cast<double *>(&tab)[k] = reinterpret_cast<const double *>(&dev_pow_tables)[k];
  constexpr bool kInLds = S > 8;
  __shared__ alignas(16) double table[kInLds ? S : 1][(S + 3) / 2 * 2];
  auto table_at = [&](int i, int l) -> double {
    return l < S ? m.A[l * RKX_MAX_STAGES + i] : l == S ? m.b[i] : m.e[i];
  };
  if constexpr (kInLds)
    for (int q = threadIdx.x; q < S * (S + 2); q += kLvBlock)
      table[q / (S + 2)][q % (S + 2)] = table_at(q / (S + 2), q % (S + 2));
  __syncthreads();

  const int lane = threadIdx.x & 63;
  const int nw = gridDim.x * (kLvBlock / 64);
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (kLvBlock / 64) +
                                                  static_cast<int>(threadIdx.x >> 6));
  const int blocks = (count + 63) >> 6;
  // this wave's systems are numbered 0 .. last-1; next: the first not handed out
  const int last = wave < blocks ? 64 * ((blocks - wave + nw - 1) / nw) : 0;
  const int wid = threadIdx.x >> 6;
  auto system_of = [&](int n) -> size_t {
    return (static_cast<size_t>(n >> 6) * nw + wave) * 64 + (n & 63);
  };
  // Ranks the window that starts at w0 by lv_length, longest first, into
  // turn[wid]: every lane counts, for its four systems, the ones before them.
  auto rank_window = [&](int w0) {
    float mine[kWindow / 64];
    int rank[kWindow / 64];
    for (int q = 0; q < kWindow / 64; ++q) {
      const size_t n = system_of(w0 + 64 * q + lane);
      const bool there = w0 + 64 * q < last && n < static_cast<size_t>(count);
      mine[q] = there ? lv_length(prm + 4 * n, y0 + 2 * n) : -1.0f;   // the rest at the end
      keys[wid][64 * q + lane] = mine[q];
      rank[q] = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int j = 0; j < kWindow; ++j) {
      const float other = keys[wid][j];
      for (int q = 0; q < kWindow / 64; ++q)
        rank[q] += (other > mine[q] || (other == mine[q] && j < 64 * q + lane)) ? 1 : 0;
    }
    for (int q = 0; q < kWindow / 64; ++q)
      turn[wid][rank[q]] = static_cast<unsigned char>(64 * q + lane);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  int next = 0;
  int window_end = 0;
  bool have = false, active = false;             // holds a system; still integrates it
  size_t k = 0;
  dev_ode p{};
  double y[2] = {0.0, 0.0};
  step_vars st{};
  st.te = te;
  st.tol = tol;
  st.ord = m.ord;
  // Few stages: the bound on attempts is part of the step limit, one test less
  // in each (64 systems, 1000 fixed steps: RK4 451 -> 415 us, RKF23 387 -> 365;
  // the schedule of 7 stages is the worse for it, 639 -> 704).
  constexpr bool kOneLimit = S <= 4;
  st.step_limit = step_limit;
  if constexpr (kOneLimit)
    st.step_limit = step_limit > 0 ? min(step_limit, kLvMaxAttempts) : kLvMaxAttempts;
  // Coefficient l of stage i: A[l][i] for i < l < S, b[i] for l = S, e[i] for
  // S + 1.  Those of 4 stages fit the scalar registers, and leave vector
  // registers for five waves (94 instead of 122).  The 44 of 8 stages do not
  // fit beside the rest and came back from spills with two lane reads each;
  // at one wave per SIMD vector registers are there for them.  The 104 of 13
  // stages are read from LDS for every attempt: left to the compiler, 265
  // scalar registers were spilled (262144 systems, tol 1e-6: 506 us, 363 from
  // LDS; 1000 fixed steps 9615, 5703).
  double kept[kInLds ? 1 : S][S + 2];
  if constexpr (!kInLds) {
#pragma unroll
    for (int i = 0; i < S; ++i) {
#pragma unroll
      for (int l = i + 1; l < S + 2; ++l) {
        kept[i][l] = table_at(i, l);
        if constexpr (S > 4)
          in_vector(kept[i][l]);
      }
    }
  }
  auto coef = [&](int l, int i) -> double {
    if constexpr (kInLds)
      return table[i][l];
    else
      return kept[i][l];
  };
  auto attempt = [&]() {
    if constexpr (kInLds)
      __asm__ volatile("" ::: "memory");          // not kept in registers between attempts
    const double h = st.h;
    double w[S][2], dy[2], er[2];
    // first stage
    double f0, f1;
    lv_pair(p, y[0], y[1], f0, f1);
#pragma unroll
    for (int l = 1; l < S; ++l) {
      const double a = h * coef(l, 0);
      w[l][0] = y[0] + a * f0;
      w[l][1] = y[1] + a * f1;
    }
    dy[0] = (h * coef(S, 0)) * f0;
    dy[1] = (h * coef(S, 0)) * f1;
    er[0] = (h * coef(S + 1, 0)) * f0;
    er[1] = (h * coef(S + 1, 0)) * f1;
    // intermediate and last stages
#pragma unroll
    for (int i = 1; i < S; ++i) {
      lv_pair(p, w[i][0], w[i][1], f0, f1);
#pragma unroll
      for (int l = i + 1; l < S; ++l) {
        const double a = h * coef(l, i);
        w[l][0] += a * f0;
        w[l][1] += a * f1;
      }
      const double hb = h * coef(S, i), he = h * coef(S + 1, i);
      dy[0] += hb * f0;
      dy[1] += hb * f1;
      er[0] += he * f0;
      er[1] += he * f1;
    }
    const double yn[2] = {y[0] + dy[0], y[1] + dy[1]};
    double q = 0.0;
    unsigned int zero = 0u;
    err_term(er[0], yn[0], y[0], q, zero);
    err_term(er[1], yn[1], y[1], q, zero);
    const int cur_before = st.cur;
    double px = 0.0, py = 0.0;
    const bool need = ctrl_decide(st, zero ? fmax(1.7E308, q) : q, px, py);
    if (st.cur != cur_before) {          // accepted: y <- y_new
      y[0] = yn[0];
      y[1] = yn[1];
    }
    ctrl_finish(st, need, need ? libm_pow(px, py, tab) : 0.0);
    active = !st.done && (kOneLimit || st.acc + st.rej < kLvMaxAttempts);
  };
  auto store = [&]() {
    yout[2 * k] = y[0];
    yout[2 * k + 1] = y[1];
    acc_out[k] = st.acc;
    rej_out[k] = st.rej;
    have = false;
  };
  // While systems are left to hand out, each attempt starts with a count of
  // the idle lanes; behind that, and for a wave of 64 systems from the start,
  // every lane just runs to its end (the count and the branches around it made
  // 64 systems' attempts 10 % longer with 4 stages and 18 % with 2: 3000
  // attempts 2303 -> 2103 us with RK4, 2022 -> 1714 with HEUN2).
  while (next < last) {
    const unsigned long long idle = __ballot(!active);
    const int nidle = __popcll(idle);
    if (nidle < kRefill) {
      if (active)
        attempt();
      continue;
    }
    if (have && !active)
      store();
    if (next == window_end) {
      if (last > 64)                             // more systems than lanes
        rank_window(next);
      window_end = min(next + kWindow, last);
    }
    const int mine = next + static_cast<int>(__popcll(idle & ((1ull << lane) - 1ull)));
    if (!active && mine < window_end) {
      k = system_of(last > 64 ? (next & ~(kWindow - 1)) + turn[wid][mine & (kWindow - 1)] : mine);
      if (k < static_cast<size_t>(count)) {
        p.c0 = prm[4 * k + 0];
        p.d0 = prm[4 * k + 1];
        p.d1 = prm[4 * k + 2];
        p.c1 = prm[4 * k + 3];
        y[0] = y0[2 * k];
        y[1] = y0[2 * k + 1];
        st.t = t0;
        st.h = h0;
        st.acc = st.rej = 0;
        st.done = !(t0 < te);
        have = true;
        active = !st.done;
      }
    }
    next = min(next + nidle, window_end);
  }
  while (active)
    attempt();
  if (have)
    store();
}

}  // namespace
}  // namespace rkx

using namespace rkx;

extern "C" int rkx_lv_ensemble(int count, const double *params_dev, const double *y0_dev,
                               double *y_dev, double t0, double te, const rkx_method *m,
                               double tol, double h0, int step_limit, int *acc_dev, int *rej_dev,
                               void *stream)
{
  if (count < 1 || !params_dev || !y0_dev || !y_dev || !acc_dev || !rej_dev || h0 <= 0.0)
    return fail(RKX_EINVAL, "rkx_lv_ensemble: bad argument (h0 must be > 0)");
  if (count > (1 << 30))
    return fail(RKX_EINVAL, "rkx_lv_ensemble: at most 2^30 systems per call");
  if (int rc = check_method(m))
    return rc;
  lv_method lm{};
  for (int i = 0; i < m->s; ++i) {
    for (int j = 0; j < i; ++j)
      lm.A[i * RKX_MAX_STAGES + j] = m->A[i][j];
    lm.b[i] = m->b[i];
    lm.e[i] = m->b[i] - m->b_hat[i];
  }
  lm.s = m->s;
  lm.ord = m->ord;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!s)
    if (int rc = default_stream(&s))
      return rc;
  // With error control, at most one wave per SIMD; more systems than lanes take
  // turns (see k_lv_ensemble).  One wave issues a step in 1.3 us (8 stages),
  // two on a SIMD in about twice that: 262144 systems, VERNER65, tol 1e-8:
  // 1.24 ms with one, 1.32 ms with two, 1.8 ms with one system per thread.
  // Fixed steps, and tables without an error estimate, give every system the
  // same number of attempts: no lane waits for another, and waves that hide
  // each other's latency are worth more, so each lane gets one system.  262144
  // systems, 1000 fixed steps, us, taking turns / a system a lane: HEUN2 1518 /
  // 786, RK4 2075 / 1219, RKF23 1723 / 1103, DOPRI54 2759 / 2245, VERNER65
  // 3084 / 2549.
  int cus = 0, dev = 0;
  RKX_HIP(hipGetDevice(&dev));
  RKX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const bool even = tol <= 0.0 || !m->has_emb;
  const int all = (count + kLvBlock - 1) / kLvBlock;   // 4 waves a workgroup
  const int grid = even ? all : std::min(all, cus);
#define RKX_LV_CASE(S_)                                                                      \
  case S_:                                                                                   \
    hipLaunchKernelGGL(k_lv_ensemble<S_>, dim3(grid), dim3(kLvBlock), 0, s, count, lm,      \
                       params_dev, y0_dev, y_dev, t0, te, tol, h0, step_limit, acc_dev,      \
                       rej_dev);                                                             \
    break;
  switch (m->s) {
    RKX_LV_CASE(2)
    RKX_LV_CASE(3)
    RKX_LV_CASE(4)
    RKX_LV_CASE(7)
    RKX_LV_CASE(8)
    RKX_LV_CASE(13)
  default:
    return fail(RKX_EINVAL, "rkx_lv_ensemble: no kernel for this stage count");
  }
#undef RKX_LV_CASE
  RKX_HIP(hipGetLastError());
  RKX_HIP(hipStreamSynchronize(s));
  return RKX_OK;
}
