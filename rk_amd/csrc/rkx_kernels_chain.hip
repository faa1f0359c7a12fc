// Stage-fused step of the diffusive periodic LV chain (cells c = 0..M-1, the
// pair (x_c, y_c) at components 2c, 2c+1, access distance 2):
//   x' = (c0 x - d0 x y) + D ((x_{c-1} + x_{c+1}) - 2x),
//   y' = (d1 x y - c1 y) + D ((y_{c-1} + y_{c+1}) - 2y).
// No reference counterpart; the scheme is the one-dimensional analogue of the
// BRUSS2D forms.  A wavefront owns a segment of 64*C cells (C cells per lane,
// both components) and evaluates all s stages of the scatter form
// (block-inline.h:253-320) with every accumulator in registers; a lane's
// outer neighbours are DPP shifts of the next lanes' edge cells, so the waves
// of a workgroup never wait for each other between the step's start and its
// end.  A segment overlaps its neighbours by s cells on each side (each
// stage's valid region shrinks by one cell) and writes 64*C - 2s cells of
// y_new.  Periodic ghost cells are loaded by index wrap.  Per step the kernel
// reads y once (plus the halo) and writes y_new once: two vectors resident.
//
// Bound by the step's start and end: at 5e5 cells the waves wait 52 % of their
// cycles and the VALUs are busy 40 % of the time.  us per step, DOPRI54,
// against one segment of 1024 cells to a workgroup with an LDS exchange and a
// barrier per stage: 1e5 cells 6.2 / 8.6, 3e5 8.6 / 12.9, 5e5 10.6 / 12.9, 1e6
// 17.2 / 20.9.
#include "rkx_patterns.hpp"

namespace rkx {
namespace {

constexpr int kCB = 256;     // lanes per workgroup: four waves, a segment each
// waves per SIMD that a kernel of C cells per lane is register-allocated for
constexpr int chain_occ(int C) { return 6 - C; }

__device__ __forceinline__ int wrap(long long c, int M)
{
  long long m = c % M;
  return static_cast<int>(m < 0 ? m + M : m);
}

// a lane's neighbours' values (the outermost lanes get 0: they are halo)
template <int CTRL>
__device__ __forceinline__ double chain_shift(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

template <class P, int C>
__global__ __launch_bounds__(kCB) __attribute__((amdgpu_waves_per_eu(chain_occ(C)))) void
k_chain(fused_launch<chain_inst> a)
{
  constexpr int s = P::s;
  constexpr int kT = 64 * C;
  __shared__ double red[kCB / 64];
  __shared__ step_lds head;

  const int T = a.ntiles;
  const int b = blockIdx.x;
  const int x8 = b & 7, q = T >> 3, rm = T & 7;
  const int tile = x8 * q + min(x8, rm) + (b >> 3);
  const int2 td = launch_tile(a, tile);
  const chain_inst I = launch_inst(a, td.x);
  const int M = I.cells;
  step_coefs<P> kc;
  kc.load(as_global(I.ref.meth));
  const step_now sn = step_begin(I.ref, a.r, td.y, head);
  if (sn.done)
    return;
  using cell2 = double __attribute__((ext_vector_type(2)));
  using gcell = const __attribute__((address_space(1))) cell2;
  using gout = __attribute__((address_space(1))) cell2;
  gcell *__restrict__ y = (gcell *) (sn.cur ? I.y1 : I.y0);
  gout *__restrict__ yn = (gout *) (sn.cur ? I.y0 : I.y1);
  dev_ode p{};
  p.c0 = I.c0;
  p.d0 = I.d0;
  p.d1 = I.d1;
  p.c1 = I.c1;
  const double D = I.diff;
  kc.scale(sn.h);

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double qmax = 0.0;
  unsigned int zero = 0u;
  for (int seg = td.y * (kCB / 64) + wv; seg < I.ntiles; seg += I.nwg * (kCB / 64)) {
    const long long out0 = static_cast<long long>(seg) * I.tile_out;  // first output cell
    const long long c0 = out0 - s + static_cast<long long>(lane) * C; // this lane's first cell
    cell2 yv[C];
    cell2 acc[C][s + 1];                 // [0] dy, [1..s-1] w_l, [s] err
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      yv[c] = y[wrap(c0 + c, M)];
    });

    static_for<s>([&](auto itg) {
      constexpr int i = decltype(itg)::value;
      cell2 cv[C];
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        cv[c] = (i == 0) ? yv[c] : acc[c][i];
      });
      const cell2 lft = {chain_shift<0x138>(cv[C - 1].x), chain_shift<0x138>(cv[C - 1].y)};
      const cell2 rgt = {chain_shift<0x130>(cv[0].x), chain_shift<0x130>(cv[0].y)};
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        cell2 l = lft, r = rgt;
        if constexpr (c > 0)
          l = cv[c - 1];
        if constexpr (c < C - 1)
          r = cv[c + 1];
        const cell2 v = cv[c];
        double gx, gy;
        lv_pair(p, v.x, v.y, gx, gy);
        const double fx = gx + D * __builtin_fma(-2.0, v.x, l.x + r.x);
        const double fy = gy + D * __builtin_fma(-2.0, v.y, l.y + r.y);
        const double *ki = kc.k[i];
        if constexpr (i == 0) {
          static_for<s>([&](auto ltg) {
            constexpr int lq = decltype(ltg)::value;
            if constexpr (lq >= 1)
              acc[c][lq] = nzA<P>(lq, 0) ? cell2{v.x + ki[lq - 1] * fx, v.y + ki[lq - 1] * fy} : v;
          });
          acc[c][0] = cell2{ki[s - 1] * fx, ki[s - 1] * fy};
          acc[c][s] = cell2{ki[s] * fx, ki[s] * fy};
        } else {
          static_for<s>([&](auto ltg) {
            constexpr int lq = decltype(ltg)::value;
            if constexpr (lq > i && nzA<P>(lq, i)) {
              acc[c][lq].x += ki[lq - i - 1] * fx;
              acc[c][lq].y += ki[lq - i - 1] * fy;
            }
          });
          if constexpr ((P::b >> i) & 1u) {
            acc[c][0].x += ki[s - i - 1] * fx;
            acc[c][0].y += ki[s - i - 1] * fy;
          }
          if constexpr ((P::e >> i) & 1u) {
            acc[c][s].x += ki[s - i] * fx;
            acc[c][s].y += ki[s - i] * fy;
          }
        }
      });
    });
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      const long long cell = c0 + c;
      const int local = lane * C + c;
      if (local >= s && local < kT - s && cell < M) {
        const cell2 o = {yv[c].x + acc[c][0].x, yv[c].y + acc[c][0].y};
        yn[cell] = o;
        err_term(acc[c][s].x, o.x, yv[c].x, qmax, zero);
        err_term(acc[c][s].y, o.y, yv[c].y, qmax, zero);
      }
    });
  }
  step_fold<kCB / 64>(head, qmax, zero, red);
}

}  // namespace

bool chain_supported(const dev_ode &p, const rkx_method &m)
{
  const int pat = pattern_of(m);
  return p.kind == RKX_LV_CHAIN && pat >= 1 && pat <= 6;
}

// Cells per lane, 2, 3 or 4: the count whose busiest SIMD has the least to do,
// in cells per lane (its segments times C), where every further round of
// resident waves costs about as much as 3 more (a round that is not full runs
// at the latency of its stages).  Measured, us per step for 2 / 3 / 4 cells:
// 1e5 cells 6.2 / 6.9 / 7.8, 3e5 8.6 / 8.5 / 9.7, 5e5 13.1 / 10.6 / 11.9,
// 7e5 15.6 / 17.0 / 15.5, 1e6 20.4 / 17.2 / 17.8.
int chain_default_cells(const dev_ode &p, const rkx_method &m)
{
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 1) {
    (void) hipGetLastError();
    cus = 256;
  }
  int best = 4;
  long long least = -1;
  for (int C = 2; C <= 4; ++C) {
    const long long segs = make_chain_inst(p, m, C, {}, nullptr, nullptr).ntiles;
    const long long simds = 4LL * cus, waves = simds * chain_occ(C);
    const long long cost =
        (segs + simds - 1) / simds * C + 3 * ((segs + waves - 1) / waves - 1);
    if (least < 0 || cost < least) {
      least = cost;
      best = C;
    }
  }
  return best;
}

chain_inst make_chain_inst(const dev_ode &p, const rkx_method &m, int C, const step_refs &ref,
                           double *y0, double *y1)
{
  chain_inst I{};
  I.cells = p.cells;
  I.tile_out = 64 * C - 2 * m.s;
  I.ntiles = (p.cells + I.tile_out - 1) / I.tile_out;
  // all resident on 256 compute units at once; longer chains loop
  const int wgs = (I.ntiles + kCB / 64 - 1) / (kCB / 64);
  I.nwg = wgs < 256 * chain_occ(C) ? wgs : 256 * chain_occ(C);
  I.c0 = p.c0;
  I.d0 = p.d0;
  I.d1 = p.d1;
  I.c1 = p.c1;
  I.diff = p.diff;
  I.y0 = y0;
  I.y1 = y1;
  I.ref = ref;
  return I;
}

hipError_t launch_chain(int pattern, int C, const fused_launch<chain_inst> &a, hipStream_t stream)
{
  if (a.ntiles <= 0)
    return hipSuccess;
  return dispatch_pattern(pattern, [&](auto pat) {
    using P = decltype(pat);
    const dim3 g(a.ntiles), b(kCB);
    switch (C) {
    case 2: hipLaunchKernelGGL((k_chain<P, 2>), g, b, 0, stream, a); break;
    case 3: hipLaunchKernelGGL((k_chain<P, 3>), g, b, 0, stream, a); break;
    case 4: hipLaunchKernelGGL((k_chain<P, 4>), g, b, 0, stream, a); break;
    default: return hipErrorInvalidConfiguration;
    }
    return hipGetLastError();
  });
}

}  // namespace rkx
