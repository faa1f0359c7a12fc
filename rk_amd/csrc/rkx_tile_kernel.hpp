// Stage-fused BRUSS2D step in square-ish tiles (the kernel template): the form
// for grids that do not fill the chip with the row sweep's bands.
//
// The row sweep (rkx_sweep_kernel.hpp) walks a band row by row: with bands of
// a few rows each step is a chain of R + 2(s-1) row iterations, a barrier
// each, however small the grid (DOPRI54: 11 us, DOPRI87 excepted, with most
// CUs idle or in the halo).  Here a workgroup of W waves holds a tile of 64
// columns x W*C rows, both components, and runs the s stages over the whole
// tile: s - 1 barriers a step.
//
// Lane = column, wave = C consecutive rows, so of a cell's four neighbours
// the two horizontal ones are DPP shifts of the lane's neighbours, the
// vertical ones the lane's own registers, except across waves: each wave
// leaves its first and last row in LDS once a stage.  u and v of a cell share
// a lane (u*u*v once, no exchange of the other component).
//
// Every stage's valid region shrinks by one cell, so a tile yields 64 - 2s
// columns and W*C - 2(s-1) rows (the first stage reads one more row of y on
// either side from memory); waves whose rows no later stage needs leave
// their stage out.  At the domain's edges nothing is lost: the first strip
// starts at column 0 and the last ends at column N-1, so the shift itself
// brings in the zero that the reference's column boundary needs in the place
// of the missing neighbour (its operand order is (vN + vS) + 2 vE, in place
// of ((vN + vS) + vW) + vE), and the factors mW, mE make the other one 2.
// Rows 0 and N-1 take their one neighbour twice (2.0*y == y + y).
//
// Bound by the latency of the step's start, the s stages and its end: at N =
// 128 (DOPRI54, 87 workgroups) the waves wait for memory and barriers 59 % of
// their cycles and the VALUs of the compute units in use are busy 28 % of the
// time, at N = 301 (VERNER65, 174 workgroups) 51 % and 37 %.
#pragma once

#include "rkx_patterns.hpp"

namespace rkx {
namespace {

// a lane's left (column - 1) and right (column + 1) neighbour; 0 beyond the wave
template <int CTRL>
__device__ __forceinline__ double wave_shift(double v)
{
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}
__device__ __forceinline__ double from_left(double v) { return wave_shift<0x138>(v); }    // wave_shr:1
__device__ __forceinline__ double from_right(double v) { return wave_shift<0x130>(v); }   // wave_shl:1

// Where a wave's cells lie, for a stage.
struct tile_place {
  int N, row;                  // the wave's (or half wave's) first row
  bool left, right;            // the lane's column is 0, N - 1
  double mE, mW, coef;
};

// Stage i of a wave's C rows: the derivatives, then their terms in the row's
// accumulators ([0] dy, [1..s-1] w_l, [s] err).  yu, yv: y with the row on
// either side; nu, nv, su, sv: the rows beyond the wave's of this stage's w.
// HALVES: a wave holds two rows side by side, in 32 lanes each.
template <class P, int C, int i, bool SMALL, bool HALVES>
__device__ __forceinline__ void tile_stage(const tile_place &t, const double *ki,
                                           const double (&yu)[C + 2], const double (&yv)[C + 2],
                                           double nu, double nv, double su, double sv,
                                           double (&au)[C][P::s + 1], double (&av)[C][P::s + 1])
{
  constexpr int s = P::s;
  // stage i of every row of the wave, before its accumulators change
  double fu[C], fv[C];
  static_for<C>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    auto wu = [&](auto kt) -> double {
      constexpr int k = decltype(kt)::value;
      if constexpr (i == 0)
        return yu[k + 1];
      else if constexpr (k < 0)
        return nu;
      else if constexpr (k >= C)
        return su;
      else
        return au[k][i];
    };
    auto wvv = [&](auto kt) -> double {
      constexpr int k = decltype(kt)::value;
      if constexpr (i == 0)
        return yv[k + 1];
      else if constexpr (k < 0)
        return nv;
      else if constexpr (k >= C)
        return sv;
      else
        return av[k][i];
    };
    const double u = wu(int_c<c>{}), v = wvv(int_c<c>{});
    double un = wu(int_c<c - 1>{}), vn = wvv(int_c<c - 1>{});
    double us = wu(int_c<c + 1>{}), vs = wvv(int_c<c + 1>{});
    if constexpr (c == 0) {
      const bool top = t.row + c == 0;
      un = top ? us : un;
      vn = top ? vs : vn;
    }
    if constexpr (SMALL || c == C - 1) {
      const bool bot = t.row + c == t.N - 1;
      us = bot ? un : us;
      vs = bot ? vn : vs;
    }
    double uE = from_right(u), vE = from_right(v);
    double uW = from_left(u), vW = from_left(v);
    if constexpr (HALVES) {                    // lane 32 starts a row of its own
      uW = t.left ? 0.0 : uW;
      vW = t.left ? 0.0 : vW;
    }
    if constexpr (SMALL) {                     // the column after the last
      uE = t.right ? 0.0 : uE;
      vE = t.right ? 0.0 : vE;
    }
    // ((vN + vS) + vW) + vE - 4c; 1, 2 and 4 times are exact
    const double lu = __builtin_fma(
        -4.0, u, __builtin_fma(t.mE, uE, __builtin_fma(t.mW, uW, un + us)));
    const double lv = __builtin_fma(
        -4.0, v, __builtin_fma(t.mE, vE, __builtin_fma(t.mW, vW, vn + vs)));
    bruss_react(u, v, lu, lv, t.coef, fu[c], fv[c]);
  });
  static_for<C>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    if constexpr (i == 0) {
      static_for<s>([&](auto lt) {
        constexpr int l = decltype(lt)::value;
        if constexpr (l >= 1) {
          au[c][l] = nzA<P>(l, 0) ? yu[c + 1] + ki[l - 1] * fu[c] : yu[c + 1];
          av[c][l] = nzA<P>(l, 0) ? yv[c + 1] + ki[l - 1] * fv[c] : yv[c + 1];
        }
      });
      au[c][0] = ki[s - 1] * fu[c];
      av[c][0] = ki[s - 1] * fv[c];
      au[c][s] = ki[s] * fu[c];
      av[c][s] = ki[s] * fv[c];
    } else {
      static_for<s>([&](auto lt) {
        constexpr int l = decltype(lt)::value;
        if constexpr (l > i && nzA<P>(l, i)) {
          au[c][l] += ki[l - i - 1] * fu[c];
          av[c][l] += ki[l - i - 1] * fv[c];
        }
      });
      if constexpr ((P::b >> i) & 1u) {
        au[c][0] += ki[s - i - 1] * fu[c];
        av[c][0] += ki[s - i - 1] * fv[c];
      }
      if constexpr ((P::e >> i) & 1u) {
        au[c][s] += ki[s - i] * fu[c];
        av[c][s] += ki[s - i] * fv[c];
      }
    }
  });
}

// SMALL: grids narrower or shorter than a tile, whose last row and column may
// lie anywhere in it.
//
// The arguments are scalars, the ones the first loads need in front: the
// hardware hands a kernel its leading scalar arguments in registers
// (build.py asks for 16), so those loads do not wait for a trip to the
// argument block first.
template <class P, int C, int W, bool SMALL>
__global__ __launch_bounds__(64 * W) void
k_tile(step_ring *ring, const dev_method *meth, double *y0, double *y1, int r, int ntiles, int N,
       int nbands, int nstrips, double coef, state *st, host_view *view)
{
  constexpr int s = P::s;
  constexpr int H = W * C;
  __shared__ double2 edge[2][W][2][64];          // first and last row of each wave
  __shared__ double red[W];
  __shared__ step_lds head;

  // XCD-aware tile order, as in the row sweep (N = 512: 11.7 us per step, and
  // 12.6 with the tiles in grid order)
  const int b = blockIdx.x;
  const int x = b & 7, q = ntiles >> 3, rm = ntiles & 7;
  const int tile = x * q + min(x, rm) + (b >> 3);
  const int strip = tile / nbands, band = tile - strip * nbands;
  const step_refs ref{st, ring, meth, view};
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // columns [c0, c1) and rows [r0, r1) of y_new; the tile starts at (tr, tc)
  constexpr int SC = 64 - 2 * s, SR = H - 2 * (s - 1);
  const int tc = SMALL ? 0 : min(strip * SC, N - 64);
  const int c0 = strip == 0 ? 0 : strip * SC + s;
  const int c1 = strip == nstrips - 1 ? N : strip * SC + 64 - s;
  const int tr = N < H ? 0 : min(band * SR, N - H);
  const int r0 = band == 0 ? 0 : band * SR + (s - 1);
  const int r1 = band == nbands - 1 ? N : band * SR + H - (s - 1);
  const int col = tc + lane;
  const int row = tr + wv * C;                   // the wave's first row
  const bool left = col == 0, right = col == N - 1;
  const tile_place T{N, row, left, right, left ? 2.0 : 1.0, right ? 2.0 : 1.0, coef};

  // Everything that comes from memory is asked for before the control is
  // waited for: the table's columns, and y (the wave's rows and the row on
  // either side) from both of its buffers, of which the control names one.
  using cell2 = double __attribute__((ext_vector_type(2)));
  using gcell = const __attribute__((address_space(1))) cell2;
  using gout = __attribute__((address_space(1))) cell2;
  step_coefs<P> kc;
  kc.load(as_global(meth));
  const int ccol = SMALL ? min(col, N - 1) : col;
  cell2 ya[2][C + 2];
  static_for<C + 2>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    const int k = max(0, min(row + c - 1, N - 1));
    const unsigned at = static_cast<unsigned>(k) * static_cast<unsigned>(N) +
                        static_cast<unsigned>(ccol);
    ya[0][c] = ((gcell *) y0)[at];
    ya[1][c] = ((gcell *) y1)[at];
  });
  const step_now sn = step_begin(ref, r, tile, head);
  if (sn.done)
    return;                                      // uniform over the instance's tiles
  gout *__restrict__ yn = (gout *) (sn.cur ? y0 : y1);
  double yu[C + 2], yv[C + 2];
  static_for<C + 2>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    yu[c] = sn.cur ? ya[1][c].x : ya[0][c].x;
    yv[c] = sn.cur ? ya[1][c].y : ya[0][c].y;
  });
  kc.scale(sn.h);

  // [0] dy, [1..s-1] w_l, [s] err
  double au[C][s + 1], av[C][s + 1];
  static_for<s>([&](auto itg) {
    constexpr int i = decltype(itg)::value;
    // rows whose stage i reaches a row of y_new
    const bool need = row + C > r0 - (s - 1 - i) && row < r1 + (s - 1 - i);
    double nu = 0.0, nv = 0.0, su = 0.0, sv = 0.0;   // rows beyond the wave's
    if constexpr (i == 0) {
      nu = yu[0];
      nv = yv[0];
      su = yu[C + 1];
      sv = yv[C + 1];
    } else {
      __syncthreads();
      const double2 up = edge[i & 1][max(wv - 1, 0)][1][lane];
      const double2 dn = edge[i & 1][min(wv + 1, W - 1)][0][lane];
      nu = up.x;
      nv = up.y;
      su = dn.x;
      sv = dn.y;
    }
    if (!need)
      return;
    tile_stage<P, C, i, SMALL, false>(T, kc.k[i], yu, yv, nu, nv, su, sv, au, av);
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      if constexpr (i + 1 < s) {
        if constexpr (c == 0)
          edge[(i + 1) & 1][wv][0][lane] = make_double2(au[c][i + 1], av[c][i + 1]);
        if constexpr (c == C - 1)
          edge[(i + 1) & 1][wv][1][lane] = make_double2(au[c][i + 1], av[c][i + 1]);
      }
    });
  });

  double qmax = 0.0;
  unsigned int zero = 0u;
  static_for<C>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    const int k = row + c;
    if (k >= r0 && k < r1 && col >= c0 && col < c1) {
      const cell2 o = {yu[c + 1] + au[c][0], yv[c + 1] + av[c][0]};
      yn[static_cast<unsigned>(k) * static_cast<unsigned>(N) + static_cast<unsigned>(col)] = o;
      err_term(au[c][s], o.x, yu[c + 1], qmax, zero);
      err_term(av[c][s], o.y, yv[c + 1], qmax, zero);
    }
  });
  step_fold<W>(head, qmax, zero, red);
}

template <class P, int C>
hipError_t launch_tile_shape(bool small, const tile_inst &I, int r, hipStream_t stream)
{
  constexpr int W = kTileWaves;
  const dim3 g(I.ntiles), b(64 * W);
  if (small)
    hipLaunchKernelGGL((k_tile<P, C, W, true>), g, b, 0, stream, I.ref.ring, I.ref.meth, I.y0,
                       I.y1, r, I.ntiles, I.N, I.nbands, I.nstrips, I.coef, I.ref.st, I.ref.view);
  else
    hipLaunchKernelGGL((k_tile<P, C, W, false>), g, b, 0, stream, I.ref.ring, I.ref.meth, I.y0,
                       I.y1, r, I.ntiles, I.N, I.nbands, I.nstrips, I.coef, I.ref.st, I.ref.view);
  return hipGetLastError();
}

template <class P>
hipError_t launch_tile_pat(int shape, bool small, const tile_inst &I, int r, hipStream_t stream)
{
  static_assert(kNumTileShapes == 4, "one case per shape");
  switch (shape) {
  case 0: return launch_tile_shape<P, kTileRows[0]>(small, I, r, stream);
  case 1: return launch_tile_shape<P, kTileRows[1]>(small, I, r, stream);
  case 2: return launch_tile_shape<P, kTileRows[2]>(small, I, r, stream);
  case 3: return launch_tile_shape<P, kTileRows[3]>(small, I, r, stream);
  default: return hipErrorInvalidConfiguration;
  }
}

}  // namespace
}  // namespace rkx
