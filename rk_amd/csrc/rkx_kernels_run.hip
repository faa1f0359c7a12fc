// BRUSS2D grids of one workgroup, several attempted steps to a launch.
//
// On a grid of at most 32 x 32 a step through k_tile is nearly all overhead:
// the launch, the trip to memory for the control's state and y, and the
// error's way back through memory.  One workgroup can hold such a grid whole, so nothing of a
// step needs another workgroup: here it keeps y in registers, reduces the
// error in LDS, and every wave runs the step control for itself (the same
// values in all of them, one barrier), for up to `steps` attempts a launch.
//
// A wave holds two blocks of C rows side by side, 32 lanes each (lane =
// column), so 8 waves cover 16 C rows; the stages are k_tile's
// (rkx_tile_kernel.hpp) without halos.  Beyond 32 columns a wave would hold
// one block, and four rows a lane and more: N = 48 would take 6 rows, twice
// k_tile's chain of work, and gain nothing over its several tiles.
//
// Bound by issue on one compute unit (N = 32 DOPRI54: its VALUs are busy 68 %
// of the time) and the control's dependent chain.
// us per step, before (k_tile; DOPRI87 the row sweep) -> here: DOPRI54 N = 32
// 8.6 -> 5.9, N = 16 8.6 -> 4.6; VERNER65 N = 32 10.3 -> 6.8; DOPRI87 N = 32
// 47 -> 13.
#include "rkx_tile_kernel.hpp"

namespace rkx {
namespace {

constexpr int kRunWaves = 8;
constexpr int kRunLanes = 32;    // columns

template <class P, int C>
__global__ __launch_bounds__(64 * kRunWaves) void
k_tile_run(step_ring *ring, const dev_method *meth, double *y0, double *y1, int r, int steps,
           int N, double coef, state *st, host_view *view)
{
  constexpr int s = P::s, W = kRunWaves, B = 2 * W;
  __shared__ double2 edge[2][B][2][kRunLanes];   // first and last row of each block
  __shared__ double red[2][W];

  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int col = lane & (kRunLanes - 1), blk = 2 * wv + (lane >> 5);
  const int row = blk * C;
  const bool left = col == 0, right = col == N - 1;
  const tile_place T{N, row, left, right, left ? 2.0 : 1.0, right ? 2.0 : 1.0, coef};

  using cell2 = double __attribute__((ext_vector_type(2)));
  using gcell = __attribute__((address_space(1))) cell2;
  step_coefs<P> kc;
  kc.load(as_global(meth));
  unsigned at[C];
  bool in[C];
  cell2 ya[2][C];
  static_for<C>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    in[c] = row + c < N && col < N;
    at[c] = static_cast<unsigned>(min(row + c, N - 1)) * static_cast<unsigned>(N) +
            static_cast<unsigned>(min(col, N - 1));
    ya[0][c] = ((gcell *) y0)[at[c]];
    ya[1][c] = ((gcell *) y1)[at[c]];
  });
  // no attempt of an earlier launch is pending: each ends with its control
  gslot *sl = (gslot *) &ring->slot[r];
  step_vars v = slot_vars(sl);
  const int traced = sl->traced;
  step_slot &next = ring->slot[(r + 1) & (kRing - 1)];
  if (__builtin_amdgcn_readfirstlane(v.done)) {  // uniform
    if (threadIdx.x == 0)
      next.v = v;                                // a launch behind this one reads it
    return;
  }
  lane_pow_tables pw;
  pw.load();
  const int cur0 = __builtin_amdgcn_readfirstlane(v.cur);
  double yu[C + 2], yv[C + 2];                   // [0], [C + 1]: the rows beyond the block's
  static_for<C>([&](auto ct) {
    constexpr int c = decltype(ct)::value;
    yu[c + 1] = cur0 ? ya[1][c].x : ya[0][c].x;
    yv[c + 1] = cur0 ? ya[1][c].y : ya[0][c].y;
  });

  const int up = max(blk - 1, 0), dn = min(blk + 1, B - 1);
  bool moved = false;
  double err = 0.0;
  for (int a = 0;;) {
    kc.scale(wave_uniform(v.h));
    edge[0][blk][0][col] = make_double2(yu[1], yv[1]);
    edge[0][blk][1][col] = make_double2(yu[C], yv[C]);
    double au[C][s + 1], av[C][s + 1];
    static_for<s>([&](auto itg) {
      constexpr int i = decltype(itg)::value;
      __syncthreads();
      const double2 n = edge[i & 1][up][1][col], q = edge[i & 1][dn][0][col];
      if constexpr (i == 0) {
        yu[0] = n.x;
        yv[0] = n.y;
        yu[C + 1] = q.x;
        yv[C + 1] = q.y;
      }
      tile_stage<P, C, i, true, true>(T, kc.k[i], yu, yv, n.x, n.y, q.x, q.y, au, av);
      if constexpr (i + 1 < s) {
        edge[(i + 1) & 1][blk][0][col] = make_double2(au[0][i + 1], av[0][i + 1]);
        edge[(i + 1) & 1][blk][1][col] = make_double2(au[C - 1][i + 1], av[C - 1][i + 1]);
      }
    });
    double qmax = 0.0;
    unsigned int zero = 0u;
    double nu[C], nv[C];
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      nu[c] = yu[c + 1] + au[c][0];
      nv[c] = yv[c + 1] + av[c][0];
      if (in[c]) {
        err_term(au[c][s], nu[c], yu[c + 1], qmax, zero);
        err_term(av[c][s], nv[c], yv[c + 1], qmax, zero);
      }
    });
    kc.load(as_global(meth));                    // for the next attempt's h
    if (zero)
      qmax = fmax(qmax, 1.7E308);
    qmax = wave_max63(qmax);
    if (lane == 63)
      red[a & 1][wv] = qmax;
    __syncthreads();
    static_assert(W == 8, "half a row of lanes");
    err = red[a & 1][lane & (W - 1)];
    err = fmax(err, dpp_keep<0x111>(err));
    err = fmax(err, dpp_keep<0x112>(err));
    err = fmax(err, dpp_keep<0x114>(err));       // lane 7: all eight
    err = __builtin_bit_cast(
        double, lane_pow_tables::lane_of(__builtin_bit_cast(unsigned long long, err), 7));
    if (traced && threadIdx.x == 0)
      trace_attempt(st, v, err);
    const int cur = v.cur;
    double px = 0.0, py = 0.0;
    const bool need = ctrl_decide(v, err, px, py);
    ctrl_finish(v, need, need ? libm_pow(px, py, pw) : 0.0);
    if (__builtin_amdgcn_readfirstlane(v.cur) != __builtin_amdgcn_readfirstlane(cur)) {
      moved = true;
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        yu[c + 1] = nu[c];
        yv[c + 1] = nv[c];
      });
    }
    if (__builtin_amdgcn_readfirstlane(v.done) || ++a == steps)
      break;
  }

  // y into the buffer that the loop's state names
  if (moved) {
    gcell *o = (gcell *) (__builtin_amdgcn_readfirstlane(v.cur) ? y1 : y0);
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      if (in[c])
        o[at[c]] = cell2{yu[c + 1], yv[c + 1]};
    });
  }
  if (threadIdx.x == 0) {
    next.v = v;
    next.pending = 0;
    next.traced = traced;
    publish(st, v, err);
    if (view)
      show(view, v);
  }
}

template <class P>
hipError_t launch_run_pat(const tile_inst &I, int r, int steps, hipStream_t stream)
{
  const dim3 g(1), b(64 * kRunWaves);
  if (I.N <= 2 * kRunWaves)
    hipLaunchKernelGGL((k_tile_run<P, 1>), g, b, 0, stream, I.ref.ring, I.ref.meth, I.y0, I.y1, r,
                       steps, I.N, I.coef, I.ref.st, I.ref.view);
  else
    hipLaunchKernelGGL((k_tile_run<P, 2>), g, b, 0, stream, I.ref.ring, I.ref.meth, I.y0, I.y1, r,
                       steps, I.N, I.coef, I.ref.st, I.ref.view);
  return hipGetLastError();
}

}  // namespace

// 2 blocks a wave of 2 rows of 32 columns
bool run_supported(int pattern, int N)
{
  return pattern >= 1 && pattern <= 7 && N <= kRunLanes && N <= 4 * kRunWaves;
}

hipError_t launch_run(int pattern, const tile_inst &I, int r, int steps, hipStream_t stream)
{
  switch (pattern) {
  case 1: return launch_run_pat<pat_dopri54>(I, r, steps, stream);
  case 2: return launch_run_pat<pat_verner65>(I, r, steps, stream);
  case 3: return launch_run_pat<pat_rkf23>(I, r, steps, stream);
  case 4: return launch_run_pat<pat_heun2>(I, r, steps, stream);
  case 5: return launch_run_pat<pat_rk4>(I, r, steps, stream);
  case 6: return launch_run_pat<pat_ssprk3>(I, r, steps, stream);
  case 7: return launch_run_pat<pat_dopri87>(I, r, steps, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace rkx
