// Stage-fused step for independent Lotka-Volterra pairs (src/problems/lv.c:
// ode_eval_comp of component i reads only its own pair, access distance 1).
//
// One thread per pair (grid-stride over a bounded number of workgroups)
// keeps every stage accumulator of the scatter form of D in registers:
// w_1..w_{s-1}, dy and err of both components receive the same products in
// the same order as the D kernels (block-inline.h:253-320; no zero skipping,
// as in seq D), so the step equals D's bitwise.  It reads y once and writes
// y_new once into the other y buffer: 16 bytes in and 16 out per pair per
// step, the low-storage form (two vectors of n) of a problem whose stencil
// needs no halo.  The error max-norm is folded per workgroup; the next step's
// kernel runs the control (step_begin).
#include "rkx_device.hpp"

#include <algorithm>

namespace rkx {
namespace {

// 256 workgroups of 16 waves: each workgroup folds its error maximum into the
// step state with atomics on one word, which queue at the end of a step, so
// fewer and larger workgroups finish faster (4e6 pairs, DOPRI54: 41 us per
// step against 90 us with 2048 workgroups of 4 waves)
constexpr int kPBlock = 1024;
constexpr int kPMaxBlocks = 256;

// Tables of up to 8 stages: h times the table (by row: h A[i][l], then h b[i],
// h e[i]) is formed by every workgroup and moved to scalar registers.  The 182
// coefficients of 13 stages do not fit there; read from LDS for every pair
// they cost three times the step (1e6 pairs: 146 us against 49), so a small
// kernel before the step's (k_lv_prepare) runs the control and writes the
// products to memory, and the step reads them with scalar loads.
constexpr int kPInRegs = 8;

__global__ __launch_bounds__(256) void k_lv_prepare(step_refs R, int r, dev_coef *cf, int s)
{
  __shared__ step_lds head;
  const step_now sn = step_begin(R, r, 0, head);
  if (sn.done)
    return;
  premult_block(*R.meth, s, sn.h, *cf, static_cast<int>(threadIdx.x), 256);
}

// What comes from memory is asked for before the step's control is waited
// for: the raw coefficients (one to a thread) and the first pair, from both
// y buffers.  The arguments the first loads need are in front, where the
// hardware hands them over in registers.
template <int S>
__global__ __launch_bounds__(kPBlock) void
k_lv_step(step_ring *ring, const dev_method *meth, double *y0, double *y1, int r, int cells,
          const dev_coef *__restrict__ pre, state *st, host_view *view, dev_ode p)
{
  constexpr bool kRegs = S <= kPInRegs;
  __shared__ double red[kPBlock / 64];
  __shared__ step_lds head;
  __shared__ double cl[kRegs ? S * (S + 2) : 1];
  using cell2 = double __attribute__((ext_vector_type(2)));
  using gcell = __attribute__((address_space(1))) cell2;
  static_assert(!kRegs || S * (S + 2) <= kPBlock, "one coefficient to a thread");
  const int k = threadIdx.x;
  double raw = 0.0;
  if constexpr (kRegs) {
    const int ci = k / (S + 2), cj = k - ci * (S + 2);
    if (k < S * (S + 2))
      raw = cj < S ? meth->A[ci * RKX_MAX_STAGES + cj] : (cj == S ? meth->b[ci] : meth->e[ci]);
  }
  const int first = blockIdx.x * kPBlock + threadIdx.x;
  const int stride = gridDim.x * kPBlock;
  const int at = min(first, cells - 1);
  const cell2 ya = ((gcell *) y0)[at], yb = ((gcell *) y1)[at];
  step_now sn;
  double cs[kRegs ? S * (S + 2) : 1];
  if constexpr (kRegs) {
    sn = step_begin(step_refs{st, ring, meth, view}, r, static_cast<int>(blockIdx.x), head);
    if (sn.done)
      return;                     // uniform: every block of the grid returns
    if (k < S * (S + 2))
      cl[k] = sn.h * raw;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < S * (S + 2); ++q)
      cs[q] = wave_uniform(cl[q]);
  } else {
    // k_lv_prepare has left this step's loop variables in the next slot
    const int rn = (r + 1) & (kRing - 1);
    gslot *now = (gslot *) &ring->slot[rn];
    sn.cur = now->v.cur;
    if (now->v.done)
      return;
    if (k == 0)
      head.err = &ring->err[rn][blockIdx.x & (kErrLines - 1)].bits;
  }
  // coefficient l of row i: l < i h A[i][l], S h b[i], S + 1 h e[i]
  auto cf = [&](int i, int l) -> double {
    if constexpr (kRegs)
      return cs[i * (S + 2) + l];
    else
      return l < S ? pre->hA[i * RKX_MAX_STAGES + l] : (l == S ? pre->hb[i] : pre->he[i]);
  };
  gcell *y = (gcell *) (sn.cur ? y1 : y0);
  gcell *ynew = (gcell *) (sn.cur ? y0 : y1);
  double qmax = 0.0;
  unsigned int zero = 0u;
  cell2 Y = sn.cur ? yb : ya;
  for (int pair = first; pair < cells; pair += stride) {
    const cell2 next = y[min(pair + stride, cells - 1)];   // ahead of its turn
    double wx[S], wy[S];          // [l]: w_l for l = 1..S-1
    double fx, fy;
    lv_pair(p, Y.x, Y.y, fx, fy);
#pragma unroll
    for (int l = 1; l < S; ++l) {
      const double a = cf(l, 0);
      wx[l] = Y.x + a * fx;
      wy[l] = Y.y + a * fy;
    }
    double dx = cf(0, S) * fx, dyv = cf(0, S) * fy;
    double ex = cf(0, S + 1) * fx, ey = cf(0, S + 1) * fy;
#pragma unroll
    for (int i = 1; i < S; ++i) {
      lv_pair(p, wx[i], wy[i], fx, fy);
#pragma unroll
      for (int l = i + 1; l < S; ++l) {
        const double a = cf(l, i);
        wx[l] += a * fx;
        wy[l] += a * fy;
      }
      dx += cf(i, S) * fx;
      dyv += cf(i, S) * fy;
      ex += cf(i, S + 1) * fx;
      ey += cf(i, S + 1) * fy;
    }
    const cell2 yn = {Y.x + dx, Y.y + dyv};
    ynew[pair] = yn;
    err_term(ex, yn.x, Y.x, qmax, zero);
    err_term(ey, yn.y, Y.y, qmax, zero);
    Y = next;
  }
  step_fold<kPBlock / 64>(head, qmax, zero, red);
}

template <int S>
hipError_t launch_s(const dev_ode &p, const step_refs &R, dev_coef *cf, double *y0, double *y1,
                    int r, hipStream_t stream)
{
  const int grid = std::max(1, std::min((p.cells + kPBlock - 1) / kPBlock, kPMaxBlocks));
  if (S > kPInRegs)
    hipLaunchKernelGGL(k_lv_prepare, dim3(1), dim3(256), 0, stream, R, r, cf, S);
  hipLaunchKernelGGL((k_lv_step<S>), dim3(grid), dim3(kPBlock), 0, stream, R.ring, R.meth, y0, y1,
                     r, p.cells, cf, R.st, R.view, p);
  return hipGetLastError();
}

}  // namespace

bool pairs_supported(const dev_ode &p, const rkx_method &m)
{
  if (p.kind != RKX_LV)
    return false;
  switch (m.s) {
  case 2: case 3: case 4: case 7: case 8: case 13: return true;
  default: return false;
  }
}

hipError_t launch_lv_step(const dev_ode &p, int s, const step_refs &R, dev_coef *cf, double *y0,
                          double *y1, int r, hipStream_t stream)
{
  switch (s) {
  case 2: return launch_s<2>(p, R, cf, y0, y1, r, stream);
  case 3: return launch_s<3>(p, R, cf, y0, y1, r, stream);
  case 4: return launch_s<4>(p, R, cf, y0, y1, r, stream);
  case 7: return launch_s<7>(p, R, cf, y0, y1, r, stream);
  case 8: return launch_s<8>(p, R, cf, y0, y1, r, stream);
  case 13: return launch_s<13>(p, R, cf, y0, y1, r, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace rkx
