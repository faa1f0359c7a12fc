// The control of the fused kernels' last attempt, run on its own: after the
// last launch of a chunk the attempt it made still awaits its control (every
// fused kernel starts with the control of the attempt before it).  Instances
// that have ended are left alone.
#include "rkx_device.hpp"

namespace rkx {
namespace {

constexpr int kFlushBlock = 64;

__global__ __launch_bounds__(kFlushBlock) void k_step_flush(state *st, int n, int r)
{
  const int i = blockIdx.x * kFlushBlock + threadIdx.x;
  // an instance that has ended is launched no more, and its older ring slots
  // keep attempts whose control has long run: nothing is pending
  if (i >= n || !st[i].ring || st[i].v.done)
    return;
  step_ring &g = *st[i].ring;
  step_slot s = g.slot[r];
  if (s.pending) {
    const double err = ring_err(g.err[r]);
    trace_attempt(st + i, s.v, err);
    double px = 0.0, py = 0.0;
    const bool need = ctrl_decide(s.v, err, px, py);
    ctrl_finish(s.v, need, need ? libm_pow(px, py, dev_pow_tables) : 0.0);
    publish(st + i, s.v, err);
    s.pending = 0;
  }
  g.slot[0] = s;
  for (int k = 0; k < kRing * kErrLines; ++k)
    g.err[k / kErrLines][k % kErrLines].bits = 0ull;
}

}  // namespace

hipError_t launch_step_flush(state *st, int n, int r, hipStream_t stream)
{
  hipLaunchKernelGGL(k_step_flush, dim3((n + kFlushBlock - 1) / kFlushBlock), dim3(kFlushBlock), 0,
                     stream, st, n, r);
  return hipGetLastError();
}

}  // namespace rkx
