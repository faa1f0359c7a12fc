// The stage-fused BRUSS2D step (rkx_sweep_kernel.hpp) for VERNER65, in a
// translation unit of its own, so that its build overlaps the other tables'.
#include "rkx_sweep_kernel.hpp"

namespace rkx {

hipError_t launch_sweep_verner65(int K, bool gen, const fused_launch<sweep_inst> &a,
                                hipStream_t stream)
{
  if (a.ntiles <= 0)
    return hipSuccess;
  return launch_pat<pat_verner65>(K, gen, a, stream);
}

int resident_blocks_verner65(int K) { return blocks_per_cu_k<pat_verner65>(K); }

}  // namespace rkx
