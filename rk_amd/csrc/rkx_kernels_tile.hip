// Host side of the tile form of the BRUSS2D step (rkx_tile_kernel.hpp): tile
// geometry, and the launches.
#include "rkx_tile_kernel.hpp"

namespace rkx {

namespace {

// Whether the grid's last row or column may lie anywhere in a tile.
bool tile_small(int shape, int N) { return N < 64 || N < kTileRows[shape] * kTileWaves; }

}  // namespace

tile_inst make_tile_inst(const dev_ode &p, const rkx_method &m, int shape, const step_refs &ref,
                         double *y0, double *y1)
{
  tile_inst I{};
  const int s = m.s, H = kTileRows[shape] * kTileWaves;
  I.N = p.N;
  I.nstrips = tile_pieces(p.N, 64, s);
  I.nbands = tile_pieces(p.N, H, s - 1);
  I.ntiles = I.nstrips * I.nbands;
  I.coef = p.coef;
  I.y0 = y0;
  I.y1 = y1;
  I.ref = ref;
  return I;
}

bool tile_supported(int pattern) { return pattern >= 1 && pattern <= 6; }

// The shape with the fewest rows per wave whose workgroups all run at once,
// one to a compute unit: a step then takes the time of one tile, which grows
// with its rows, and a second round would double it.  Grids beyond the
// tallest tile's one round belong to the row sweep, whose bands waste less
// on halos.  Measured, us per step, tile against the best of 28 sweep shapes:
// DOPRI54 N=48 8.6 / 10.1, N=128 8.3 / 10.2, N=301 10.1 / 11.0, N=512 12.2 /
// 15.6, N=650 15.4 / 17.0 (tallest tile in two rounds at N=717: 30.6 / 21.0);
// VERNER65 N=128 9.2 / 11.9, N=301 11.1 / 13.4, N=512 17.2 / 18.6, N=640 17.7
// / 21.5; RKF23 N=128 5.9 / 6.4, N=512 7.5 / 8.6.
int tile_default_shape(const dev_ode &p, const rkx_method &m)
{
  if (!tile_supported(sweep_pattern(m)))
    return -1;
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 1) {
    (void) hipGetLastError();
    cus = 256;
  }
  for (int k = 0; k < kNumTileShapes; ++k) {
    if (kTileRows[k] * kTileWaves <= 2 * (m.s - 1) && p.N > kTileRows[k] * kTileWaves)
      continue;                                  // no rows left between the halos
    if (make_tile_inst(p, m, k, {}, nullptr, nullptr).ntiles <= cus)
      return k;
  }
  return -1;
}

hipError_t launch_tile_step(int pattern, int shape, const tile_inst &I, int r, hipStream_t stream)
{
  const bool small = tile_small(shape, I.N);
  switch (pattern) {
  case 1: return launch_tile_pat<pat_dopri54>(shape, small, I, r, stream);
  case 2: return launch_tile_pat<pat_verner65>(shape, small, I, r, stream);
  case 3: return launch_tile_pat<pat_rkf23>(shape, small, I, r, stream);
  case 4: return launch_tile_pat<pat_heun2>(shape, small, I, r, stream);
  case 5: return launch_tile_pat<pat_rk4>(shape, small, I, r, stream);
  case 6: return launch_tile_pat<pat_ssprk3>(shape, small, I, r, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace rkx
