// Host side of the stage-fused BRUSS2D step (rkx_sweep_kernel.hpp): tile
// geometry and defaults, and the launches of the kernels of the tables with
// a compiled zero pattern (VERNER65's and DOPRI87's are built in
// rkx_kernels_sweep_verner65.hip and rkx_kernels_sweep_dopri87.hip).
#include "rkx_sweep_kernel.hpp"

#include <algorithm>

namespace rkx {

namespace {

int query_resident_blocks(int pattern, int K)
{
  switch (pattern) {
  case 1: return blocks_per_cu_k<pat_dopri54>(K);
  case 2: return resident_blocks_verner65(K);
  case 3: return blocks_per_cu_k<pat_rkf23>(K);
  case 4: return blocks_per_cu_k<pat_heun2>(K);
  case 5: return blocks_per_cu_k<pat_rk4>(K);
  case 6: return blocks_per_cu_k<pat_ssprk3>(K);
  case 7: return resident_blocks_dopri87(K);
  default: return 0;
  }
}

// A property of the built kernels, asked of the runtime once each (a solve's
// default tile would otherwise ask for every strip width).
int resident_blocks(int pattern, int K)
{
  constexpr int kPat = 8, kWidth = 5;
  static std::atomic<int> known[kPat][kWidth];   // 1 + the answer; 0: not asked yet
  if (pattern < 0 || pattern >= kPat || K < 0 || K >= kWidth)
    return 0;
  int v = known[pattern][K].load(std::memory_order_relaxed);
  if (v == 0) {
    v = 1 + query_resident_blocks(pattern, K);
    known[pattern][K].store(v, std::memory_order_relaxed);
  }
  return v - 1;
}

}  // namespace

bool sweep_supported(const dev_ode &p, const rkx_method &m)
{
  return p.kind == RKX_BRUSS2D && p.N >= 2 && pattern_of(m) != 0;
}

namespace {

// Strips of an N-column grid for strips of 64K lanes: as many full-width
// strips (64K - 2s output columns) as fit, and the columns left over either
// in a narrow strip of 32K lanes whose bands are paired two to a workgroup
// (K even, and they fit its 32K - 2s output columns), or else in one more
// strip, the strips then evened out.
struct strip_geom {
  int nwide;      // full-width strips
  int oc;         // output columns per full-width strip
  int split;      // 1: a narrow last strip of paired bands
  // workgroups for nb bands per strip
  long long wgs(long long nb) const { return nwide * nb + split * ((nb + 1) / 2); }
};

strip_geom strips_of(int N, int s, int K)
{
  const int oc_max = 64 * K - 2 * s;
  const int oc_half = (K % 2 == 0) ? 32 * K - 2 * s : 0;
  const int nfull = N / oc_max;
  const int rem = N - nfull * oc_max;
  if (rem > 0 && rem <= oc_half)
    return strip_geom{nfull, oc_max, 1};
  const int nstrips = (N + oc_max - 1) / oc_max;
  return strip_geom{nstrips, (N + nstrips - 1) / nstrips, 0};
}

// Relative time of one step whose workgroups all run at once: the row
// iterations of a band (plus about 5 for the step's start and end) times what
// one costs at the waves per SIMD that per_cu workgroups of a compute unit
// come to.  Measured, DOPRI54: 0.53 us an iteration at one wave per SIMD, 0.70
// at two, whatever the strip width that makes them up, and in proportion
// beyond (FP64 issue).
double sweep_time(int K, int per_cu, long long iters)
{
  const int wps = (2 * K * per_cu + 3) / 4;
  return static_cast<double>(iters + 5) * (wps < 2 ? 0.76 : 0.5 * wps);
}

// Most bands per strip whose workgroups fit `slots`.
long long bands_for_slots(const strip_geom &g, long long slots)
{
  long long nb = static_cast<long long>(static_cast<double>(slots) / (g.nwide + 0.5 * g.split));
  while (nb > 1 && g.wgs(nb) > slots)
    --nb;
  return nb < 1 ? 1 : nb;
}

}  // namespace

namespace {

bool full_trips_of(int pattern)
{
  switch (pattern) {
  case 1: return pat_dopri54::full_trips;
  case 2: return pat_verner65::full_trips;
  case 3: return pat_rkf23::full_trips;
  case 4: return pat_heun2::full_trips;
  case 5: return pat_rk4::full_trips;
  case 6: return pat_ssprk3::full_trips;
  case 7: return pat_dopri87::full_trips;
  default: return false;
  }
}

}  // namespace

bool sweep_single_reflect(int pattern, int s, int N)
{
  return N > s + prefetch_rows(s) + 3 + (full_trips_of(pattern) ? s + 1 : 0);
}

bool sweep_inst_single_reflect(int pattern, int s, const sweep_inst &I)
{
  if (!sweep_single_reflect(pattern, s, I.N))
    return false;
  // the last paired band loads rows up to nbands*R + s - 1 + prefetch
  return !I.split ||
         static_cast<long long>(I.nbands) * I.R + s - 1 + prefetch_rows(s) <= 2LL * (I.N - 1);
}

int sweep_tile_iters(int pattern, int s, const sweep_inst &I, int t)
{
  if (t >= I.nwide * I.nbands)
    return I.R + 2 * (s - 1);                   // paired: the full band height
  const int band = t % I.nbands;
  const int rows = std::min(I.R, I.N - band * I.R);
  return sweep_band_rows(pattern, s, rows) + 2 * (s - 1);
}

int sweep_band_rows(int pattern, int s, int rows)
{
  if (!full_trips_of(pattern))
    return rows;
  return trip_iters(s, rows + 2 * (s - 1)) - 2 * (s - 1);
}

// Default tile: strips of 64*K columns (2K waves per workgroup) and the band
// height R for which all strips x bands tiles are resident at once (one
// dispatch round: a second, partial round would leave most CUs idle while it
// runs), with bands as tall as that allows (the s-1 halo rows a band
// recomputes are a smaller share of taller bands).  Every count of workgroups
// per CU up to the resident maximum is a candidate, and the one with the
// shortest modelled step (sweep_time) wins.  The model it replaces priced
// lanes x iterations, as if a wider strip's idle lanes lengthened the step:
// VERNER65 N=717 33.2 us per step with its choice and 22.6 with this one,
// DOPRI54 N=1000 29.4 / 27.0, DOPRI87 N=300 65.9 / 45.3.
// A grid so wide that one band per strip gives fewer tiles than CUs (N =
// 32767, K = 4: 136 strips) or more than fit at once (DOPRI87, N = 32767:
// 322 strips of 2 waves) instead takes shorter bands over several rounds
// when that shortens the step: a CU then works through its tiles in turn,
// ceil(tiles / CUs) x the row iterations of one.
sweep_cfg sweep_default_cfg(const dev_ode &p, const rkx_method &m)
{
  const int s = m.s;
  const int N = p.N;
  const int pat = pattern_of(m);
  const bool trips = full_trips_of(pat);
  int cus = 0, dev = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus < 1) {
    (void) hipGetLastError();
    cus = 256;
  }
  auto band_rows_for = [&](long long bands) {
    if (bands < 1)
      bands = 1;
    int rows = static_cast<int>((N + bands - 1) / bands);
    return sweep_band_rows(pat, s, rows < 4 ? 4 : rows);
  };
  sweep_cfg best{2, 4};
  double best_cost = 1e300;
  for (int K = 1; K <= 4; ++K) {
    const int oc = 64 * K - 2 * s;
    if (oc < 1)
      continue;
    const strip_geom g = strips_of(N, s, K);
    const int res = resident_blocks(pat, K);
    if (res < 1)
      continue;                                     // too wide for this table's kernel
    for (int per_cu = 1; per_cu <= res; ++per_cu) {
      const int rows = band_rows_for(bands_for_slots(g, static_cast<long long>(cus) * per_cu));
      long long iters = rows + 2 * (s - 1);
      if (trips)
        iters = trip_iters(s, static_cast<int>(iters));
      const long long tiles = g.wgs((N + rows - 1) / rows);
      const long long rounds = (tiles + cus * per_cu - 1) / (cus * per_cu);
      const int there = static_cast<int>(std::min<long long>(per_cu, (tiles + cus - 1) / cus));
      const double cost = static_cast<double>(rounds) * sweep_time(K, there, iters);
      if (cost <= best_cost) {                      // wider strips: less halo traffic
        best_cost = cost;
        best = sweep_cfg{K, rows};
      }
    }
  }
  // several rounds for grids too wide for one band per strip to fill the CUs
  const strip_geom g = strips_of(N, s, best.waves);
  auto round_time = [&](int rows) {
    const long long tiles = g.wgs((N + rows - 1) / rows);
    long long iters = rows + 2 * (s - 1);
    if (trips)
      iters = trip_iters(s, static_cast<int>(iters));
    return static_cast<double>((tiles + cus - 1) / cus) * static_cast<double>(iters + 4);
  };
  const long long tiles = g.wgs((N + best.rows - 1) / best.rows);
  if (tiles < cus || tiles > static_cast<long long>(cus) * resident_blocks(pat, best.waves)) {
    double best_time = round_time(best.rows);
    for (int k = 2; k <= 16; ++k) {
      const int rows = band_rows_for(bands_for_slots(g, static_cast<long long>(k) * cus));
      const double t = round_time(rows);
      if (t < best_time) {
        best_time = t;
        best.rows = rows;
      }
    }
  }
  return best;
}

// Geometry of one instance's tiles for strips of 64*K columns and bands of R rows.
sweep_inst make_sweep_inst(const dev_ode &p, const rkx_method &m, const sweep_cfg &c,
                           const step_refs &ref, double *y0, double *y1)
{
  sweep_inst I{};
  const strip_geom g = strips_of(p.N, m.s, c.waves);
  I.N = p.N;
  I.R = sweep_band_rows(pattern_of(m), m.s, c.rows);
  I.OC = g.oc;
  I.nwide = g.nwide;
  I.split = g.split;
  I.nstrips = g.nwide + g.split;
  I.nbands = (p.N + I.R - 1) / I.R;
  I.ntiles = static_cast<int>(g.wgs(I.nbands));
  I.coef = p.coef;
  I.y0 = y0;
  I.y1 = y1;
  I.ref = ref;
  return I;
}

int sweep_pattern(const rkx_method &m) { return pattern_of(m); }

int sweep_resident_blocks(int pattern, int K) { return resident_blocks(pattern, K); }

hipError_t launch_sweep(int pattern, int K, bool gen, const fused_launch<sweep_inst> &a,
                        hipStream_t stream)
{
  if (a.ntiles <= 0)
    return hipSuccess;
  switch (pattern) {
  case 1: return launch_pat<pat_dopri54>(K, gen, a, stream);
  case 2: return launch_sweep_verner65(K, gen, a, stream);
  case 3: return launch_pat<pat_rkf23>(K, gen, a, stream);
  case 4: return launch_pat<pat_heun2>(K, gen, a, stream);
  case 5: return launch_pat<pat_rk4>(K, gen, a, stream);
  case 6: return launch_pat<pat_ssprk3>(K, gen, a, stream);
  case 7: return launch_sweep_dopri87(K, gen, a, stream);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace rkx
