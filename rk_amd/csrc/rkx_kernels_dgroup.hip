// The D form of the BRUSS2D step, several stages to a kernel.
//
// Seq D (src/impl/seq/D.c:58-78) runs its stages one after another over full
// vectors: stage i reads w_i and adds h*A[l][i]*F to every later w_l, dy and
// err (block-inline.h:253-320).  One kernel per stage moves 69 vectors a
// DOPRI54 step (1.1 GB at N = 1000: 204 us, the memory's rate).  Here a kernel
// takes a group of up to four stages i0 .. i0+G-1 over a tile: the w of the
// group's own later stages are read with a halo and completed in registers,
// and each w_l behind the group is read and written once, receiving the G
// terms in D's order (zero coefficients are not skipped, as in D, so every
// sum equals D's bitwise).  DOPRI54 then moves 13 vectors a step in two
// kernels.  Storage is D's: y (2 buffers), w_1..w_{s-1}, dy, err.
//
// The tile is the one of rkx_tile_kernel.hpp: 64 columns (lane = column) x
// 8 waves of C rows, u and v in one lane, horizontal neighbours by DPP,
// vertical ones across waves through LDS; it yields 64 - 2G columns and
// 8C - 2(G-1) rows.  Every kernel of the step starts with the control of the
// attempt before it; the last one folds the error.
#include "rkx_tile_kernel.hpp"

#include <algorithm>

namespace rkx {
namespace {

constexpr int kGroupRows = 4;                    // rows per wave

template <int G, bool FIRST, bool LAST, bool SMALL>
__global__ __launch_bounds__(64 * kTileWaves) void k_d_group(stage_group a)
{
  constexpr int C = kGroupRows, W = kTileWaves, H = W * C;
  __shared__ double2 edge[2][W][2][64];
  __shared__ double red[W];
  __shared__ double cl[G][RKX_MAX_STAGES + 2];   // h A[l][i0+g] (l < s), h b, h e
  __shared__ step_lds head;

  const int s = a.s, i0 = a.i0, N = a.N;
  // only the step's last kernel writes the next slot
  const step_now sn = step_begin(a.ref, a.r, LAST ? static_cast<int>(blockIdx.x) : 1, head);
  if (sn.done)
    return;
  for (int k = threadIdx.x; k < G * (s + 2); k += 64 * W) {
    const int g = k / (s + 2), l = k - g * (s + 2);
    const dev_method *m = a.ref.meth;
    const double c = l < s ? m->A[l * RKX_MAX_STAGES + i0 + g]
                           : (l == s ? m->b[i0 + g] : m->e[i0 + g]);
    cl[g][l] = sn.h * c;
  }
  using cell2 = double __attribute__((ext_vector_type(2)));
  using gcell = __attribute__((address_space(1))) cell2;
  const size_t cells = static_cast<size_t>(N) * N;
  gcell *y = (gcell *) (sn.cur ? a.y1 : a.y0);
  gcell *yn = (gcell *) (sn.cur ? a.y0 : a.y1);
  gcell *w = (gcell *) a.w;                      // w_l at (l - 1) * cells
  gcell *dy = (gcell *) a.dy, *er = (gcell *) a.err;

  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int SC = 64 - 2 * G, SR = H - 2 * (G - 1);
  double qmax = 0.0;
  unsigned int zero = 0u;
  // a bounded number of workgroups, each over several tiles: the table's
  // coefficients and the control are formed once per workgroup
  for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
    __syncthreads();                             // cl; the tile before is done with edge
    const int strip = t / a.nbands, band = t - strip * a.nbands;
    const int tc = SMALL ? 0 : min(strip * SC, N - 64);
    const int c0 = strip == 0 ? 0 : strip * SC + G;
    const int c1 = strip == a.nstrips - 1 ? N : strip * SC + 64 - G;
    const int tr = N < H ? 0 : min(band * SR, N - H);
    const int r0 = band == 0 ? 0 : band * SR + (G - 1);
    const int r1 = band == a.nbands - 1 ? N : band * SR + H - (G - 1);
    const int col = tc + lane;
    const int row = tr + wv * C;
    const bool left = col == 0, right = col == N - 1;
    const double mE = left ? 2.0 : 1.0, mW = right ? 2.0 : 1.0;
    const int ccol = SMALL ? min(col, N - 1) : col;
    auto at = [&](int k) -> unsigned {
      return static_cast<unsigned>(max(0, min(k, N - 1))) * static_cast<unsigned>(N) +
             static_cast<unsigned>(ccol);
    };

    // [0]: the group's first vector (y or w_i0) with the row on either side
    cell2 v0[C + 2];
    cell2 wg[G][C];                              // [g >= 1]: w_{i0+g}
    cell2 F[G][C];
    gcell *src = FIRST ? y : w + (i0 - 1) * cells;
    static_for<C + 2>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      v0[c] = src[at(row + c - 1)];
    });
    static_for<G>([&](auto gt) {
      constexpr int g = decltype(gt)::value;
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        F[g][c] = cell2{0.0, 0.0};
        if constexpr (g == 0 || FIRST)
          wg[g][c] = v0[c + 1];
        else
          wg[g][c] = (w + (i0 + g - 1) * cells)[at(row + c)];
      });
    });

    static_for<G>([&](auto gt) {
      constexpr int g = decltype(gt)::value;
      const bool need = row + C > r0 - (G - 1 - g) && row < r1 + (G - 1 - g);
      cell2 north = v0[0], south = v0[C + 1];
      if constexpr (g > 0) {
        __syncthreads();
        const double2 up = edge[g & 1][max(wv - 1, 0)][1][lane];
        const double2 dn = edge[g & 1][min(wv + 1, W - 1)][0][lane];
        north = cell2{up.x, up.y};
        south = cell2{dn.x, dn.y};
      }
      if (!need)
        return;
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        const cell2 m = wg[g][c];
        cell2 n, sth;
        if constexpr (c == 0)
          n = north;
        else
          n = wg[g][c - 1];
        if constexpr (c == C - 1)
          sth = south;
        else
          sth = wg[g][c + 1];
        if constexpr (SMALL || c == 0) {
          const bool top = row + c == 0;
          n.x = top ? sth.x : n.x;
          n.y = top ? sth.y : n.y;
        }
        if constexpr (SMALL || c == C - 1) {
          const bool bot = row + c == N - 1;
          sth.x = bot ? n.x : sth.x;
          sth.y = bot ? n.y : sth.y;
        }
        double uE = from_right(m.x), vE = from_right(m.y);
        if constexpr (SMALL) {
          uE = right ? 0.0 : uE;
          vE = right ? 0.0 : vE;
        }
        const double lu = __builtin_fma(
            -4.0, m.x, __builtin_fma(mE, uE, __builtin_fma(mW, from_left(m.x), n.x + sth.x)));
        const double lv = __builtin_fma(
            -4.0, m.y, __builtin_fma(mE, vE, __builtin_fma(mW, from_left(m.y), n.y + sth.y)));
        double fu, fv;
        bruss_react(m.x, m.y, lu, lv, a.coef, fu, fv);
        F[g][c] = cell2{fu, fv};
      });
      static_for<G>([&](auto jt) {
        constexpr int j = decltype(jt)::value;
        if constexpr (j > g) {
          const double k = cl[g][i0 + j];
          static_for<C>([&](auto ct) {
            constexpr int c = decltype(ct)::value;
            wg[j][c].x += k * F[g][c].x;
            wg[j][c].y += k * F[g][c].y;
          });
        }
      });
      if constexpr (g + 1 < G) {
        edge[(g + 1) & 1][wv][0][lane] = make_double2(wg[g + 1][0].x, wg[g + 1][0].y);
        edge[(g + 1) & 1][wv][1][lane] = make_double2(wg[g + 1][C - 1].x, wg[g + 1][C - 1].y);
      }
    });

    // the vectors behind the group, dy and err (LAST: y_new and the error
    // term), each a pass over the wave's own rows
    const bool cin = col >= c0 && col < c1;
    bool in[C];
    unsigned pos[C];
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      in[c] = cin && row + c >= r0 && row + c < r1;
      pos[c] = at(row + c);
    });
    if constexpr (!LAST) {
      for (int l = i0 + G; l < s; ++l) {
        gcell *wl = w + (l - 1) * cells;
        double k[G];
        static_for<G>([&](auto gt) { k[decltype(gt)::value] = cl[decltype(gt)::value][l]; });
        cell2 o[C];
        static_for<C>([&](auto ct) {
          constexpr int c = decltype(ct)::value;
          if constexpr (FIRST)
            o[c] = v0[c + 1];
          else
            o[c] = in[c] ? wl[pos[c]] : cell2{0.0, 0.0};
        });
        static_for<C>([&](auto ct) {
          constexpr int c = decltype(ct)::value;
          static_for<G>([&](auto gt) {
            constexpr int g = decltype(gt)::value;
            o[c].x += k[g] * F[g][c].x;
            o[c].y += k[g] * F[g][c].y;
          });
          if (in[c])
            wl[pos[c]] = o[c];
        });
      }
    }
    double kb[G], ke[G];
    static_for<G>([&](auto gt) {
      constexpr int g = decltype(gt)::value;
      kb[g] = cl[g][s];
      ke[g] = cl[g][s + 1];
    });
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      if (in[c]) {
        cell2 d, e;
        if constexpr (!FIRST) {
          d = dy[pos[c]];
          e = er[pos[c]];
        }
        static_for<G>([&](auto gt) {
          constexpr int g = decltype(gt)::value;
          if constexpr (FIRST && g == 0) {
            d = cell2{kb[0] * F[0][c].x, kb[0] * F[0][c].y};
            e = cell2{ke[0] * F[0][c].x, ke[0] * F[0][c].y};
          } else {
            d.x += kb[g] * F[g][c].x;
            d.y += kb[g] * F[g][c].y;
            e.x += ke[g] * F[g][c].x;
            e.y += ke[g] * F[g][c].y;
          }
        });
        if constexpr (LAST) {
          const cell2 yo = FIRST ? v0[c + 1] : y[pos[c]];
          const cell2 o = {yo.x + d.x, yo.y + d.y};
          yn[pos[c]] = o;
          err_term(e.x, o.x, yo.x, qmax, zero);
          err_term(e.y, o.y, yo.y, qmax, zero);
        } else {
          dy[pos[c]] = d;
          er[pos[c]] = e;
        }
      }
    });
  }
  if constexpr (LAST)
    step_fold<W>(head, qmax, zero, red);
}

template <int G, bool FIRST, bool LAST>
hipError_t launch_group(const stage_group &a, int grid, hipStream_t stream)
{
  if (a.N < 64 || a.N < kTileWaves * kGroupRows)
    hipLaunchKernelGGL((k_d_group<G, FIRST, LAST, true>), dim3(grid), dim3(64 * kTileWaves), 0,
                       stream, a);
  else
    hipLaunchKernelGGL((k_d_group<G, FIRST, LAST, false>), dim3(grid), dim3(64 * kTileWaves), 0,
                       stream, a);
  return hipGetLastError();
}

template <int G>
hipError_t launch_group(bool first, bool last, const stage_group &a, int grid, hipStream_t stream)
{
  if (first)
    return last ? launch_group<G, true, true>(a, grid, stream)
                : launch_group<G, true, false>(a, grid, stream);
  return last ? launch_group<G, false, true>(a, grid, stream)
              : launch_group<G, false, false>(a, grid, stream);
}

}  // namespace

hipError_t launch_d_groups(stage_group a, hipStream_t stream)
{
  // as few groups of up to four stages as there must be, of even sizes
  const int groups = (a.s + 3) / 4;
  const int H = kTileWaves * kGroupRows;
  for (int q = 0; q < groups; ++q) {
    const int i0 = q * a.s / groups, G = (q + 1) * a.s / groups - i0;
    a.i0 = i0;
    a.nstrips = tile_pieces(a.N, 64, G);
    a.nbands = tile_pieces(a.N, H, G - 1);
    a.ntiles = a.nstrips * a.nbands;
    const int grid = std::min(a.ntiles, kGroupBlocks);
    hipError_t e = hipErrorInvalidValue;
    switch (G) {
    case 2: e = launch_group<2>(q == 0, q == groups - 1, a, grid, stream); break;
    case 3: e = launch_group<3>(q == 0, q == groups - 1, a, grid, stream); break;
    case 4: e = launch_group<4>(q == 0, q == groups - 1, a, grid, stream); break;
    default: break;
    }
    if (e != hipSuccess)
      return e;
  }
  return hipSuccess;
}

}  // namespace rkx
