// The full-storage loop orders of a BRUSS2D step, several stages to a kernel.
//
// Seq D (src/impl/seq/D.c:58-78) runs its stages one after another over full
// vectors: stage i reads w_i and adds h*A[l][i]*F to every later w_l, dy and
// err (block-inline.h:253-320).  One kernel per stage moves 69 vectors a
// DOPRI54 step (1.1 GB at N = 1000: 204 us, the memory's rate); the gather
// orders A, E and F (src/impl/seq/A.c, E.c, F.c), which form each w_l from the
// stage derivatives v_i, move 49 to 56.  Here a kernel takes a group of up to
// four stages i0 .. i0+G-1 over a tile and completes the w of the group in
// registers:
//
//   D         the w of the group's own later stages are read with a halo, and
//             each w_l behind the group is read and written once, receiving
//             the G terms: 15 vectors a DOPRI54 step in two kernels;
//   A, E, F   y and v_0 .. v_{i0-1} are read with a halo and gathered into the
//             group's w, and the group's v are written; the step's last kernel
//             also gathers dy and err, and writes y_new: 9 vectors.
//
// Every sum receives its terms in the reference's order, in A without those
// of zero coefficients (of the table), in D, E and F with them, so each equals
// the one-stage kernels' bitwise.  Storage is the form's own (the w of A, E and
// F stays unused here).  N = 1000, per step, one stage a kernel -> groups:
// DOPRI54 D 211 -> 51 us, A 201 -> 52, E 205 -> 50, F 165 -> 50; DOPRI87
// D 555 -> 179, A 404 -> 132, E 451 -> 130, F 379 -> 130.
//
// The tile is the one of rkx_tile_kernel.hpp: 64 columns (lane = column) x
// 8 waves of C = 2 or 4 rows, u and v in one lane, horizontal neighbours by DPP,
// vertical ones across waves through LDS; it yields 64 - 2G columns and
// 8C - 2(G-1) rows.  Every kernel of the step starts with the control of the
// attempt before it; the last one folds the error.
//
// Bound by memory: N = 1000 DOPRI54, D 240 MB a step at 4.6 TB/s; the VALUs are
// busy 25 to 34 % of the time.
#include "rkx_tile_kernel.hpp"

#include <algorithm>

namespace rkx {
namespace {

// rows per wave: the fewer that still let all tiles of a kernel run at once
// (halo rows are cheaper then than a second row's time in every wave), else 4.
// us per step, 2 / 4 rows: DOPRI54 D N = 200 15.4 / 18.4, N = 500 25.7 / 27.6,
// N = 700 36.9 / 34.0, N = 1000 59.5 / 51.9.
constexpr int kGroupRows[] = {2, 4};

using cell2 = double __attribute__((ext_vector_type(2)));
using gcell = __attribute__((address_space(1))) cell2;

// What a workgroup keeps in LDS: the waves' edge rows, and the step's products
// h A[l][i0+g] (l < s), h b, h e of the group's stages (D), or h A[i0+g][j],
// and h b, h e of all stages (gather).
struct group_lds {
  double2 edge[2][kTileWaves][2][64];
  double red[kTileWaves];
  step_lds head;
};

// One tile: where it lies, and the group's stages over it.
template <int G, int C, bool SMALL>
struct group_tile {
  static constexpr int W = kTileWaves, H = W * C;
  int N, lane, wv;
  int c0, c1, r0, r1;          // columns and rows of y_new
  int col, row;                // the lane's column, the wave's first row
  int ccol;                    // in-bounds column
  double mE, mW;

  __device__ __forceinline__ group_tile(const stage_group &a, int t)
  {
    constexpr int SC = 64 - 2 * G, SR = H - 2 * (G - 1);
    N = a.N;
    lane = threadIdx.x & 63;
    wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int strip = t / a.nbands, band = t - strip * a.nbands;
    const int tc = SMALL ? 0 : min(strip * SC, N - 64);
    c0 = strip == 0 ? 0 : strip * SC + G;
    c1 = strip == a.nstrips - 1 ? N : strip * SC + 64 - G;
    const int tr = N < H ? 0 : min(band * SR, N - H);
    r0 = band == 0 ? 0 : band * SR + (G - 1);
    r1 = band == a.nbands - 1 ? N : band * SR + H - (G - 1);
    col = tc + lane;
    row = tr + wv * C;
    ccol = SMALL ? min(col, N - 1) : col;
    mE = col == 0 ? 2.0 : 1.0;
    mW = col == N - 1 ? 2.0 : 1.0;
  }
  // position of row k in the lane's column (rows clamped into the grid)
  __device__ __forceinline__ unsigned at(int k) const
  {
    return static_cast<unsigned>(max(0, min(k, N - 1))) * static_cast<unsigned>(N) +
           static_cast<unsigned>(ccol);
  }
  // F[g] of the group's stages from wg[g] (w_{i0+g} without the group's own
  // terms) and the rows beyond the wave's of w_i0.  coef(j, g): the product
  // with which stage g enters wg[j], or 0 with use(j, g) false.
  template <class COEF, class USE>
  __device__ __forceinline__ void stages(group_lds &x, double rcoef, cell2 first_n, cell2 first_s,
                                         cell2 (&wg)[G][C], cell2 (&F)[G][C], COEF &&coef,
                                         USE &&use) const
  {
    const bool right = col == N - 1;
    static_for<G>([&](auto gt) {
      constexpr int g = decltype(gt)::value;
      const bool need = row + C > r0 - (G - 1 - g) && row < r1 + (G - 1 - g);
      cell2 north = first_n, south = first_s;
      if constexpr (g > 0) {
        __syncthreads();
        const double2 up = x.edge[g & 1][max(wv - 1, 0)][1][lane];
        const double2 dn = x.edge[g & 1][min(wv + 1, W - 1)][0][lane];
        north = cell2{up.x, up.y};
        south = cell2{dn.x, dn.y};
      }
      if (!need)
        return;
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        const cell2 m = wg[g][c];
        cell2 n = north, sth = south;
        if constexpr (c > 0)
          n = wg[g][c - 1];
        if constexpr (c < C - 1)
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
        bruss_react(m.x, m.y, lu, lv, rcoef, fu, fv);
        F[g][c] = cell2{fu, fv};
      });
      static_for<G>([&](auto jt) {
        constexpr int j = decltype(jt)::value;
        if constexpr (j > g) {
          if (use(j, g)) {
            const double k = coef(j, g);
            static_for<C>([&](auto ct) {
              constexpr int c = decltype(ct)::value;
              wg[j][c].x += k * F[g][c].x;
              wg[j][c].y += k * F[g][c].y;
            });
          }
        }
      });
      if constexpr (g + 1 < G) {
        x.edge[(g + 1) & 1][wv][0][lane] = make_double2(wg[g + 1][0].x, wg[g + 1][0].y);
        x.edge[(g + 1) & 1][wv][1][lane] = make_double2(wg[g + 1][C - 1].x, wg[g + 1][C - 1].y);
      }
    });
  }
};

template <int G, int C, bool FIRST, bool LAST, bool SMALL>
__global__ __launch_bounds__(64 * kTileWaves) void k_d_group(stage_group a)
{
  constexpr int W = kTileWaves;
  __shared__ group_lds x;
  __shared__ double cl[G][RKX_MAX_STAGES + 2];   // h A[l][i0+g] (l < s), h b, h e

  const int s = a.s, i0 = a.i0;
  // only the step's last kernel writes the next slot
  const step_now sn = step_begin(a.ref, a.r, LAST ? static_cast<int>(blockIdx.x) : 1, x.head);
  if (sn.done)
    return;
  for (int k = threadIdx.x; k < G * (s + 2); k += 64 * W) {
    const int g = k / (s + 2), l = k - g * (s + 2);
    const dev_method *m = a.ref.meth;
    const double c = l < s ? m->A[l * RKX_MAX_STAGES + i0 + g]
                           : (l == s ? m->b[i0 + g] : m->e[i0 + g]);
    cl[g][l] = sn.h * c;
  }
  const size_t cells = static_cast<size_t>(a.N) * a.N;
  gcell *y = (gcell *) (sn.cur ? a.y1 : a.y0);
  gcell *yn = (gcell *) (sn.cur ? a.y0 : a.y1);
  gcell *w = (gcell *) a.w;                      // w_l at (l - 1) * cells
  gcell *dy = (gcell *) a.dy, *er = (gcell *) a.err;

  double qmax = 0.0;
  unsigned int zero = 0u;
  // a bounded number of workgroups, each over several tiles: the table's
  // coefficients and the control are formed once per workgroup
  for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
    __syncthreads();                             // cl; the tile before is done with edge
    const group_tile<G, C, SMALL> T(a, t);
    // the group's first vector (y or w_i0) with the row on either side
    cell2 v0[C + 2];
    cell2 wg[G][C];                              // [g >= 1]: w_{i0+g}
    cell2 F[G][C];
    gcell *src = FIRST ? y : w + (i0 - 1) * cells;
    static_for<C + 2>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      v0[c] = src[T.at(T.row + c - 1)];
    });
    static_for<G>([&](auto gt) {
      constexpr int g = decltype(gt)::value;
      static_for<C>([&](auto ct) {
        constexpr int c = decltype(ct)::value;
        F[g][c] = cell2{0.0, 0.0};
        if constexpr (g == 0 || FIRST)
          wg[g][c] = v0[c + 1];
        else
          wg[g][c] = (w + (i0 + g - 1) * cells)[T.at(T.row + c)];
      });
    });
    T.stages(x, a.coef, v0[0], v0[C + 1], wg, F,
             [&](int j, int g) { return cl[g][i0 + j]; }, [](int, int) { return true; });

    // the vectors behind the group, dy and err (LAST: y_new and the error
    // term), each a pass over the wave's own rows
    const bool cin = T.col >= T.c0 && T.col < T.c1;
    bool in[C];
    unsigned pos[C];
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      in[c] = cin && T.row + c >= T.r0 && T.row + c < T.r1;
      pos[c] = T.at(T.row + c);
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
    step_fold<W>(x.head, qmax, zero, x.red);
}

// A (SKIP), E and F.  nz: the masks of the table's non-zero entries.
template <int G, int C, bool FIRST, bool LAST, bool SMALL, bool SKIP>
__global__ __launch_bounds__(64 * kTileWaves) void k_g_group(stage_group a, gather_masks nz)
{
  constexpr int W = kTileWaves;
  __shared__ group_lds x;
  __shared__ double cl[G][RKX_MAX_STAGES];       // h A[i0+g][j]
  __shared__ double cb[RKX_MAX_STAGES], ce[RKX_MAX_STAGES];

  const int s = a.s, i0 = a.i0;
  const step_now sn = step_begin(a.ref, a.r, LAST ? static_cast<int>(blockIdx.x) : 1, x.head);
  if (sn.done)
    return;
  {
    const dev_method *m = a.ref.meth;
    for (int k = threadIdx.x; k < G * s; k += 64 * W)
      cl[k / s][k % s] = sn.h * m->A[(i0 + k / s) * RKX_MAX_STAGES + k % s];
    if (static_cast<int>(threadIdx.x) < s) {
      cb[threadIdx.x] = sn.h * m->b[threadIdx.x];
      ce[threadIdx.x] = sn.h * m->e[threadIdx.x];
    }
  }
  unsigned row_nz[G];
  static_for<G>([&](auto gt) {
    row_nz[decltype(gt)::value] = SKIP ? nz.rowA[i0 + decltype(gt)::value] : ~0u;
  });
  // the first term of dy and err is a product whatever its weight is
  const unsigned nzb = SKIP ? nz.b | 1u : ~0u, nze = SKIP ? nz.e | 1u : ~0u;
  const size_t cells = static_cast<size_t>(a.N) * a.N;
  gcell *y = (gcell *) (sn.cur ? a.y1 : a.y0);
  gcell *yn = (gcell *) (sn.cur ? a.y0 : a.y1);
  gcell *v = (gcell *) a.w;                      // v_i at i * cells

  double qmax = 0.0;
  unsigned int zero = 0u;
  for (int t = blockIdx.x; t < a.ntiles; t += gridDim.x) {
    __syncthreads();
    const group_tile<G, C, SMALL> T(a, t);
    cell2 yo[C], north, south;                   // y; w_i0 beyond the wave's rows
    cell2 wg[G][C], F[G][C], d[C], e[C];
    north = y[T.at(T.row - 1)];
    south = y[T.at(T.row + C)];
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      yo[c] = y[T.at(T.row + c)];
      d[c] = e[c] = cell2{0.0, 0.0};
      static_for<G>([&](auto gt) {
        wg[decltype(gt)::value][c] = yo[c];
        F[decltype(gt)::value][c] = cell2{0.0, 0.0};
      });
    });
    if constexpr (!FIRST) {
      for (int j = 0; j < i0; ++j) {
        gcell *vj = v + j * cells;
        cell2 V[C];
        const cell2 vn = vj[T.at(T.row - 1)], vs = vj[T.at(T.row + C)];
        static_for<C>([&](auto ct) {
          constexpr int c = decltype(ct)::value;
          V[c] = vj[T.at(T.row + c)];
        });
        static_for<G>([&](auto gt) {
          constexpr int g = decltype(gt)::value;
          if ((row_nz[g] >> j) & 1u) {
            const double k = cl[g][j];
            static_for<C>([&](auto ct) {
              constexpr int c = decltype(ct)::value;
              wg[g][c].x += k * V[c].x;
              wg[g][c].y += k * V[c].y;
            });
            if constexpr (g == 0) {
              north.x += k * vn.x;
              north.y += k * vn.y;
              south.x += k * vs.x;
              south.y += k * vs.y;
            }
          }
        });
        if constexpr (LAST) {
          const double kb = cb[j], ke = ce[j];
          static_for<C>([&](auto ct) {
            constexpr int c = decltype(ct)::value;
            if (j == 0) {
              d[c] = cell2{kb * V[c].x, kb * V[c].y};
              e[c] = cell2{ke * V[c].x, ke * V[c].y};
            } else {
              if ((nzb >> j) & 1u) {
                d[c].x += kb * V[c].x;
                d[c].y += kb * V[c].y;
              }
              if ((nze >> j) & 1u) {
                e[c].x += ke * V[c].x;
                e[c].y += ke * V[c].y;
              }
            }
          });
        }
      }
    }
    T.stages(x, a.coef, north, south, wg, F,
             [&](int j, int g) { return cl[j][i0 + g]; },
             [&](int j, int g) { return ((row_nz[j] >> (i0 + g)) & 1u) != 0u; });

    const bool cin = T.col >= T.c0 && T.col < T.c1;
    static_for<C>([&](auto ct) {
      constexpr int c = decltype(ct)::value;
      if (cin && T.row + c >= T.r0 && T.row + c < T.r1) {
        const unsigned pos = T.at(T.row + c);
        if constexpr (!LAST) {
          static_for<G>([&](auto gt) {
            constexpr int g = decltype(gt)::value;
            (v + (i0 + g) * cells)[pos] = F[g][c];
          });
        } else {
          static_for<G>([&](auto gt) {
            constexpr int g = decltype(gt)::value;
            const int j = i0 + g;
            const double kb = cb[j], ke = ce[j];
            if (FIRST && g == 0) {
              d[c] = cell2{kb * F[g][c].x, kb * F[g][c].y};
              e[c] = cell2{ke * F[g][c].x, ke * F[g][c].y};
            } else {
              if ((nzb >> j) & 1u) {
                d[c].x += kb * F[g][c].x;
                d[c].y += kb * F[g][c].y;
              }
              if ((nze >> j) & 1u) {
                e[c].x += ke * F[g][c].x;
                e[c].y += ke * F[g][c].y;
              }
            }
          });
          const cell2 o = {yo[c].x + d[c].x, yo[c].y + d[c].y};
          yn[pos] = o;
          err_term(e[c].x, o.x, yo[c].x, qmax, zero);
          err_term(e[c].y, o.y, yo[c].y, qmax, zero);
        }
      }
    });
  }
  if constexpr (LAST)
    step_fold<W>(x.head, qmax, zero, x.red);
}

template <int G, int C, bool FIRST, bool LAST, bool SMALL>
void launch_kernel(int form, const stage_group &a, const gather_masks &nz, int grid,
                   hipStream_t stream)
{
  const dim3 g(grid), b(64 * kTileWaves);
  if (form == RKX_IMPL_D)
    hipLaunchKernelGGL((k_d_group<G, C, FIRST, LAST, SMALL>), g, b, 0, stream, a);
  else if (form == RKX_IMPL_A)
    hipLaunchKernelGGL((k_g_group<G, C, FIRST, LAST, SMALL, true>), g, b, 0, stream, a, nz);
  else
    hipLaunchKernelGGL((k_g_group<G, C, FIRST, LAST, SMALL, false>), g, b, 0, stream, a, nz);
}

template <int G, int C, bool FIRST, bool LAST>
hipError_t launch_group(int form, const stage_group &a, const gather_masks &nz, int grid,
                        hipStream_t stream)
{
  if (a.N < 64 || a.N < kTileWaves * C)
    launch_kernel<G, C, FIRST, LAST, true>(form, a, nz, grid, stream);
  else
    launch_kernel<G, C, FIRST, LAST, false>(form, a, nz, grid, stream);
  return hipGetLastError();
}

template <int G, int C>
hipError_t launch_group(bool first, bool last, int form, const stage_group &a,
                        const gather_masks &nz, int grid, hipStream_t stream)
{
  if (first)
    return last ? launch_group<G, C, true, true>(form, a, nz, grid, stream)
                : launch_group<G, C, true, false>(form, a, nz, grid, stream);
  return last ? launch_group<G, C, false, true>(form, a, nz, grid, stream)
              : launch_group<G, C, false, false>(form, a, nz, grid, stream);
}

// as few groups of up to four stages as there must be, of even sizes
int stage_groups(int s) { return (s + 3) / 4; }

template <int C>
hipError_t launch_shape(int form, stage_group a, const gather_masks &nz, hipStream_t stream)
{
  const int groups = stage_groups(a.s);
  for (int q = 0; q < groups; ++q) {
    const int i0 = q * a.s / groups, G = (q + 1) * a.s / groups - i0;
    a.i0 = i0;
    a.nstrips = tile_pieces(a.N, 64, G);
    a.nbands = tile_pieces(a.N, kTileWaves * C, G - 1);
    a.ntiles = a.nstrips * a.nbands;
    const bool first = q == 0, last = q == groups - 1;
    const int grid = std::min(a.ntiles, kGroupBlocks);
    hipError_t e = hipErrorInvalidValue;
    switch (G) {
    case 2: e = launch_group<2, C>(first, last, form, a, nz, grid, stream); break;
    case 3: e = launch_group<3, C>(first, last, form, a, nz, grid, stream); break;
    case 4: e = launch_group<4, C>(first, last, form, a, nz, grid, stream); break;
    default: break;
    }
    if (e != hipSuccess)
      return e;
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_groups(int form, const stage_group &a, const gather_masks &nz, hipStream_t stream)
{
  // the largest group's tiles are the most
  const int G = (a.s + stage_groups(a.s) - 1) / stage_groups(a.s);
  const int tiles = tile_pieces(a.N, 64, G) * tile_pieces(a.N, kTileWaves * kGroupRows[0], G - 1);
  return tiles <= kGroupBlocks ? launch_shape<kGroupRows[0]>(form, a, nz, stream)
                               : launch_shape<kGroupRows[1]>(form, a, nz, stream);
}

}  // namespace rkx
