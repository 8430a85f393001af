// k_bidiag: Householder bidiagonalisation X = Q_L B Q_R^T of a tall r x s matrix in one
// launch (LAPACK dgebrd semantics: upper bidiagonal B, left reflector H_j on X(j:r, j),
// right reflector G_j on X(j, j+1:s)); included by svd.hip.
//
// Distribution: workgroup g of G owns the rows i = (NW sl + w) G + g of X, slot sl of wave
// w, in registers; lane l holds the columns l + 64 q.  Step j:
//   A. every row owner has its x_i = X(i, j) (i > j); each workgroup forms the partial
//      sums S_c = sum_{own i > j} x_i X(i, c) (c >= j; S_j is its share of sigma^2), and
//      the owner of row j publishes that row (before the update);
//   exchange: every workgroup gets row j and the sums of S over all workgroups;
//   B. every wave forms the left reflector (alpha = X(j, j), beta = -sign(alpha)
//      sqrt(alpha^2 + sigma^2), tau_L = (beta - alpha) / beta, u = [1, x / (alpha -
//      beta)]), z = u^T X(j:, c) = X(j, c) + S_c / (alpha - beta), and updates its rows,
//      X(i, c) -= tau_L u_i z_c; row j after the update is y_c = X(j, c) - tau_L z_c.
//      One wave-wide sum then gives |y_{j+2:}|^2 and, for each of its rows,
//      a_i = X(i, j+2:) . y_{j+2:}; the right reflector v = [1, y_{j+2:} scal_R] and
//      X(i, :) v = X(i, j+1) + scal_R a_i follow without another sum, the rows take
//      X(i, c) -= tau_R (X(i, :) v) v_c, and X(i, j+1) is the next step's x_i.
// The columns are walked in blocks of 64: the lanes' registers always hold the columns
// from the current block on (the block's own in q = 0, so no register is picked by a
// run-time index), and when a block is done the rows that are still active store its
// column of u's and the registers move down by one.  Row j is stored by its owner as
// soon as it is finished.  Output in place: X(i, j) = u_j[i] for i > j, X(j, j) = d_j,
// X(j, j+1) = e_j, X(j, c) = v_j[c] for c > j + 1; d, e, tau_L, tau_R.
//
// Exchange (group.h: words are polled until they are there), thread t handling the
// columns c = t mod NT, by MODE:
//   kOneGroup  one workgroup, through LDS;
//   kOneXcd    G workgroups on XCD `want` (want < 0: anywhere): each publishes its S, everyone adds the G values
//              of every column in order;
//   kAllXcds   8 GW workgroups, GW on each XCD: each publishes its S to its XCD; workgroup w
//              of each XCD adds its slice of the columns over that XCD's GW workgroups;
//              the eight workgroups w trade their slices across the XCDs, add them, and
//              publish the sums and row j's slice to their XCD, where everyone reads them.
//              (All-to-all reads would move G^2 s doubles per column.)
// Every sum has a fixed order: the result does not depend on timing.  A column leaves
// the exchange two steps after it is finished, by blocks of 64 (lo below), so that the
// buffer rotation's condition holds for every column that still takes part.
#pragma once
#include "group.h"

namespace nsmi {
namespace {

enum BidiagMode { kOneGroup, kOneXcd, kOneXcdSliced, kAllXcds };

// Exchange memory, in rows of SP = 64 CL doubles: PS [slots][3] (slots: GMAX workgroups, or
// 32 for each XCD; the slots no workgroup fills hold zeros, so readers take all of them
// without a look at G), Y [3], then RS [3] or, over all XCDs, XP [8][3] and RS [8][3][2].
struct BidiagExchange {
  int slots, per, used;  // PS slots, slots per group, slots filled in each group
  size_t words, ps_words;
};
inline BidiagExchange bidiag_exchange(int cl, int gmax, int groups, bool all) {
  const size_t sp = size_t(64) * cl;
  BidiagExchange x;
  x.per = all ? 32 : gmax;
  x.slots = all ? 32 * kXcds : gmax;
  x.used = groups;
  x.ps_words = 3 * sp * x.slots;
  x.words = x.ps_words + 3 * sp * (2 + (all ? 3 * kXcds : 0));
  return x;
}

// waves per SIMD: the workgroups of a one-XCD group keep to half of a CU's registers, so that
// two fit a CU
constexpr int bidiag_occupancy(int nw, BidiagMode mode) {
  return mode == kOneXcd || mode == kOneXcdSliced ? nw / 2 : 1;
}

template <int CL, int RW, int NW, BidiagMode MODE, int GMAX = 16>
__global__ __launch_bounds__(64 * NW, bidiag_occupancy(NW, MODE)) void k_bidiag(
    double* __restrict__ X, int r, int s, double* __restrict__ d, double* __restrict__ e, double* __restrict__ tauL,
    double* __restrict__ tauR, double* __restrict__ xch, unsigned* __restrict__ ctl, int groups, int want) {
  constexpr int STEP = CL > 16 ? 4 : (CL > 8 ? 2 : 1);
  constexpr int NP = 64 * (CL + STEP - 1), NT = 64 * NW, NY = (64 * CL + NT - 1) / NT;
  __shared__ double comb[NW][NP];    // from the current block on
  __shared__ double yrow[NP];        // row j from the current block on, in its owner's workgroup
  __shared__ double ys[NP], zs[NP];  // row j and the sums by column, zero for c <= j and c >= s
  __shared__ double part[MODE == kAllXcds || MODE == kOneXcdSliced ? NW : 1][64];
  __shared__ double s_alpha, s_sig;
  __shared__ int s_ok, s_place;
  // beside one workgroup of another group, wherever that one lies in a CU's 160 KB
  static_assert(MODE == kAllXcds || sizeof(comb) + sizeof(yrow) + sizeof(ys) + sizeof(zs) + sizeof(part) < 160 * 1024 / 3,
                "two workgroups of one-XCD groups share a CU");
  // the wave's index and the workgroup's place are wave-uniform: branches on them are scalar
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned* const fail = ctl + kCtlFail;
  int G = 1, g = 0, xx = 0, ww = 0;
  const int GW = groups;
  bool local = true;
  constexpr bool ALL = MODE == kAllXcds, SLICED = ALL || MODE == kOneXcdSliced;
  if (MODE == kOneXcd || MODE == kOneXcdSliced) {
    G = groups;
    local = want >= 0;
    g = local ? place_one_xcd(ctl, G, want, &s_place) : place_spread(ctl, &s_place);
    if (g < 0) return;
  } else if (MODE == kAllXcds) {
    if (!place_all_xcds(ctl, GW, want, &xx, &ww, &local, &s_place)) return;
    G = kXcds * GW;
    g = ww * kXcds + xx;
  }
  if (MODE != kOneGroup && told_to_give_up(ctl, g)) return;
  constexpr int SP = 64 * CL, SLOTS = ALL ? 32 * kXcds : GMAX;
  double* const PS = xch;                               // [SLOTS][3][SP], an XCD's workgroups together
  double* const Yx = PS + 3 * SLOTS * SP;               // [3][SP]
  double* const XP = Yx + 3 * SP;                       // [8][3][SP]
  double* const RS = XP + (ALL ? 3 * kXcds * SP + 6 * SP * xx : 0); // [3][2][SP] of this XCD
  double* const myPS = PS + 3 * SP * (ALL ? 32 * xx + ww : g);
  const bool ylocal = !ALL && local;

  double row[RW][CL];
  double xi[RW];
  int rid[RW];
#pragma unroll
  for (int sl = 0; sl < RW; ++sl) {
    const int i = rid[sl] = (sl * NW + wave) * G + g;
#pragma unroll
    for (int q = 0; q < CL; ++q) {
      const int c = lane + 64 * q;
      row[sl][q] = (i < r && c < s) ? X[size_t(i) * s + c] : 0.0;
    }
    xi[sl] = i > 0 ? lane_bcast(row[sl][0], 0) : 0.0;
  }
  for (int c = tid; c < NP; c += NT) ys[c] = zs[c] = 0.0;
  if (tid == 0) s_ok = 1;
  const int chunk = (s + GW - 1) / GW;  // SLICED: columns per workgroup of an XCD
  bool finite = true;
  int p = 0, pm = 2, jg = 0;  // j mod 3, (j - 1) mod 3, j mod G
  int cb = 0;  // the current block's first column
  const auto block = [&](auto ca) __attribute__((always_inline)) {
    constexpr int CA = decltype(ca)::value;
    const int jend = min(64, s - cb);
    for (int jl = 0; jl < jend; ++jl) {
      const int j = cb + jl;
      // A.
#pragma unroll
      for (int q = 0; q < CA; ++q) {
        double acc = xi[0] * row[0][q];
#pragma unroll
        for (int sl = 1; sl < RW; ++sl) acc = fma(xi[sl], row[sl][q], acc);
        comb[wave][lane + 64 * q] = acc;
      }
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) {
        if (rid[sl] == j) {
#pragma unroll
          for (int q = 0; q < CA; ++q) yrow[lane + 64 * q] = row[sl][q];
        }
      }
      __syncthreads();
      if constexpr (MODE == kOneGroup) {
#pragma unroll
        for (int u = 0; u < NY; ++u) {
          const int c = tid + NT * u;
          if (c < cb || c >= s) continue;
          double t = 0.0;
#pragma unroll
          for (int w = 0; w < NW; ++w) t += comb[w][c - cb];
          const double yv = yrow[c - cb];
          zs[c] = c > j ? t : 0.0;
          ys[c] = c > j ? yv : 0.0;
          if (c == j) {
            s_alpha = yv;
            s_sig = t;
          }
        }
      } else {
        const int lo = 64 * (max(j - 2, 0) >> 6);
        const bool owner = jg == g;
        stores_done();  // the emptied words
#pragma unroll
        for (int u = 0; u < NY; ++u) {
          const int c = tid + NT * u;
          if (c < lo || c >= s) continue;
          double t = 0.0, yv = 0.0;
          if (c >= cb) {
#pragma unroll
            for (int w = 0; w < NW; ++w) t += comb[w][c - cb];
            if (owner) yv = not_empty(yrow[c - cb]);
          }
          st_group(myPS + p * SP + c, t, local);
          if (owner) st_group(Yx + p * SP + c, yv, ylocal);
        }
        if constexpr (SLICED) {
          // this workgroup's slice of the columns (at most 64): the sum over its XCD, part
          // of the workgroups per wave, then over the XCDs by wave 0.  Lanes without a
          // column read the slice's last one.
          const int c0 = (ALL ? ww : g) * chunk, ce = min(c0 + chunk, s);
          if (c0 < s && ce > lo) {
            const int c = max(lo, min(c0 + lane, ce - 1));
            const bool live = c == c0 + lane;
            constexpr int NB = (ALL ? 32 : GMAX) / NW;
            const double* const src = PS + 3 * SP * (32 * xx + wave) + p * SP + c;
            double v[NB], t;
            if (!load_words(v, [&](int b) { return src + 3 * SP * NW * b; }, fail)) s_ok = 0;
            t = 0.0;
#pragma unroll
            for (int b = 0; b < NB; ++b) t += v[b];
            part[wave][lane] = t;
            __syncthreads();
            if (wave == 0) {
              t = 0.0;
#pragma unroll
              for (int w = 0; w < NW; ++w) t += part[w][lane];
              if (MODE == kOneXcdSliced && live) {
                st_group(RS + p * SP + c, t, local);
                if (j > 0) st_group(RS + pm * SP + c, empty_word(), local);
              }
            }
            if (ALL && wave == 0) {
              if (live) st_agent(XP + (3 * xx + p) * SP + c, t);
              double x[kXcds + 1];  // the eight sums, then row j
              if (!load_words(x, [&](int q) { return q < kXcds ? XP + (3 * q + p) * SP + c : Yx + p * SP + c; }, fail))
                s_ok = 0;
              t = 0.0;
#pragma unroll
              for (int q = 0; q < kXcds; ++q) t += x[q];
              if (live) {
                st_group(RS + 2 * p * SP + c, t, local);
                st_group(RS + (2 * p + 1) * SP + c, x[kXcds], local);
                if (j > 0) {
                  st_agent(XP + (3 * xx + pm) * SP + c, empty_word());
                  st_group(RS + 2 * pm * SP + c, empty_word(), local);
                  st_group(RS + (2 * pm + 1) * SP + c, empty_word(), local);
                }
              }
            }
          }
        }
        // every thread: the sums and row j of its columns (threads without one read the last)
        double zv[NY], yv[NY];
        if constexpr (SLICED) {
          double v[2 * NY];
          if (!load_words(v, [&](int i) {
                const int c = tid + NT * (i >> 1), cc = c >= lo && c < s ? c : s - 1;
                if (ALL) return RS + (2 * p + (i & 1)) * SP + cc;
                return ((i & 1) ? Yx : RS) + p * SP + cc;
              }, fail))
            s_ok = 0;
#pragma unroll
          for (int u = 0; u < NY; ++u) {
            zv[u] = v[2 * u];
            yv[u] = v[2 * u + 1];
          }
        } else {
#pragma unroll
          for (int u = 0; u < NY; ++u) {
            const int c = tid + NT * u, cc = c >= lo && c < s ? c : s - 1;
            double v[GMAX + 1];
            if (!load_words(v, [&](int b) { return b < GMAX ? PS + (p * SP + cc + 3 * SP * b) : Yx + p * SP + cc; }, fail))
              s_ok = 0;
            double t = 0.0;
#pragma unroll
            for (int b = 0; b < GMAX; ++b) t += v[b];
            zv[u] = t;
            yv[u] = v[GMAX];
          }
        }
        const bool was_owner = (jg == 0 ? G - 1 : jg - 1) == g;  // of row j - 1
#pragma unroll
        for (int u = 0; u < NY; ++u) {
          const int c = tid + NT * u;
          if (c < lo || c >= s) continue;
          zs[c] = c > j ? zv[u] : 0.0;
          ys[c] = c > j ? yv[u] : 0.0;
          if (c == j) {
            s_alpha = yv[u];
            s_sig = zv[u];
          }
          // everyone heard from has finished reading step j - 1
          if (j > 0) {
            st_group(myPS + pm * SP + c, empty_word(), local);
            if (was_owner) st_group(Yx + pm * SP + c, empty_word(), ylocal);
          }
        }
      }
      __syncthreads();
      if (MODE != kOneGroup && !s_ok) return false;
      // B. left reflector
      double beta, tl, scal;
      reflector(s_alpha, s_sig, &beta, &tl, &scal);
      double f[RW], un[RW], red[RW + 1];
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) {
        un[sl] = xi[sl] * scal;  // zero for rows up to j
        f[sl] = tl * un[sl];
        red[sl] = 0.0;
      }
      red[RW] = 0.0;
      // column j + 1 (the next step's x, not part of y_{j+2:}) is lane jl + 1 of block 0, or
      // lane 0 of block 1
      const bool at0 = lane == jl + 1, at1 = jl == 63 && lane == 0;
      double y2[CA], xn[RW], alpha2 = 0.0;
#pragma unroll
      for (int q = 0; q < CA; ++q) {
        const double yc = ys[cb + lane + 64 * q];
        const double zc = fma(scal, zs[cb + lane + 64 * q], yc);
        y2[q] = fma(-tl, zc, yc);
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) row[sl][q] = fma(-f[sl], zc, row[sl][q]);
        if (q == 0) {
          alpha2 = lane_bcast(y2[0], min(jl + 1, 63));
#pragma unroll
          for (int sl = 0; sl < RW; ++sl) xn[sl] = lane_bcast(row[sl][0], min(jl + 1, 63));
          if (at0) y2[0] = 0.0;
        }
        if constexpr (CA > 1) {
          if (q == 1) {
            if (jl == 63) {
              alpha2 = lane_bcast(y2[1], 0);
#pragma unroll
              for (int sl = 0; sl < RW; ++sl) xn[sl] = lane_bcast(row[sl][1], 0);
            }
            if (at1) y2[1] = 0.0;
          }
        }
        red[RW] = fma(y2[q], y2[q], red[RW]);
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) red[sl] = fma(row[sl][q], y2[q], red[sl]);
      }
      if (j + 1 >= s) {  // no column j + 1 (jl = 63: lane 63 above is column j)
        alpha2 = 0.0;
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) xn[sl] = 0.0;
      }
      wave_sums<RW + 1>(red);
      double beta2, tr, scal2;
      reflector(alpha2, red[RW], &beta2, &tr, &scal2);
      double h[RW];
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) {
        const double hv = tr * fma(scal2, red[sl], xn[sl]);
        h[sl] = hv * scal2;
        xn[sl] -= hv;
        xi[sl] = rid[sl] > j + 1 ? xn[sl] : 0.0;
      }
#pragma unroll
      for (int q = 0; q < CA; ++q) {
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) row[sl][q] = fma(-h[sl], y2[q], row[sl][q]);
        if (q == 0) {
#pragma unroll
          for (int sl = 0; sl < RW; ++sl) row[sl][0] = at0 ? xn[sl] : (lane == jl ? un[sl] : row[sl][0]);
        }
        if constexpr (CA > 1) {
          if (q == 1) {
#pragma unroll
            for (int sl = 0; sl < RW; ++sl) row[sl][1] = at1 ? xn[sl] : row[sl][1];
          }
        }
      }
      // row j is finished: its owner stores d_j, e_j and v_j (u's of earlier blocks are stored)
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) {
        if (rid[sl] == j) {
          double* const xr = X + size_t(j) * s + cb;
#pragma unroll
          for (int q = 0; q < CA; ++q) {  // the columns left: cb + 64 CA >= s
            const int c = lane + 64 * q;
            double v = y2[q] * scal2;
            if (q == 0) v = lane < jl ? row[sl][0] : (lane == jl ? beta : (at0 ? beta2 : v));
            if (q == 1 && at1) v = beta2;
            if (cb + c < s) xr[c] = v;
          }
          if (lane == 0) {
            d[j] = beta;
            tauL[j] = tl;
            if (j + 1 < s) {
              e[j] = beta2;
              tauR[j] = tr;
            }
          }
          finite = finite && isfinite(beta) && isfinite(beta2);
        }
      }
      pm = p;
      p = p == 2 ? 0 : p + 1;
      jg = jg + 1 == G ? 0 : jg + 1;
    }
    // the block's columns are done: u's of the rows that are still active, registers down by one
#pragma unroll
    for (int sl = 0; sl < RW; ++sl) {
      const int i = rid[sl];
      if (i >= cb + jend && i < r && lane < jend) X[size_t(i) * s + cb + lane] = row[sl][0];
#pragma unroll
      for (int q = 0; q + 1 < CA; ++q) row[sl][q] = row[sl][q + 1];
    }
    return true;
  };
  const bool done = column_blocks<CL, STEP>(s, s, cb, block);
  if (MODE != kOneGroup && tid == 0 && (!done || g == 0)) ended_at(ctl, done ? s : cb);
  if (!done) return;
  if (lane == 0 && !finite) ctl[kCtlNonFinite] = 1u;
}

}  // namespace
}  // namespace nsmi
