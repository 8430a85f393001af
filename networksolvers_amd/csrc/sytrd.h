// k_sytrd: Householder tridiagonalisation Q^T A Q = T of a symmetric n x n matrix in one
// launch (LAPACK dsytd2 "lower" semantics on the column-major view); included by eig.hip.
//   for j = 0 .. n-2:  x = A(j+1:n, j), alpha = x_0, sigma^2 = |x_1:|^2, beta, tau, scal
//     (reflector, group.h), v = [1, x_1: scal], e_j = beta, p = tau A22 v,
//     w = p - (tau/2)(p.v) v,  A22 -= v w^T + w v^T,  d_j = A(j, j)
//
// Distribution: row i sits in the registers of one wave, wave w of workgroup g of G owning
// the rows (NW sl + w) G + g; lane l holds the columns from the current block of 64 on (as
// in bidiag.h, so every register index is a constant).  Every wave keeps its own copy of
// x, v, w at its lanes' columns.  Step j:
//   1. one wave-wide sum gives sigma^2 and, for each of the wave's rows i > j, the sum of
//      A(i, k) x_k over k > j + 1; p_i = tau (A(i, j+1) + scal sum) follows;
//   2. the wave publishes its p_i, and the owner of row j+1 that row (= column j+1 before
//      the update) as Y;
//   3. exchange: p and Y to everyone, as words that are polled until they are there
//      (group.h), the whole group on one XCD (want) or, past what one holds, over all
//      of them (want < 0);
//   4. w from a second wave-wide sum (p.v), the next column x_k = Y_k - v_k w_{j+1} - w_k,
//      d_{j+1} = Y_{j+1} - 2 w_{j+1}, and the rank-2 update of the wave's rows.
// v_i and p_i of a wave's own rows are the published ones (v through the wave's LDS copy):
// every wave uses the same v and w, so the update is one orthogonal similarity.
// The owner of row min(j + 2, n - 1) writes step j's results once the exchange is over
// (so nobody is still loading A) and empties step j - 1's Y.  A wave leaves after publishing its last row: it reads
// nothing any more, so nobody needs to hear from it before emptying a word.
// SHARED: the threads of a workgroup read each word once and pass it on through LDS (two
// workgroup barriers per step, NW times fewer reads); otherwise every wave reads all words
// itself and the waves run without any barrier.
// Output: d, e, tau, and v_j(k) for k >= j + 2 in A[j n + k].
#pragma once
#include "group.h"

namespace nsmi {
namespace {

// up to 512 columns two workgroups fit a CU (the register bound)
template <int CL, int RW, int NW, bool SHARED>
__global__ __launch_bounds__(64 * NW, CL > 8 ? 1 : NW / 2) void k_sytrd(
    double* __restrict__ A, int n, double* __restrict__ d, double* __restrict__ e, double* __restrict__ tau,
    double* __restrict__ xch, unsigned* __restrict__ ctl, int G, int want) {
  constexpr int STEP = CL > 8 ? 2 : 1;
  constexpr int NP = 64 * (CL + STEP - 1), NT = 64 * NW, NY = (64 * CL + NT - 1) / NT, SP = 64 * CL;
  __shared__ double vl[NW][NP];                           // each wave's v, by column
  __shared__ double ps[SHARED ? NP : 1], yv[SHARED ? NP : 1];
  __shared__ int s_ok, s_place;
  static_assert(CL > 8 || sizeof(vl) + sizeof(ps) + sizeof(yv) < 160 * 1024 / 3,
                "two workgroups of one-XCD groups share a CU");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned* const fail = ctl + kCtlFail;
  const bool local = want >= 0;  // else a group over all XCDs: the words go past L2
  const int g = local ? place_one_xcd(ctl, G, want, &s_place) : place_spread(ctl, &s_place);
  if (g < 0 || told_to_give_up(ctl, g)) return;
  double* const P = xch;            // [3][SP]
  double* const Y = xch + 3 * SP;   // [3][SP]

  double row[RW][CL], xs[CL];
  int rid[RW];
#pragma unroll
  for (int sl = 0; sl < RW; ++sl) {
    const int i = rid[sl] = (sl * NW + wave) * G + g;
#pragma unroll
    for (int q = 0; q < CL; ++q) {
      const int k = lane + 64 * q;
      row[sl][q] = (i < n && k < n) ? A[size_t(i) * n + k] : 0.0;
    }
  }
  // the last row of this wave (SHARED: of this workgroup)
  int last = -1;
  if (SHARED) {
    if (g < n) last = g + G * ((n - 1 - g) / G);
  } else {
#pragma unroll
    for (int sl = 0; sl < RW; ++sl) last = rid[sl] < n ? rid[sl] : last;
  }
  // x_0 = column 0 = row 0 (symmetric), without its first two entries; alpha = A(1, 0)
#pragma unroll
  for (int q = 0; q < CL; ++q) {
    const int k = lane + 64 * q;
    xs[q] = k >= 1 && k < n ? A[k] : 0.0;
  }
  double alpha = lane_bcast(xs[0], 1);
  if (lane <= 1) xs[0] = 0.0;
  bool finite = true;
  if (rid[0] == 0) {
    const double d0 = lane_bcast(row[0][0], 0);
    if (lane == 0) d[0] = d0;
    finite = isfinite(d0);
  }
  if (tid == 0) s_ok = 1;
  if (SHARED) {
    for (int k = tid; k < NP; k += NT) ps[k] = yv[k] = 0.0;
    __syncthreads();
  }
  int p3 = 0, pm = 2, cb = 0;
  bool left = false;
  const auto block = [&](auto ca) __attribute__((always_inline)) {
    constexpr int CA = decltype(ca)::value;
    const int jend = min(64, n - 1 - cb);
    for (int jl = 0; jl < jend; ++jl) {
      const int j = cb + jl;
      // 1. sums over the columns k > j + 1 (xs is zero up to j + 1)
      double red[RW + 1];
#pragma unroll
      for (int sl = 0; sl <= RW; ++sl) red[sl] = 0.0;
#pragma unroll
      for (int q = 0; q < CA; ++q) {
        red[RW] = fma(xs[q], xs[q], red[RW]);
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) red[sl] = fma(row[sl][q], xs[q], red[sl]);
      }
      // A(i, j+1) of the own rows: lane jl + 1 of block 0, or lane 0 of block 1
      const bool at0 = lane == jl + 1, at1 = jl == 63 && lane == 0;
      double a1[RW];
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) a1[sl] = lane_bcast(row[sl][0], min(jl + 1, 63));
      if constexpr (CA > 1)
        if (jl == 63) {
#pragma unroll
          for (int sl = 0; sl < RW; ++sl) a1[sl] = lane_bcast(row[sl][1], 0);
        }
      wave_sums<RW + 1>(red);
      double beta, t, scal;
      reflector(alpha, red[RW], &beta, &t, &scal);
      double v[CA];
#pragma unroll
      for (int q = 0; q < CA; ++q) v[q] = xs[q] * scal;
      v[0] = at0 ? 1.0 : v[0];
      if constexpr (CA > 1) v[1] = at1 ? 1.0 : v[1];
#pragma unroll
      for (int q = 0; q < CA; ++q) vl[wave][cb + lane + 64 * q] = v[q];
      wave_sync_lds();
      // 2.
      double pr[RW];
      stores_done();  // the emptied words
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) {
        pr[sl] = t * fma(scal, red[sl], a1[sl]);
        if (rid[sl] <= j || rid[sl] >= n) continue;  // uniform per wave
        if (lane == 0) st_group(P + p3 * SP + rid[sl], pr[sl], local);
        if (rid[sl] == j + 1) {
#pragma unroll
          for (int q = 0; q < CA; ++q) {
            const int k = cb + lane + 64 * q;
            if (k > j && k < n) st_group(Y + p3 * SP + k, not_empty(row[sl][q]), local);
          }
        }
      }
      if (last <= j + 1 && j + 2 < n) {
        left = true;
        return false;
      }
      // 3. (lanes and threads without a column read the last one)
      double pk[SHARED ? 1 : CA], yk[SHARED ? 1 : CA];  // SHARED: read from LDS where they are used
      const auto p_at = [&](int q) { return SHARED ? ps[cb + lane + 64 * q] : pk[SHARED ? 0 : q]; };
      const auto y_at = [&](int q) { return SHARED ? yv[cb + lane + 64 * q] : yk[SHARED ? 0 : q]; };
      if constexpr (SHARED) {
        double w[2 * NY];
        if (!load_words(w, [&](int i) {
              const int k = tid + NT * (i >> 1);
              return ((i & 1) ? Y : P) + p3 * SP + (k > j && k < n ? k : n - 1);
            }, fail))
          s_ok = 0;
        __syncthreads();  // the previous step's reads of ps and yv are over
#pragma unroll
        for (int u = 0; u < NY; ++u) {
          const int k = tid + NT * u;
          if (k < NP && k < n) {
            ps[k] = k > j ? w[2 * u] : 0.0;
            yv[k] = k > j ? w[2 * u + 1] : 0.0;
          }
        }
        __syncthreads();
        if (!s_ok) return false;
      } else {
        double w[2 * CA];
        if (!load_words(w, [&](int i) {
              const int k = cb + lane + 64 * (i >> 1);
              return ((i & 1) ? Y : P) + p3 * SP + (k > j && k < n ? k : n - 1);
            }, fail))
          return false;
#pragma unroll
        for (int q = 0; q < CA; ++q) {
          const int k = cb + lane + 64 * q;
          const bool in = k > j && k < n;
          pk[q] = in ? w[2 * q] : 0.0;
          yk[q] = in ? w[2 * q + 1] : 0.0;
        }
      }
      // everyone heard from has finished reading step j - 1
      if (j > 0) {
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) {
          if (rid[sl] < j || rid[sl] >= n) continue;
          if (lane == 0) st_group(P + pm * SP + rid[sl], empty_word(), local);
        }
      }
      // 4.
      double pv[1] = {0.0};
#pragma unroll
      for (int q = 0; q < CA; ++q) pv[0] = fma(p_at(q), v[q], pv[0]);
      double vi[RW];
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) vi[sl] = vl[wave][min(rid[sl], NP - 1)];
      double p1, y1;
      if constexpr (SHARED) {
        p1 = ps[j + 1];
        y1 = yv[j + 1];
      } else {
        p1 = lane_bcast(pk[0], min(jl + 1, 63));
        y1 = lane_bcast(yk[0], min(jl + 1, 63));
        if constexpr (CA > 1)
          if (jl == 63) {
            p1 = lane_bcast(pk[1], 0);
            y1 = lane_bcast(yk[1], 0);
          }
      }
      wave_sums<1>(pv);
      const double cc = 0.5 * t * pv[0];
      const double w1 = p1 - cc;  // w_{j+1}, as v_{j+1} = 1
      double wi[RW];
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) wi[sl] = fma(-cc, vi[sl], pr[sl]);
#pragma unroll
      for (int q = 0; q < CA; ++q) {
        const double ww = fma(-cc, v[q], p_at(q));
        xs[q] = fma(-v[q], w1, y_at(q)) - ww;
#pragma unroll
        for (int sl = 0; sl < RW; ++sl) row[sl][q] = fma(-vi[sl], ww, fma(-wi[sl], v[q], row[sl][q]));
      }
      // the next column: alpha is its entry j + 2, xs keeps the entries beyond
      if (at0 || lane == jl) xs[0] = 0.0;
      if constexpr (CA > 1) {
        if (jl < 62) {
          alpha = lane_bcast(xs[0], min(jl + 2, 63));
        } else {
          alpha = lane_bcast(xs[1], jl - 62);
          if (jl == 63 ? lane <= 1 : lane == 0) xs[1] = 0.0;
        }
      } else {
        alpha = lane_bcast(xs[0], min(jl + 2, 63));
      }
      if (lane == jl + 2) xs[0] = 0.0;
      const int writer = min(j + 2, n - 1);
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) {
        if (rid[sl] != writer) continue;
        const double dn = y1 - 2.0 * w1;
#pragma unroll
        for (int q = 0; q < CA; ++q) {
          const int k = cb + lane + 64 * q;
          if (k >= j + 2 && k < n) A[size_t(j) * n + k] = v[q];
          // step j - 1's Y (whose writer may have left)
          if (j > 0 && k >= j && k < n) st_group(Y + pm * SP + k, empty_word(), local);
        }
        if (lane == 0) {
          e[j] = beta;
          tau[j] = t;
          d[j + 1] = dn;
        }
        finite = finite && isfinite(beta) && isfinite(dn);
      }
      pm = p3;
      p3 = p3 == 2 ? 0 : p3 + 1;
    }
#pragma unroll
    for (int q = 0; q + 1 < CA; ++q) {
      xs[q] = xs[q + 1];
#pragma unroll
      for (int sl = 0; sl < RW; ++sl) row[sl][q] = row[sl][q + 1];
    }
    xs[CA - 1] = 0.0;  // beyond the matrix
    return true;
  };
  const bool done = column_blocks<CL, STEP>(n - 1, n, cb, block);
  if ((done || left) && lane == 0 && !finite) ctl[kCtlNonFinite] = 1u;
  if (lane == 0 && (g == 0 || !(done || left))) ended_at(ctl, done || left ? n : cb);
}

}  // namespace
}  // namespace nsmi
