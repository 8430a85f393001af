// The truncation's own dense eigensolver and SVD (inserter.jl:23 -> ITensors
// factorize -> LAPACK gesdd on the "svd" route, syevd on the "eigen" route):
//
//  * k_bidiag (bidiag.h): Householder bidiagonalisation X = Q_L B Q_R^T of a tall r x s
//    matrix (r >= s, s <= 2048, r <= 4096, r <= 2048 for s > 1024) in one launch;
//  * k_tri_bisect: eigenvalues of a symmetric tridiagonal matrix by Sturm-count
//    multisection, one wave per eigenvalue.  Applied to the Golub-Kahan matrix of
//    B (zero diagonal, off-diagonal d_0, e_0, d_1, e_1, ...; eigenvalues +-sigma)
//    it gives the singular values with the accuracy of a bidiagonal SVD;
//  * k_tri_invit_lds / _glb: eigenvectors for given eigenvalues by inverse
//    iteration (LU with partial pivoting of T - lambda I), one wave per vector,
//    the factors in LDS (N <= 1024) or in global memory (N <= 4096).  The
//    Golub-Kahan eigenvector of sigma is (v_0, u_0, v_1, u_1, ...) / sqrt(2) with
//    B v = sigma u, B^T u = sigma v;
//  * k_chol_inv + GEMMs: CholQR in two passes, by blocks of 64 columns with two
//    block Gram-Schmidt projections (CGS2), turning the inverse-iteration vectors
//    into an orthonormal set (vectors of clustered eigenvalues are only
//    independent, not orthogonal, after inverse iteration);
//  * k_build_vt_left / _right: the reflector rows for the compact-WY
//    back-transformation (apply_reflectors, eig.hip).
#include "internal.h"
#include "wave.h"

namespace nsmi {
namespace {

constexpr double kEps = 2.220446049250313e-16;
constexpr double kSafeMin = 2.2250738585072014e-308;

// ---------------------------------------------------------------- bisection
//
// Eigenvalues of a symmetric tridiagonal T by Sturm counts: the number of eigenvalues
// below sigma is the number of negative pivots of the LDL^T factorisation of T - sigma
// I, q_0 = a_0 - sigma, q_i = a_i - sigma - b_{i-1}^2 / q_{i-1}, a pivot within pivmin of
// zero counting as negative and replaced by -pivmin (LAPACK dlaebz).  One wave per wanted
// eigenvalue (ascending index t): each pass evaluates the count at 64 shifts inside the
// bracket [lo, hi) (count(lo) <= t < count(hi)) and keeps the sub-bracket where the count
// crosses t; it stops at relative width 2 eps (plus pivmin), which for the Golub-Kahan
// matrix is the relative accuracy of the singular values (LAPACK's bidiagonal SVD keeps
// singular values far below eps sigma_max, and with cutoff 0 whether such a value is kept
// depends on it).  The first pass has one shift at zero and the others a factor 2 apart
// down to 2^-63 of the bound; after it a bracket around zero puts one shift at zero, a
// bracket of one sign whose ends differ by more than a factor 2 takes shifts spaced
// geometrically between its inner end (at least 2 pivmin) and its outer end, any other
// takes them evenly: 10 passes for a value above 2^-63 of the bound.  (Two or four waves
// per eigenvalue save one or two passes, but do 1.8 or 3.2 times the work: with the five
// sectors of a block-sparse bond side by side the split went from 2.4 to 3.2 ms.)
//
// T is scaled by a power of two to a norm bound in [1, 2), so pivmin = 2^-500 is far below
// every resolved eigenvalue and 1 / pivmin far from overflow.  A step's chain is the
// reciprocal, three multiply-adds and one select; the guard is tested beside them, and
// what a guarded pivot leads to replaces the next one.
// GK (a Golub-Kahan matrix: zero diagonal, off-diagonal d_0, e_0, d_1, ...; the wanted
// eigenvalues are its non-negative half): the pivots are taken in pairs.  With u the even
// pivot and m = sigma u + d^2, the odd pivot is -m / u and the next even one -sigma +
// e^2 u / m: one reciprocal for two pivots, half the chain.  Every operation's rounding is
// still a relative perturbation of a few ulps in some d^2 or e^2, so the singular values
// keep their relative accuracy.
// Steps go in blocks whose LDS reads are issued a block ahead, padded so that a block has
// no branches.  Measured against one reciprocal per pivot and 12 passes: 394 singular
// values 379 -> 216 us, 2048 3180 -> 1870 us, 154 eigenvalues of order 154 100 -> 81 us.
//
// recip: 1 / y by the hardware reciprocal and two Newton steps r += r (1 - y r), within an
// ulp or two of the rounded quotient on a dependency chain half as long as a division's.
__device__ __forceinline__ double recip(double y) {
  double r = __builtin_amdgcn_rcp(y);
  r = fma(fma(-y, r, 1.0), r, r);
  return fma(fma(-y, r, 1.0), r, r);
}

constexpr double kPivMin = 0x1p-500, kPivMinInv = 0x1p500;

// shift idx of the 64 of a pass over [lo, hi)
__device__ inline double bisect_shift(int idx, bool first, double lo, double hi) {
  if (first) return idx == 0 ? 0.0 : ldexp(hi, idx - 64);
  constexpr double kFloor = 2.0 * kPivMin;
  const double frac = double(idx + 1) * (1.0 / 65.0);
  double sig;
  if (lo >= 0.0 && hi > 2.0 * fmax(lo, kFloor)) {
    const double lb = log2(fmax(lo, kFloor)), lh = log2(hi);
    sig = exp2(lb + (lh - lb) * frac);
  } else if (hi <= 0.0 && -lo > 2.0 * fmax(-hi, kFloor)) {
    const double lb = log2(fmax(-hi, kFloor)), lh = log2(-lo);
    sig = -exp2(lb + (lh - lb) * (1.0 - frac));
  } else {
    sig = lo + (hi - lo) * frac;
    const double prev = lo + (hi - lo) * (double(idx) * (1.0 / 65.0));
    if (lo < 0.0 && hi > 0.0 && sig >= 0.0 && prev < 0.0) sig = 0.0;
  }
  return fmin(fmax(sig, lo), hi);
}

// r y - c for r = 1 / m from the hardware reciprocal and one third-order correction, the
// correction folded into the result: with e = 1 - m r0, 1 / m = r0 (1 + e + e^2 + ...), so
// y r0 (e + e^2) + (y r0 - c); two multiply-adds of chain after the reciprocal and e
__device__ __forceinline__ double div_sub(double y, double m, double c) {
  const double r = __builtin_amdgcn_rcp(m);
  const double e = fma(-m, r, 1.0);
  return fma(y * r, fma(e, e, e), fma(y, r, -c));
}

// steps of a block, and the LDS of `steps` padded steps (16 bytes each)
constexpr int kB = 8;
constexpr size_t bisect_lds(int steps) { return 16 * size_t((steps + kB - 1) / kB * kB + kB); }
// 64 KiB with the kernel's 32 static bytes: order 4081 with a diagonal, 4096 without
constexpr size_t kBisectLds = 64 * 1024 - 32;
static_assert(bisect_lds(kSytrdMax - 1) <= kBisectLds && bisect_lds(kTriSolveMaxN / 2) <= kBisectLds,
              "the tridiagonal reduction's largest order and the Golub-Kahan one's");

template <bool GK>
__global__ __launch_bounds__(256) void k_tri_bisect(const double* __restrict__ a, const double* __restrict__ b, int N,
                                                    int i0, int count, double* __restrict__ lam) {
  // (d_i^2, e_i^2) of pair i (GK), or (b_i^2, a_{i+1}) of step i, padded to whole blocks
  extern __shared__ __align__(16) double sm[];
  double2* const st = reinterpret_cast<double2*>(sm);
  __shared__ double redb[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double bound = 0.0;
  for (int i = tid; i < N; i += 256)
    bound = fmax(bound, fabs(GK ? 0.0 : a[i]) + (i > 0 ? fabs(b[i - 1]) : 0.0) + (i + 1 < N ? fabs(b[i]) : 0.0));
  bound = wave_max(bound);
  if (lane == 0) redb[wave] = bound;
  __syncthreads();
  bound = fmax(fmax(redb[0], redb[1]), fmax(redb[2], redb[3]));
  const int ex = bound > 0.0 && isfinite(bound) ? ilogb(bound) : 0;
  const int steps = GK ? N / 2 : N - 1, padded = (steps + kB - 1) / kB * kB + kB;
  for (int i = tid; i < padded; i += 256) {
    // a padding step is decoupled and has no negative pivot (T), or one of two (GK)
    double x = GK ? 4.0 : 0.0, y = GK ? 0.0 : 16.0;
    if (GK) {
      if (i < steps) x = ldexp(b[2 * i], -ex);
      if (2 * i + 1 < N - 1) y = ldexp(b[2 * i + 1], -ex);
      y *= y;
    } else if (i < steps) {
      x = ldexp(b[i], -ex);
      y = ldexp(a[i + 1], -ex);
    }
    st[i] = make_double2(x * x, y);
  }
  __syncthreads();
  const int which = blockIdx.x * 4 + wave;
  if (which >= count) return;
  const double a0 = GK ? 0.0 : ldexp(a[0], -ex);
  bound = ldexp(bound, -ex);
  const int t = N - 1 - (i0 + which);
  double hi = bound + 4.0 * kEps * bound + 2.0 * kPivMin, lo = GK ? 0.0 : -hi;
  for (int pass = 0; pass < 64; ++pass) {
    const double sig = bisect_shift(lane, pass == 0, lo, hi);
    int cnt = 0;
    double u = a0 - sig;
    double2 nx[kB];
#pragma unroll
    for (int s = 0; s < kB; ++s) nx[s] = st[s];
    for (int i = 0; i < steps; i += kB) {
      double2 w[kB];  // this block's entries, read while the previous block ran
#pragma unroll
      for (int s = 0; s < kB; ++s) {
        w[s] = nx[s];
        nx[s] = st[i + kB + s];
      }
#pragma unroll
      for (int s = 0; s < kB; ++s) {
        if (GK) {
          const double m = fma(sig, u, w[s].x);
          // the odd pivot -m / u is negative when the signs agree
          const int su = __double2hiint(u), sx = su ^ __double2hiint(m);
          cnt += int(unsigned(su) >> 31) - int(unsigned(sx) >> 31);
          const double un = div_sub(w[s].y * u, m, sig);
          // an odd pivot of zero leads to an even one of the opposite sign beyond 1 / pivmin
          u = fabs(m) <= 0x1p-1000 ? fma(w[s].y, sx < 0 ? -kPivMinInv : kPivMinInv, -sig) : un;
        } else {
          cnt += u <= kPivMin;
          const double c = w[s].y - sig;
          const double un = -div_sub(w[s].x, u, c);
          u = fabs(u) <= kPivMin ? fma(w[s].x, kPivMinInv, c) : un;
        }
      }
    }
    // GK: one per pair from the signs, less the padding's one per pair
    cnt += GK ? steps : int(u <= kPivMin);
    const int k = __popcll(__ballot(cnt <= t));  // the shifts at or below lambda_t (a prefix)
    const double nlo = k > 0 ? __shfl(sig, k - 1, 64) : lo;
    const double nhi = k < 64 ? __shfl(sig, k, 64) : hi;
    lo = nlo;
    hi = nhi;
    if (hi - lo <= 2.0 * kEps * fmax(fabs(lo), fabs(hi)) + 2.0 * kPivMin) break;
  }
  if (lane == 0) lam[which] = ldexp(0.5 * (lo + hi), ex);
}

// ---------------------------------------------------------------- inverse iteration
__device__ inline double hash_unit(unsigned long long x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  x ^= x >> 31;
  return double(x >> 11) * (2.0 / 9007199254740992.0) - 1.0;  // [-1, 1)
}

// Inverse iteration, the method shared by the two kernels below: the eigenvector of T
// (diagonal a, zero when null; off-diagonal b) for lam[j], by `iters` solves with
// T - lam I factored once with partial pivoting (rows i and i + 1 swapped when |b_i|
// exceeds the current pivot, as LAPACK dlagtf; a pivot below eps ||T|| replaced by
// +-eps ||T||); the first right-hand side is a hashed pseudo-random vector, the later
// ones the normalised previous solution.  The result, or its even (part 0) / odd
// (part 1) entries, is normalised into column j of Y (len x m, row-major); a part whose
// norm is below 1e-3 of the vector's (a Golub-Kahan eigenvalue ~0, whose u and v parts
// are not determined) becomes a hashed pseudo-random vector, completed by the
// orthonormalisation.

// one elimination step of the factorisation (the values of the step's row i + 1 given):
// 1 / U(i, i), U(i, i + 1) / U(i, i), U(i, i + 2) / U(i, i), the multiplier, the swap
struct InvitStep {
  double u0, u1, u2, ml;
  int sw;
};
__device__ __forceinline__ InvitStep invit_factor_step(double& cd, double& cu, double nd, double nbv, double nu,
                                                       double tiny) {
  InvitStep o;
  const bool swp = fabs(cd) < fabs(nbv);
  const double num = swp ? cd : nbv, den = swp ? nbv : cd;
  o.ml = den != 0.0 ? num * recip(den) : 0.0;
  double u0 = den;
  o.u1 = swp ? nd : cu;
  o.u2 = swp ? nu : 0.0;
  o.sw = swp ? 1 : 0;
  const double ncd = swp ? cu - o.ml * nd : nd - o.ml * cu;
  cu = swp ? -o.ml * nu : nu;
  cd = ncd;
  if (fabs(u0) < tiny) u0 = u0 < 0.0 ? -tiny : tiny;
  o.u0 = recip(u0);
  o.u1 *= o.u0;
  o.u2 *= o.u0;
  return o;
}

// N > kInvitLdsMaxN (up to 4096): one wave per vector, the factors in global memory
// (per vector f0, f1, f2, the multipliers, the rhs / solution: 5 N doubles, and N swap
// flags), staged through the lanes 64 steps at a time: lane l loads (and stores) entry
// i0 + l of a block with one coalesced access per array, each step takes entry i0 + u
// as a broadcast from lane u (readlane), and the next block's loads are issued before
// the current block's steps, so their latency hides behind 64 steps of the chain.
// Passes are separated by a workgroup fence (the lanes read entries other lanes wrote).
constexpr int kGl = 64;
__global__ __launch_bounds__(64) void k_tri_invit_glb(const double* __restrict__ a, const double* __restrict__ b,
                                                      int N, const double* __restrict__ lam, int m,
                                                      double* __restrict__ fac, int* __restrict__ swf,
                                                      double* __restrict__ Y, int part, int iters, unsigned seed) {
  const int lane = threadIdx.x, j = blockIdx.x;
  if (j >= m) return;
  double tn = 0.0;
  for (int i = lane; i < N; i += 64)
    tn = fmax(tn, fabs(a ? a[i] : 0.0) + (i > 0 ? fabs(b[i - 1]) : 0.0) + (i + 1 < N ? fabs(b[i]) : 0.0));
  tn = wave_max(tn);
  const double tiny = kEps * fmax(tn, kSafeMin / kEps);
  double* const f0 = fac + size_t(j) * 5 * N;
  double* const f1 = f0 + N;
  double* const f2 = f1 + N;
  double* const fm = f2 + N;
  double* const zz = fm + N;
  int* const sw = swf + size_t(j) * N;
  const double lj = lam[j];
  const unsigned long long key = (unsigned long long)(seed) << 40 ^ (unsigned long long)(j) << 20;

  // factor T - lam I = P L U: steps i = 0 .. N - 2
  {
    double cd = (a ? a[0] : 0.0) - lj;
    double cu = N > 1 ? b[0] : 0.0;
    auto load = [&](int i0, double& nd, double& nb, double& nu) {
      const int i = i0 + lane;
      nd = i + 1 < N ? (a ? a[i + 1] : 0.0) - lj : 0.0;
      nb = i + 1 < N ? b[i] : 0.0;
      nu = i + 2 < N ? b[i + 1] : 0.0;
    };
    double nd, nb, nu;
    load(0, nd, nb, nu);
    for (int i0 = 0; i0 + 1 < N; i0 += kGl) {
      double nd2, nb2, nu2;
      load(i0 + kGl, nd2, nb2, nu2);
      const int steps = min(kGl, N - 1 - i0);
      double r0 = 0.0, r1 = 0.0, r2 = 0.0, r3 = 0.0;
      int r4 = 0;
      for (int u = 0; u < steps; ++u) {
        const InvitStep o = invit_factor_step(cd, cu, lane_bcast(nd, u), lane_bcast(nb, u), lane_bcast(nu, u), tiny);
        if (lane == u) {
          r0 = o.u0;
          r1 = o.u1;
          r2 = o.u2;
          r3 = o.ml;
          r4 = o.sw;
        }
      }
      if (lane < steps) {
        f0[i0 + lane] = r0;
        f1[i0 + lane] = r1;
        f2[i0 + lane] = r2;
        fm[i0 + lane] = r3;
        sw[i0 + lane] = r4;
      }
      nd = nd2;
      nb = nb2;
      nu = nu2;
    }
    if (fabs(cd) < tiny) cd = cd < 0.0 ? -tiny : tiny;
    if (lane == 0) {
      f0[N - 1] = recip(cd);
      f1[N - 1] = 0.0;
      f2[N - 1] = 0.0;
    }
  }
  for (int i = lane; i < N; i += 64) zz[i] = hash_unit(key + unsigned(i));
  __threadfence_block();

  double inv = 1.0, ne = 0.0, no = 0.0;
  for (int it = 0; it < iters; ++it) {
    const double sc = it == 0 ? 1.0 : inv;
    // eliminate the right-hand side in place (step i reads entry i + 1, writes entry i)
    double cy = zz[0] * sc;
    {
      auto load = [&](int i0, double& zb, double& mb, double& pb, int& sb) {
        const int i = i0 + lane;
        zb = i + 1 < N ? zz[i + 1] : 0.0;
        mb = i + 1 < N ? fm[i] : 0.0;
        pb = i + 1 < N ? f0[i] : 0.0;
        sb = i + 1 < N ? sw[i] : 0;
      };
      double zb, mb, pb;
      int sb;
      load(0, zb, mb, pb, sb);
      for (int i0 = 0; i0 + 1 < N; i0 += kGl) {
        double zb2, mb2, pb2;
        int sb2;
        load(i0 + kGl, zb2, mb2, pb2, sb2);
        const int steps = min(kGl, N - 1 - i0);
        double y = 0.0;
        for (int u = 0; u < steps; ++u) {
          const double ny = lane_bcast(zb, u) * sc, cm = lane_bcast(mb, u), cp = lane_bcast(pb, u);
          const int cs = __builtin_amdgcn_readlane(sb, u);
          const double yo = (cs ? ny : cy) * cp;
          if (lane == u) y = yo;
          cy = cs ? cy - cm * ny : ny - cm * cy;
        }
        if (lane < steps) zz[i0 + lane] = y;
        zb = zb2;
        mb = mb2;
        pb = pb2;
        sb = sb2;
      }
    }
    __threadfence_block();
    // back substitution in place, blocks of steps i0, i0 - 1, ... from the top
    double z1 = cy * f0[N - 1], z2 = 0.0;
    double nrm = z1 * z1;
    ne = ((N - 1) & 1) ? 0.0 : z1 * z1;
    no = ((N - 1) & 1) ? z1 * z1 : 0.0;
    if (lane == 0) zz[N - 1] = z1;
    {
      auto load = [&](int i0, double& g1, double& g2, double& yb) {
        const int i = i0 - lane;
        g1 = i >= 0 ? f1[i] : 0.0;
        g2 = i >= 0 ? f2[i] : 0.0;
        yb = i >= 0 ? zz[i] : 0.0;
      };
      double g1, g2, yb;
      load(N - 2, g1, g2, yb);
      for (int i0 = N - 2; i0 >= 0; i0 -= kGl) {
        double g1n, g2n, ybn;
        load(i0 - kGl, g1n, g2n, ybn);
        const int steps = min(kGl, i0 + 1);
        double zo = 0.0;
        for (int u = 0; u < steps; ++u) {
          const double zi = fma(-lane_bcast(g1, u), z1, fma(-lane_bcast(g2, u), z2, lane_bcast(yb, u)));
          if (lane == u) zo = zi;
          nrm += zi * zi;
          if ((i0 - u) & 1)
            no += zi * zi;
          else
            ne += zi * zi;
          z2 = z1;
          z1 = zi;
        }
        if (lane < steps) zz[i0 - lane] = zo;
        g1 = g1n;
        g2 = g2n;
        yb = ybn;
      }
    }
    __threadfence_block();
    inv = 1.0 / sqrt(nrm);
    ne *= inv * inv;
    no *= inv * inv;
  }
  const size_t M = size_t(m);
  if (part < 0) {
    for (int i = lane; i < N; i += 64) Y[size_t(i) * M + j] = zz[i] * inv;
    return;
  }
  const int len = part == 0 ? (N + 1) / 2 : N / 2;
  const double pn = part == 0 ? ne : no;
  if (pn >= 1e-6) {
    const double f = inv / sqrt(pn);
    for (int i = lane; i < len; i += 64) Y[size_t(i) * M + j] = zz[2 * i + part] * f;
  } else {
    for (int i = lane; i < len; i += 64) Y[size_t(i) * M + j] = hash_unit(key ^ 0x5555ull + unsigned(i));
  }
}

// The same inverse iteration with one wave per vector and the factors in LDS (for
// N <= kInvitLdsMaxN).  T - lam I is factored once (the same pivoting and tiny-pivot
// rule; the pivot choice is one select, so each step has one reciprocal on its
// dependency chain: the multiplier), and each of the `iters` passes only eliminates
// its right-hand side with the stored multipliers (scaling each eliminated entry by
// its pivot's reciprocal on the way) and back-substitutes with U's rows divided by
// their pivots beforehand, z_i = y'_i - U'(i, i + 2) z_{i+2} - U'(i, i + 1) z_{i+1}: one
// multiply-add per step on the dependency chain.  Every lane of the wave runs the same
// recurrence (the values are wave-uniform); lane 0 keeps 1 / U(i, i), U'(i, i + 1),
// U'(i, i + 2), the multiplier and the row swap in the wave's LDS slice, which the
// wave reads back as broadcasts.
// The steps go in blocks of kBlk with no bounds checks inside (T's off-diagonal is
// padded with a zero at N - 1), the block's LDS reads issued before its arithmetic,
// its stores after it; a tail of fewer than kBlk steps follows.  The right-hand side,
// its eliminated form and the solution share one LDS vector (each step reads entry
// i + 1 and writes entry i).
// W waves (vectors) per workgroup, so that the dynamic LDS stays within 64 KiB.
constexpr int kInvitLdsMaxN = 1024, kBlk = 8;

template <int kInvitWaves>
__global__ __launch_bounds__(64 * kInvitWaves) void k_tri_invit_lds(const double* __restrict__ a,
                                                                    const double* __restrict__ b, int N,
                                                                    const double* __restrict__ lam, int m,
                                                                    double* __restrict__ Y, int part, int iters,
                                                                    unsigned seed) {
  extern __shared__ double sm[];
  double* const as = sm;                // N when a is given
  double* const bs = sm + (a ? N : 0);  // N: b, then a zero at N - 1
  __shared__ double red[kInvitWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double tn = 0.0;
  for (int i = tid; i < N; i += 64 * kInvitWaves) {
    const double ai = a ? a[i] : 0.0;
    if (a) as[i] = ai;
    bs[i] = i + 1 < N ? b[i] : 0.0;
    tn = fmax(tn, fabs(ai) + (i > 0 ? fabs(b[i - 1]) : 0.0) + (i + 1 < N ? fabs(b[i]) : 0.0));
  }
  tn = wave_max(tn);
  if (lane == 0) red[wave] = tn;
  __syncthreads();
  tn = red[0];
  for (int w = 1; w < kInvitWaves; ++w) tn = fmax(tn, red[w]);
  const int j = blockIdx.x * kInvitWaves + wave;
  if (j >= m) return;
  double* const f0 = sm + (a ? N : 0) + N + size_t(wave) * 5 * N;  // 1 / U(i, i)
  double* const f1 = f0 + N;                                        // U(i, i + 1) / U(i, i)
  double* const f2 = f1 + N;                                        // U(i, i + 2) / U(i, i)
  double* const fm = f2 + N;                                        // multiplier
  double* const zz = fm + N;                                        // rhs / solution
  int* const sw = reinterpret_cast<int*>(sm + (a ? N : 0) + N + size_t(kInvitWaves) * 5 * N) + size_t(wave) * N;
  const double tiny = kEps * fmax(tn, kSafeMin / kEps);
  const double lj = lam[j];
  const unsigned long long key = (unsigned long long)(seed) << 40 ^ (unsigned long long)(j) << 20;
  const int nfull = (N - 1) / kBlk * kBlk;  // steps 0 .. nfull - 1 in full blocks

  // factor T - lam I = P L U (steps i = 0 .. N - 2 eliminate row i + 1)
  {
    double cd = (a ? as[0] : 0.0) - lj;
    double cu = bs[0];
    for (int i0 = 0; i0 < nfull; i0 += kBlk) {
      double nd[kBlk], nb[kBlk + 1];
#pragma unroll
      for (int u = 0; u < kBlk; ++u) nd[u] = (a ? as[i0 + u + 1] : 0.0) - lj;
#pragma unroll
      for (int u = 0; u <= kBlk; ++u) nb[u] = bs[i0 + u];
      InvitStep o[kBlk];
#pragma unroll
      for (int u = 0; u < kBlk; ++u) o[u] = invit_factor_step(cd, cu, nd[u], nb[u], nb[u + 1], tiny);
      if (lane == 0) {
#pragma unroll
        for (int u = 0; u < kBlk; ++u) {
          f0[i0 + u] = o[u].u0;
          f1[i0 + u] = o[u].u1;
          f2[i0 + u] = o[u].u2;
          fm[i0 + u] = o[u].ml;
          sw[i0 + u] = o[u].sw;
        }
      }
    }
    for (int i = nfull; i + 1 < N; ++i) {
      const InvitStep o = invit_factor_step(cd, cu, (a ? as[i + 1] : 0.0) - lj, bs[i], bs[i + 1], tiny);
      if (lane == 0) {
        f0[i] = o.u0;
        f1[i] = o.u1;
        f2[i] = o.u2;
        fm[i] = o.ml;
        sw[i] = o.sw;
      }
    }
    if (fabs(cd) < tiny) cd = cd < 0.0 ? -tiny : tiny;
    if (lane == 0) {
      f0[N - 1] = recip(cd);
      f1[N - 1] = 0.0;
      f2[N - 1] = 0.0;
    }
  }
  // the first right-hand side: a hashed pseudo-random vector
  for (int i = lane; i < N; i += 64) zz[i] = hash_unit(key + unsigned(i));
  wave_sync_lds();

  double inv = 1.0, ne = 0.0, no = 0.0;
  for (int it = 0; it < iters; ++it) {
    const double sc = it == 0 ? 1.0 : inv;
    // eliminate the right-hand side (sc * zz) with the stored multipliers, in place
    double cy = zz[0] * sc;
    for (int i0 = 0; i0 < nfull; i0 += kBlk) {
      double rhs[kBlk], cm[kBlk], cp[kBlk], yo[kBlk];
      int cs[kBlk];
#pragma unroll
      for (int u = 0; u < kBlk; ++u) {
        rhs[u] = zz[i0 + u + 1] * sc;
        cm[u] = fm[i0 + u];
        cs[u] = sw[i0 + u];
        cp[u] = f0[i0 + u];
      }
#pragma unroll
      for (int u = 0; u < kBlk; ++u) {
        yo[u] = (cs[u] ? rhs[u] : cy) * cp[u];
        cy = cs[u] ? cy - cm[u] * rhs[u] : rhs[u] - cm[u] * cy;
      }
      wave_sync_lds();  // the block's reads of zz before lane 0 overwrites entries
      if (lane == 0) {
#pragma unroll
        for (int u = 0; u < kBlk; ++u) zz[i0 + u] = yo[u];
      }
    }
    for (int i = nfull; i + 1 < N; ++i) {
      const double ny = zz[i + 1] * sc;
      const double y = (sw[i] ? ny : cy) * f0[i];
      cy = sw[i] ? cy - fm[i] * ny : ny - fm[i] * cy;
      wave_sync_lds();
      if (lane == 0) zz[i] = y;
    }
    wave_sync_lds();
    // back substitution, in place: steps i = N - 2 .. 0, full blocks from the top
    double z1 = cy * f0[N - 1], z2 = 0.0;
    double nrm = z1 * z1;
    ne = ((N - 1) & 1) ? 0.0 : z1 * z1;
    no = ((N - 1) & 1) ? z1 * z1 : 0.0;
    if (lane == 0) zz[N - 1] = z1;
    int i0 = N - 2;
    for (; i0 >= kBlk - 1; i0 -= kBlk) {
      double c1[kBlk], c2[kBlk], cy2[kBlk], zo[kBlk];
#pragma unroll
      for (int u = 0; u < kBlk; ++u) {
        c1[u] = f1[i0 - u];
        c2[u] = f2[i0 - u];
        cy2[u] = zz[i0 - u];
      }
      double sq[2] = {0.0, 0.0};  // squares of the steps u even / odd
#pragma unroll
      for (int u = 0; u < kBlk; ++u) {
        const double zi = fma(-c1[u], z1, fma(-c2[u], z2, cy2[u]));
        zo[u] = zi;
        sq[u & 1] += zi * zi;
        z2 = z1;
        z1 = zi;
      }
      nrm += sq[0] + sq[1];
      if (i0 & 1) {
        no += sq[0];
        ne += sq[1];
      } else {
        ne += sq[0];
        no += sq[1];
      }
      wave_sync_lds();  // the block's reads of zz before lane 0 overwrites them
      if (lane == 0) {
#pragma unroll
        for (int u = 0; u < kBlk; ++u) zz[i0 - u] = zo[u];
      }
    }
    for (; i0 >= 0; --i0) {
      const double zi = fma(-f1[i0], z1, fma(-f2[i0], z2, zz[i0]));
      nrm += zi * zi;
      if (i0 & 1)
        no += zi * zi;
      else
        ne += zi * zi;
      z2 = z1;
      z1 = zi;
      wave_sync_lds();
      if (lane == 0) zz[i0] = zi;
    }
    wave_sync_lds();  // the solution's stores before the next pass reads it
    inv = 1.0 / sqrt(nrm);
    ne *= inv * inv;
    no *= inv * inv;
  }
  const size_t M = size_t(m);
  if (part < 0) {
    for (int i = lane; i < N; i += 64) Y[size_t(i) * M + j] = zz[i] * inv;
    return;
  }
  const int len = part == 0 ? (N + 1) / 2 : N / 2;
  const double pn = part == 0 ? ne : no;
  if (pn >= 1e-6) {
    const double f = inv / sqrt(pn);
    for (int i = lane; i < len; i += 64) Y[size_t(i) * M + j] = zz[2 * i + part] * f;
  } else {
    for (int i = lane; i < len; i += 64) Y[size_t(i) * M + j] = hash_unit(key ^ 0x5555ull + unsigned(i));
  }
}

// ---------------------------------------------------------------- CholQR pieces
constexpr int kCholMax = 64;

// G (b x b, row stride ldg) = R^T R with R upper triangular; writes R^{-1} (b x b,
// row-major, zero below the diagonal).  One wave; lane c works on column c of G, held
// in LDS (consecutive lanes, consecutive addresses) and padded to 64 x 64 with the
// identity (whose factor and inverse are the identity again).  Cholesky by rows: step
// j takes the pivot (a pivot that is not positive and finite raises *fail and is
// replaced by 1, so the kernel still ends), every lane scales its entry of row j
// (R(j, c) = G'(j, c) / R(j, j)) in place, then updates its column with that row
// read as broadcasts: G'(i, c) -= R(j, i) R(j, c), i > j.  The inverse by back
// substitution, lane c solving for column c of R^{-1}: X(i, c) = (delta_ic -
// sum_{t > i} R(i, t) X(t, c)) / R(i, i) (zero for i > c by construction).  The
// entries below R's diagonal are never read.  A G within 1e-8 of the identity takes
// the first-order inverse instead (below).
__global__ __launch_bounds__(64) void k_chol_inv(const double* __restrict__ Gm, int b, int ldg,
                                                 double* __restrict__ Rinv, unsigned* fail) {
  __shared__ double A[kCholMax][kCholMax];
  __shared__ double X[kCholMax][kCholMax];
  __shared__ double Rj[kCholMax];  // row j of R, a separate array: the update's reads of it
                                   // cannot alias its writes to A, so they are issued together
  const int c = threadIdx.x;
  const int cc = c < b ? c : 0;
  for (int i = 0; i < kCholMax; ++i) {
    const double g = Gm[size_t(i < b ? i : 0) * ldg + cc];  // clamped address, every lane loads
    A[i][c] = (i < b && c < b) ? g : (i == c ? 1.0 : 0.0);
  }
  wave_sync_lds();
  // G = I + E with max |E| <= 1e-8 (the second CholQR pass, and a first one whose
  // vectors are already orthogonal to that level): R = I + F + O(E^2) with F the upper
  // triangle of E (halved on the diagonal), R^{-1} = I - F + O(E^2), exact to 1e-16.
  double em = 0.0;
  for (int i = 0; i < b; ++i) em = fmax(em, fabs(A[i][c] - (i == c ? 1.0 : 0.0)));
  em = wave_max(c < b ? em : 0.0);
  if (em <= 1e-8) {
    if (c < b)
      for (int i = 0; i < b; ++i)
        Rinv[size_t(i) * b + c] = i < c ? -A[i][c] : (i == c ? 1.0 - 0.5 * (A[i][i] - 1.0) : 0.0);
    return;
  }
  bool bad = false;
  for (int j = 0; j < kCholMax; ++j) {
    double pv = A[j][j];
    if (!(pv > 0.0) || !isfinite(pv)) {
      bad = true;
      pv = 1.0;
    }
    const double rjj = sqrt(pv);
    const double r = c > j ? A[j][c] / rjj : (c == j ? rjj : 0.0);
    A[j][c] = r;
    Rj[c] = r;
    wave_sync_lds();
#pragma unroll 8
    for (int i = j + 1; i < kCholMax; ++i) A[i][c] -= Rj[i] * r;
    wave_sync_lds();
  }
  if (bad && c == 0) atomicOr(fail, 1u);
  for (int i = kCholMax - 1; i >= 0; --i) {
    double acc = (i == c) ? 1.0 : 0.0;
#pragma unroll 4
    for (int t = i + 1; t < kCholMax; ++t) acc -= A[i][t] * X[t][c];
    X[i][c] = acc / A[i][i];
    wave_sync_lds();
  }
  if (c < b)
    for (int i = 0; i < b; ++i) Rinv[size_t(i) * b + c] = X[i][c];
}

// Y[:, c0 + c] = T[:, c] (T: len x bw row-major; Y row stride ldy)
__global__ void k_put_cols(const double* __restrict__ T, int64_t len, int bw, double* __restrict__ Y, int64_t ldy,
                           int c0) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= len * bw) return;
  const int64_t i = t / bw;
  const int c = int(t % bw);
  Y[i * ldy + c0 + c] = T[t];
}

// ---------------------------------------------------------------- reflector rows
// Vt (s x r): row j = u_j (zero before j, 1 at j, X(i, j) below), zero when tau_L[j] == 0
__global__ void k_build_vt_left(const double* __restrict__ X, int r, int s, const double* __restrict__ tau,
                                double* __restrict__ Vt) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(s) * r) return;
  const int64_t j = t / r, i = t % r;
  double v = 0.0;
  if (tau[j] != 0.0) v = i < j ? 0.0 : (i == j ? 1.0 : X[i * s + j]);
  Vt[t] = v;
}

// Vt ((s - 1) x s): row j = v_j (zero up to j, 1 at j + 1, X(j, c) beyond), zero when tau_R[j] == 0
__global__ void k_build_vt_right(const double* __restrict__ X, int s, const double* __restrict__ tau,
                                 double* __restrict__ Vt) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= int64_t(s - 1) * s) return;
  const int64_t j = t / s, c = t % s;
  double v = 0.0;
  if (tau[j] != 0.0) v = c <= j ? 0.0 : (c == j + 1 ? 1.0 : X[j * s + c]);
  Vt[t] = v;
}

// Golub-Kahan off-diagonal: gk[2 i] = d_i, gk[2 i + 1] = e_i
__global__ void k_gk_offdiag(const double* __restrict__ d, const double* __restrict__ e, int s,
                             double* __restrict__ gk) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 2 * s - 1) return;
  gk[t] = (t & 1) ? e[t >> 1] : d[t >> 1];
}

inline unsigned nblk(int64_t n, int t = 256) { return unsigned((n + t - 1) / t); }

GemmDesc gd(int64_t M, int64_t N, int64_t K, bool ta, bool tb, int64_t lda, int64_t ldb, int64_t ldc) {
  GemmDesc g{};
  g.M = M;
  g.N = N;
  g.K = K;
  g.transA = ta;
  g.transB = tb;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.batch = 1;
  return g;
}

}  // namespace

void gk_offdiag(nsmi_ctx* ctx, const double* d, const double* e, int s, double* gk) {
  if (s < 1) return;
  hipLaunchKernelGGL(k_gk_offdiag, dim3(nblk(2 * s - 1)), dim3(256), 0, ctx->stream, d, e, s, gk);
  NSMI_LAUNCH_CHECK();
}

void tri_bisect(nsmi_ctx* ctx, const double* a, const double* b, int N, int i0, int count, double* lam) {
  require(N >= 1 && N <= kTriSolveMaxN, "tridiagonal eigensolver: size outside [1, 4096]");
  require(i0 >= 0 && count >= 0 && i0 + count <= N, "tridiagonal eigensolver: bad eigenvalue range");
  require(a || (N % 2 == 0 && i0 + count <= N / 2), "tridiagonal eigensolver: Golub-Kahan range");
  if (count == 0) return;
  const int steps = a ? N - 1 : N / 2;
  const size_t shm = bisect_lds(steps);
  require(shm <= kBisectLds, "tridiagonal eigensolver: order above what its LDS holds");
  ProfScope ps(ctx, NSMI_K_FACT_SOLVE, 0.0, 0.0);
  const dim3 grid(unsigned((count + 3) / 4)), block(256);
  if (a)
    hipLaunchKernelGGL(k_tri_bisect<false>, grid, block, shm, ctx->stream, a, b, N, i0, count, lam);
  else
    hipLaunchKernelGGL(k_tri_bisect<true>, grid, block, shm, ctx->stream, a, b, N, i0, count, lam);
  NSMI_LAUNCH_CHECK();
}

void tri_invit(nsmi_ctx* ctx, const double* a, const double* b, int N, const double* lam, int m, double* Y, int part) {
  require(N >= 1 && N <= kTriSolveMaxN, "tridiagonal eigensolver: size outside [1, 4096]");
  if (m == 0) return;
  const size_t shm = sizeof(double) * (size_t(a ? N : 0) + size_t(std::max(N - 1, 1)));
  ProfScope ps(ctx, NSMI_K_FACT_SOLVE, 0.0, 0.0);
  if (N <= kInvitLdsMaxN) {
    // dynamic LDS: T (<= 16 KiB, the off-diagonal padded to N) + 5 N doubles and N ints
    // per wave (<= 44 KiB)
    const size_t shm_t = sizeof(double) * (size_t(a ? N : 0) + size_t(N));
    if (N <= 384) {
      const size_t shm_w = shm_t + (sizeof(double) * 5 + sizeof(int)) * size_t(N) * 2;
      hipLaunchKernelGGL(k_tri_invit_lds<2>, dim3(unsigned((m + 1) / 2)), dim3(128), shm_w, ctx->stream, a, b, N,
                         lam, m, Y, part, 3, 0x2545u);
    } else {
      const size_t shm_w = shm_t + (sizeof(double) * 5 + sizeof(int)) * size_t(N);
      hipLaunchKernelGGL(k_tri_invit_lds<1>, dim3(unsigned(m)), dim3(64), shm_w, ctx->stream, a, b, N, lam, m, Y,
                         part, 3, 0x2545u);
    }
    NSMI_LAUNCH_CHECK();
    return;
  }
  Scratch fac(ctx, sizeof(double) * 5 * size_t(N) * m), swf(ctx, sizeof(int) * size_t(N) * m);
  hipLaunchKernelGGL(k_tri_invit_glb, dim3(unsigned(m)), dim3(64), 0, ctx->stream, a, b, N, lam, m, fac.as<double>(),
                     swf.as<int>(), Y, part, 3, 0x2545u);
  NSMI_LAUNCH_CHECK();
}

// Columns of Y (len x k, row-major) made orthonormal in order: blocks of up to 64
// columns, each projected against the finished columns (classical Gram-Schmidt) and
// orthonormalised by CholQR, twice.  *fail (device) is raised when a block is not
// numerically independent.
void orthonormalize_cols(nsmi_ctx* ctx, double* Y, int64_t len, int k, unsigned* fail) {
  if (k == 0) return;
  require(k <= len, "orthonormalize: more vectors than their length");
  Scratch Gs(ctx, sizeof(double) * kCholMax * kCholMax), Ri(ctx, sizeof(double) * kCholMax * kCholMax),
      T(ctx, sizeof(double) * size_t(len) * kCholMax), Cp(ctx, sizeof(double) * size_t(k) * kCholMax);
  ProfScope ps(ctx, NSMI_K_FACT_GEMM, 4.0 * double(len) * k * k, 0.0);
  for (int c0 = 0; c0 < k; c0 += kCholMax) {
    const int bw = std::min(kCholMax, k - c0);
    for (int pass = 0; pass < 2; ++pass) {
      if (c0 > 0) {
        // C = Y[:, :c0]^T Y[:, c0:c0+bw];  Y[:, c0:] -= Y[:, :c0] C
        gemm_f64(ctx, gd(c0, bw, len, true, false, k, k, bw), 1.0, Y, Y + c0, 0.0, Cp.as<double>(), kRoleFact);
        gemm_f64(ctx, gd(len, bw, c0, false, false, k, bw, k), -1.0, Y, Cp.as<double>(), 1.0, Y + c0, kRoleFact);
      }
      gemm_f64(ctx, gd(bw, bw, len, true, false, k, k, bw), 1.0, Y + c0, Y + c0, 0.0, Gs.as<double>(), kRoleFact);
      hipLaunchKernelGGL(k_chol_inv, dim3(1), dim3(64), 0, ctx->stream, Gs.as<double>(), bw, bw, Ri.as<double>(),
                         fail);
      NSMI_LAUNCH_CHECK();
      gemm_f64(ctx, gd(len, bw, bw, false, false, k, bw, bw), 1.0, Y + c0, Ri.as<double>(), 0.0, T.as<double>(),
               kRoleFact);
      hipLaunchKernelGGL(k_put_cols, dim3(nblk(len * bw)), dim3(256), 0, ctx->stream, T.as<double>(), len, bw, Y,
                         int64_t(k), c0);
      NSMI_LAUNCH_CHECK();
    }
  }
}

void bidiag_reflectors_left(nsmi_ctx* ctx, const double* X, int r, int s, const double* tau, double* Vt) {
  hipLaunchKernelGGL(k_build_vt_left, dim3(nblk(int64_t(s) * r)), dim3(256), 0, ctx->stream, X, r, s, tau, Vt);
  NSMI_LAUNCH_CHECK();
}

void bidiag_reflectors_right(nsmi_ctx* ctx, const double* X, int s, const double* tau, double* Vt) {
  if (s < 2) return;
  hipLaunchKernelGGL(k_build_vt_right, dim3(nblk(int64_t(s - 1) * s)), dim3(256), 0, ctx->stream, X, s, tau, Vt);
  NSMI_LAUNCH_CHECK();
}

}  // namespace nsmi
