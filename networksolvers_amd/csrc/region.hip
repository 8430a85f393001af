// Region-step contractions: two-site / one-site effective Hamiltonian apply,
// environment updates, theta formation and the Lanczos eigensolver.
//
// H_eff apply (operator_map.jl:3-10, order ((L.theta).W1W2).R):
//   GEMM1  T1[(a' w), (s1 s2 b)] = L[(a' w), a] . theta[a, (s1 s2 b)]          (NN)
//   MIX    T3[a', (s1' s2' v), b] = sum_{w s1 s2} W12[(s1' s2' v), (w s1 s2)] T1 (per a', b)
//   GEMM2  y[(a' s1' s2'), b'] = T3[(a' s1' s2'), (v b)] . R[b', (v b)]^T        (NT)
// W12 = W1 . W2 over the shared MPO bond is formed once per operator on the host.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>

#include "internal.h"

using namespace nsmi;

struct nsmi_heff {
  const nsmi_tensor* L = nullptr;
  const nsmi_tensor* R = nullptr;
  int precision = NSMI_PREC_FP64;
  int nsite = 2;
  bool cplx = false;  // ComplexF64 environments and states (real MPO)
  int64_t cl = 0, cr = 0, D0 = 0, D2 = 0, dphys = 0;  // dphys = d1*d2 (2-site) or d
  int P = 0, Q = 0;
  double* Mx = nullptr;  // device P x Q mixing matrix
  void* T1 = nullptr;    // GEMM1 output
  void* T3 = nullptr;    // mixing output
  float* L32 = nullptr;
  float* R32 = nullptr;
  // BF16 forms: operand planes (K padded to 32), per-apply workspace
  uint16_t *Lhi = nullptr, *Llo = nullptr, *Rhi = nullptr, *Rlo = nullptr;
  uint16_t *xThi = nullptr, *xTlo = nullptr, *T3hi = nullptr, *T3lo = nullptr;
  float* T1f = nullptr;
  int64_t Kp1 = 0, Kp2 = 0;
  double flops_gemm1 = 0, flops_gemm2 = 0, flops_mix = 0;
  int64_t n = 0;  // elements of theta
  nsmi::NetProgram* net = nullptr;  // tree regions: a general contraction program instead of the fixed form
  nsmi::BsProgram* bs = nullptr;    // quantum-number regions: a block program
};

namespace nsmi {

namespace {

constexpr int kMixThreads = 256;

// Y[o, p, i] = sum_q Mx[p, q] X[o, q, i]: one thread per (o, i) holds the Q inputs in registers;
// blockIdx.z selects a chunk of PC outputs, so small operators still fill the device.  The
// coefficient addresses are wave-uniform (scalar loads), and four outputs accumulate at a time
// as independent chains.  Every output sums q in ascending order, whatever the chunking.
template <typename TI, typename TO, int QMAX>
__global__ __launch_bounds__(kMixThreads) void k_mix(const TI* __restrict__ X, TO* __restrict__ Y,
                                                     const double* __restrict__ Mx, int64_t O, int P, int Q,
                                                     int64_t I, int PC) {
  const int64_t i = int64_t(blockIdx.x) * kMixThreads + threadIdx.x;
  if (i >= I) return;
  const int pb = int(blockIdx.z) * PC;
  const int pe = min(P, pb + PC);
  for (int64_t o = blockIdx.y; o < O; o += gridDim.y) {
    const TI* xo = X + o * Q * I + i;
    TO* yo = Y + o * int64_t(P) * I + i;
    double x[QMAX];
#pragma unroll
    for (int q = 0; q < QMAX; ++q) x[q] = (q < Q) ? double(xo[int64_t(q) * I]) : 0.0;
    for (int p = pb; p < pe; p += 4) {
      const double* m0 = Mx + int64_t(p) * Q;
      const double* m1 = Mx + int64_t(min(p + 1, pe - 1)) * Q;
      const double* m2 = Mx + int64_t(min(p + 2, pe - 1)) * Q;
      const double* m3 = Mx + int64_t(min(p + 3, pe - 1)) * Q;
      double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll
      for (int q = 0; q < QMAX; ++q)
        if (q < Q) {
          a0 += m0[q] * x[q];
          a1 += m1[q] * x[q];
          a2 += m2[q] * x[q];
          a3 += m3[q] * x[q];
        }
      yo[int64_t(p) * I] = TO(a0);
      if (p + 1 < pe) yo[int64_t(p + 1) * I] = TO(a1);
      if (p + 2 < pe) yo[int64_t(p + 2) * I] = TO(a2);
      if (p + 3 < pe) yo[int64_t(p + 3) * I] = TO(a3);
    }
  }
}

template <typename TI, typename TO>
void mix_launch(nsmi_ctx* ctx, const TI* X, TO* Y, const double* Mx, int64_t O, int P, int Q, int64_t I,
                int cls) {
  require(P >= 1 && Q >= 1 && P <= 64 && Q <= 64, "mix: P, Q must be in [1, 64]");
  if (O == 0 || I == 0) return;
  ProfScope ps(ctx, cls, 2.0 * double(O) * double(I) * P * Q,
               double(O) * double(I) * (P * sizeof(TO) + Q * sizeof(TI)));
  // split the outputs into chunks of at least four until the grid holds ~2048 waves
  const int64_t oy = std::min<int64_t>(O, 65535);
  const int64_t waves = oy * ((I + 63) / 64);
  const int64_t want = std::max<int64_t>(1, (2048 + waves - 1) / waves);
  const int split = int(std::min<int64_t>((P + 3) / 4, want));
  const int PC = (P + split - 1) / split;
  const unsigned gz = unsigned((P + PC - 1) / PC);
  dim3 grid(unsigned((I + kMixThreads - 1) / kMixThreads), unsigned(oy), gz);
  if (Q <= 8)
    hipLaunchKernelGGL((k_mix<TI, TO, 8>), grid, dim3(kMixThreads), 0, ctx->stream, X, Y, Mx, O, P, Q, I, PC);
  else if (Q <= 16)
    hipLaunchKernelGGL((k_mix<TI, TO, 16>), grid, dim3(kMixThreads), 0, ctx->stream, X, Y, Mx, O, P, Q, I, PC);
  else if (Q <= 32)
    hipLaunchKernelGGL((k_mix<TI, TO, 32>), grid, dim3(kMixThreads), 0, ctx->stream, X, Y, Mx, O, P, Q, I, PC);
  else
    hipLaunchKernelGGL((k_mix<TI, TO, 64>), grid, dim3(kMixThreads), 0, ctx->stream, X, Y, Mx, O, P, Q, I, PC);
  NSMI_LAUNCH_CHECK();
}

GemmDesc desc(int64_t M, int64_t N, int64_t K, bool ta, bool tb) {
  GemmDesc g{};
  g.M = M;
  g.N = N;
  g.K = K;
  g.transA = ta;
  g.transB = tb;
  g.lda = ta ? M : K;
  g.ldb = tb ? K : N;
  g.ldc = N;
  g.batch = 1;
  return g;
}

const double* dptr(const nsmi_tensor* t) { return static_cast<const double*>(t->data); }
double* dptr(nsmi_tensor* t) { return static_cast<double*>(t->data); }

void check_f64(const nsmi_tensor* t, const char* what) {
  require(t != nullptr, std::string(what) + " is null");
  if (t->dtype != NSMI_F64) fail(NSMI_ERR_UNSUPPORTED, std::string(what) + ": only F64 tensors are served");
}

size_t prec_elt(int prec) { return prec == NSMI_PREC_FP64 ? 8 : 4; }

// Mx[(s1' s2' v), (w s1 s2)] = sum_u W1[w,u,s1',s1] W2[u,v,s2',s2]
__global__ void k_build_w12(const double* __restrict__ W1, const double* __restrict__ W2, double* __restrict__ Mx,
                            int D0, int Dm, int D2, int d1, int d2) {
  const int P = d1 * d2 * D2, Q = D0 * d1 * d2;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= P * Q) return;
  const int p = t / Q, q = t % Q;
  const int v = p % D2, a2 = (p / D2) % d2, a1 = p / (D2 * d2);
  const int b2 = q % d2, b1 = (q / d2) % d1, w = q / (d1 * d2);
  double acc = 0.0;
  for (int u = 0; u < Dm; ++u)
    acc += W1[((w * Dm + u) * d1 + a1) * d1 + b1] * W2[((u * D2 + v) * d2 + a2) * d2 + b2];
  Mx[t] = acc;
}

// mode 0: Mx[(s' v), (w s)] = W[w, v, s', s]     (H_eff 1-site, left environment)
// mode 1: Mx[(w s), (s' v)] = W[w, v, s', s]     (right environment)
__global__ void k_build_w1(const double* __restrict__ W, double* __restrict__ Mx, int Dl, int Dr, int d, int mode) {
  const int n = Dl * Dr * d * d;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int s = t % d, sp = (t / d) % d, v = (t / (d * d)) % Dr, w = t / (d * d * Dr);
  const double x = W[t];
  if (mode == 0) {
    const int Q = Dl * d;
    Mx[(sp * Dr + v) * Q + (w * d + s)] = x;
  } else {
    const int Q = d * Dr;
    Mx[(w * d + s) * Q + (sp * Dr + v)] = x;
  }
}

// round-to-nearest-even FP32 -> BF16 bits (finite inputs)
__device__ inline uint16_t bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}
__device__ inline float bf16_f32(uint16_t h) { return __uint_as_float(uint32_t(h) << 16); }

// hi = bf16(v), lo = bf16(v - hi) for every (r, k < Kp); zero beyond K.
__global__ void k_split_rows(const double* __restrict__ X, int64_t rows, int64_t K, int64_t Kp,
                             uint16_t* __restrict__ hi, uint16_t* __restrict__ lo) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= rows * Kp) return;
  const int64_t r = t / Kp, k = t % Kp;
  const double v = k < K ? X[r * K + k] : 0.0;
  const uint16_t h = bf16_rne(float(v));
  hi[t] = h;
  if (lo) lo[t] = bf16_rne(float(v - double(bf16_f32(h))));
}

// transposing split: source X is K x rows (row stride rows); out[r][k] = X[k][r]
__global__ void k_split_transpose(const double* __restrict__ X, int64_t rows, int64_t K, int64_t Kp,
                                  uint16_t* __restrict__ hi, uint16_t* __restrict__ lo) {
  __shared__ double tile[32][33];
  const int64_t r0 = int64_t(blockIdx.x) * 32, k0 = int64_t(blockIdx.y) * 32;
  for (int j = threadIdx.y; j < 32; j += blockDim.y) {
    const int64_t k = k0 + j, r = r0 + threadIdx.x;
    tile[j][threadIdx.x] = (k < K && r < rows) ? X[k * rows + r] : 0.0;
  }
  __syncthreads();
  for (int j = threadIdx.y; j < 32; j += blockDim.y) {
    const int64_t r = r0 + j, k = k0 + threadIdx.x;
    if (r < rows && k < Kp) {
      const double v = tile[threadIdx.x][j];
      const uint16_t h = bf16_rne(float(v));
      hi[r * Kp + k] = h;
      if (lo) lo[r * Kp + k] = bf16_rne(float(v - double(bf16_f32(h))));
    }
  }
}

// H_eff mixing written as GEMM2's bf16 operand:
// Y[(o*S + p/D2), (p%D2)*I + i] = sum_q Mx[p][q] X[o][q][i],  S = P / D2,
// for the PC outputs p of blockIdx.z (a multiple of 4).  Mx is padded with zeros to QMAX columns
// and four rows in LDS, so the sums have no branches, four of them run side by side and
// their coefficients come as 16-byte broadcasts: with a test of q < Q at every term and one
// sum at a time the kernel waited for each LDS read (613 x 487, d = 2: 31 -> 16 us, 48 MB; the
// whole apply at 400 x 300, d = 3: 273 -> 108 us, at 8 x 8: 29 -> 11). Two columns per thread, to
// share those reads, gained nothing.
template <int QMAX>
__global__ __launch_bounds__(256) void k_mix_bf16_rows(const float* __restrict__ X, uint16_t* __restrict__ Yhi,
                                                       uint16_t* __restrict__ Ylo, const double* __restrict__ Mx,
                                                       int64_t O, int P, int Q, int64_t I, int D2, int64_t Kp, int PC) {
  __shared__ __align__(16) float sM[64 * QMAX];
  const int pb = blockIdx.z * PC, pe = min(pb + PC, P), PR = (pe - pb + 3) & ~3;
  for (int t = threadIdx.x; t < PR * QMAX; t += 256) {
    const int p = pb + t / QMAX, q = t % QMAX;
    sM[t] = p < pe && q < Q ? float(Mx[p * Q + q]) : 0.f;
  }
  __syncthreads();
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= I) return;
  const int S = P / D2;
  for (int64_t o = blockIdx.y; o < O; o += gridDim.y) {
    const float* xo = X + o * Q * I + i;
    float x[QMAX];
#pragma unroll
    for (int q = 0; q < QMAX; ++q) x[q] = (q < Q) ? xo[int64_t(q) * I] : 0.f;
    for (int p = pb; p < pe; p += 4) {
      const float* m = sM + (p - pb) * QMAX;
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < QMAX; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] += m[j * QMAX + q] * x[q];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (p + j < pe) {
          const int64_t idx = (o * S + (p + j) / D2) * Kp + int64_t((p + j) % D2) * I + i;
          const uint16_t h = bf16_rne(acc[j]);
          Yhi[idx] = h;
          if (Ylo) Ylo[idx] = bf16_rne(acc[j] - bf16_f32(h));
        }
    }
  }
}

void build_w1(nsmi_ctx* ctx, const double* W, double* Mx, int Dl, int Dr, int d, int mode) {
  const int n = Dl * Dr * d * d;
  hipLaunchKernelGGL(k_build_w1, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, W, Mx, Dl, Dr, d, mode);
  NSMI_LAUNCH_CHECK();
}

}  // namespace

void mix_f64(nsmi_ctx* ctx, const double* X, double* Y, const double* Mx, int64_t O, int P, int Q, int64_t I,
             int cls) {
  mix_launch<double, double>(ctx, X, Y, Mx, O, P, Q, I, cls);
}
void mix_f32(nsmi_ctx* ctx, const float* X, float* Y, const double* Mx, int64_t O, int P, int Q, int64_t I,
             int cls) {
  mix_launch<float, float>(ctx, X, Y, Mx, O, P, Q, I, cls);
}

void split_bf16_pad(nsmi_ctx* ctx, const double* X, int64_t rows, int64_t K, int64_t Kp, uint16_t* hi, uint16_t* lo,
                    int transpose) {
  if (rows == 0 || Kp == 0) return;
  if (!transpose) {
    const int64_t n = rows * Kp;
    hipLaunchKernelGGL(k_split_rows, dim3(unsigned((n + 255) / 256)), dim3(256), 0, ctx->stream, X, rows, K, Kp, hi, lo);
  } else {
    dim3 grid(unsigned((rows + 31) / 32), unsigned((Kp + 31) / 32));
    hipLaunchKernelGGL(k_split_transpose, grid, dim3(32, 8), 0, ctx->stream, X, rows, K, Kp, hi, lo);
  }
  NSMI_LAUNCH_CHECK();
}

void mix_f32_to_bf16_rows(nsmi_ctx* ctx, const float* X, uint16_t* Yhi, uint16_t* Ylo, const double* Mx, int64_t O,
                          int P, int Q, int64_t I, int D2, int64_t Kp, int cls) {
  require(P >= 1 && Q >= 1 && P <= 64 && Q <= 64 && D2 >= 1 && P % D2 == 0, "mix_bf16: bad P, Q, D2");
  if (O == 0 || I == 0) return;
  ProfScope ps(ctx, cls, 2.0 * double(O) * double(I) * P * Q, double(O) * double(I) * (P * 4.0 + Q * 4.0));
  // the outputs split into chunks of 4 k until the grid holds about 2048 waves
  const int64_t oy = std::min<int64_t>(O, 65535), ix = (I + 255) / 256, waves = 4 * ix * oy;
  const int64_t want = std::max<int64_t>(1, (2048 + waves - 1) / waves);
  const int quads = (P + 3) / 4, split = int(std::min<int64_t>(quads, want));
  const int PC = 4 * ((quads + split - 1) / split);
  const dim3 grid{unsigned(ix), unsigned(oy), unsigned((P + PC - 1) / PC)};
#define NSMI_MIX_GO(QMAX)                                                                                          \
  hipLaunchKernelGGL((k_mix_bf16_rows<QMAX>), grid, dim3(256), 0, ctx->stream, X, Yhi, Ylo, Mx, O, P, Q, I, D2, Kp, \
                     PC)
  if (Q <= 12) NSMI_MIX_GO(12);
  else if (Q <= 20) NSMI_MIX_GO(20);
  else if (Q <= 32) NSMI_MIX_GO(32);
  else if (Q <= 48) NSMI_MIX_GO(48);
  else NSMI_MIX_GO(64);
#undef NSMI_MIX_GO
  NSMI_LAUNCH_CHECK();
}

// Cyclic Jacobi eigensolver for small dense symmetric matrices (host), used for
// the Krylov projected problems; eigenvalues ascending, eigenvectors as columns
// of V (row-major n x n).  The rotated element is set to zero and not left to rounding: its residue
// (about 1e-17 of the norm) kept the sum of squares above the stopping bound, so that every
// call ran all of its 100 sweeps (10 x 10 tridiagonal: 330-485 us, now 6-14; 3 x 3: 22-28, now
// 0.5-0.7; residuals 2e-16 to 1e-15 of the norm, now 4e-17 to 5e-16).  A and the
// transposed V are updated by rows, which vectorises; A's columns mirror them.
void small_sym_eigh(int n, const double* Ain, double* w, double* V) {
  std::vector<double> A(Ain, Ain + size_t(n) * n), Vt(size_t(n) * n, 0.0);
  for (int i = 0; i < n; ++i) Vt[i * n + i] = 1.0;
  const auto rotate = [n](double* __restrict__ x, double* __restrict__ y, double c, double s) {
    for (int k = 0; k < n; ++k) {
      const double xk = x[k], yk = y[k];
      x[k] = c * xk - s * yk;
      y[k] = s * xk + c * yk;
    }
  };
  for (int sweep = 0; sweep < 100; ++sweep) {
    double off = 0.0, tot = 0.0;
    for (int i = 0; i < n; ++i)
      for (int j = 0; j < n; ++j) {
        tot += A[i * n + j] * A[i * n + j];
        if (i != j) off += A[i * n + j] * A[i * n + j];
      }
    if (off <= 1e-34 * tot || off == 0.0) break;
    for (int p = 0; p < n - 1; ++p)
      for (int q = p + 1; q < n; ++q) {
        const double apq = A[p * n + q];
        if (apq == 0.0) continue;
        const double app = A[p * n + p], aqq = A[q * n + q];
        const double theta = (aqq - app) / (2.0 * apq);
        const double t = (theta >= 0 ? 1.0 : -1.0) / (std::fabs(theta) + std::sqrt(theta * theta + 1.0));
        const double c = 1.0 / std::sqrt(t * t + 1.0), s = t * c;
        rotate(&A[p * n], &A[q * n], c, s);
        A[p * n + p] = app - t * apq;
        A[q * n + q] = aqq + t * apq;
        A[p * n + q] = A[q * n + p] = 0.0;
        for (int k = 0; k < n; ++k) {
          A[k * n + p] = A[p * n + k];
          A[k * n + q] = A[q * n + k];
        }
        rotate(&Vt[p * n], &Vt[q * n], c, s);
      }
  }
  std::vector<int> idx(n);
  std::iota(idx.begin(), idx.end(), 0);
  std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) { return A[a * n + a] < A[b * n + b]; });
  for (int j = 0; j < n; ++j) {
    w[j] = A[idx[j] * n + idx[j]];
    for (int i = 0; i < n; ++i) V[i * n + j] = Vt[idx[j] * n + i];
  }
}

}  // namespace nsmi

// ------------------------------------------------------------------ H_eff
static void heff_apply_impl(nsmi_ctx* ctx, nsmi_heff* op, const double* x, double* y, int prec) {
  if (op->net) {
    net_apply(ctx, op->net, x, y);
    return;
  }
  if (op->bs) {
    bs_run(ctx, op->bs, x, y);
    return;
  }
  const int64_t M1 = op->cl * op->D0, K1 = op->cl, N1 = op->dphys * op->cr;
  const int64_t M2 = op->cl * op->dphys, K2 = op->D2 * op->cr, N2 = op->cr;
  GemmDesc g1 = desc(M1, N1, K1, false, false);
  GemmDesc g2 = desc(M2, N2, K2, false, true);
  if (op->cplx && prec == NSMI_PREC_FP32) {
    // ComplexF32 form: x in, y out as ComplexF64; GEMMs on FP32 MFMA
    float* T1 = static_cast<float*>(op->T1);
    float* T3 = static_cast<float*>(op->T3);
    Scratch xs(ctx, sizeof(float) * 2 * op->n), ys(ctx, sizeof(float) * 2 * op->n);
    vec_to_f32(ctx, xs.as<float>(), x, 2 * op->n);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM1, 4.0 * op->flops_gemm1, 8.0 * (M1 * K1 + K1 * N1 + M1 * N1), true);
      gemm_c64(ctx, g1, op->L32, false, xs.as<float>(), false, T1, kRoleHeff1);
    }
    mix_f32(ctx, T1, T3, op->Mx, op->cl, op->P, op->Q, 2 * op->cr, NSMI_K_HEFF_MIX);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM2, 4.0 * op->flops_gemm2, 8.0 * (M2 * K2 + K2 * N2 + M2 * N2), true);
      gemm_c64(ctx, g2, T3, false, op->R32, false, ys.as<float>(), kRoleHeff2);
    }
    vec_f32_to_f64(ctx, y, ys.as<float>(), 2 * op->n);
    return;
  }
  if (op->cplx) {
    // complex GEMMs; the real MPO mixing acts on interleaved (re, im) pairs as on
    // a real array with a doubled innermost extent
    double* T1 = static_cast<double*>(op->T1);
    double* T3 = static_cast<double*>(op->T3);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM1, 4.0 * op->flops_gemm1, 16.0 * (M1 * K1 + K1 * N1 + M1 * N1), true);
      gemm_c128(ctx, g1, dptr(op->L), false, x, false, T1, kRoleHeff1);
    }
    mix_f64(ctx, T1, T3, op->Mx, op->cl, op->P, op->Q, 2 * op->cr, NSMI_K_HEFF_MIX);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM2, 4.0 * op->flops_gemm2, 16.0 * (M2 * K2 + K2 * N2 + M2 * N2), true);
      gemm_c128(ctx, g2, T3, false, dptr(op->R), false, y, kRoleHeff2);
    }
    return;
  }
  if (prec == NSMI_PREC_FP64) {
    double* T1 = static_cast<double*>(op->T1);
    double* T3 = static_cast<double*>(op->T3);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM1, op->flops_gemm1, 8.0 * (M1 * K1 + K1 * N1 + M1 * N1), true);
      gemm_f64(ctx, g1, 1.0, dptr(op->L), x, 0.0, T1, kRoleHeff1);
    }
    mix_f64(ctx, T1, T3, op->Mx, op->cl, op->P, op->Q, op->cr, NSMI_K_HEFF_MIX);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM2, op->flops_gemm2, 8.0 * (M2 * K2 + K2 * N2 + M2 * N2), true);
      gemm_f64(ctx, g2, 1.0, T3, dptr(op->R), 0.0, y, kRoleHeff2);
    }
    return;
  }
  if (prec == NSMI_PREC_FP32) {
    // x is rounded to FP32 as GEMM1 stages it and y widened to FP64 as GEMM2 stores it
    float* T1 = static_cast<float*>(op->T1);
    float* T3 = static_cast<float*>(op->T3);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM1, op->flops_gemm1, 4.0 * (M1 * K1 + M1 * N1) + 8.0 * K1 * N1, true);
      gemm_f32_heff1_bd(ctx, g1, op->L32, x, T1);
    }
    mix_f32(ctx, T1, T3, op->Mx, op->cl, op->P, op->Q, op->cr, NSMI_K_HEFF_MIX);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM2, op->flops_gemm2, 4.0 * (M2 * K2 + K2 * N2) + 8.0 * M2 * N2, true);
      gemm_f32_heff2_cd(ctx, g2, T3, op->R32, y);
    }
    return;
  }
  if (prec == NSMI_PREC_BF16X3 || prec == NSMI_PREC_BF16) {
    // theta^T split into bf16 planes: GEMM1 is L . theta as an NT product
    const int terms = prec == NSMI_PREC_BF16X3 ? 3 : 1;
    split_bf16_pad(ctx, x, N1, K1, op->Kp1, op->xThi, op->xTlo, 1);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM1, op->flops_gemm1, 2.0 * terms * (M1 + N1) * op->Kp1 + 4.0 * M1 * N1, true);
      gemm_bf16_nt(ctx, M1, N1, op->Kp1, op->Lhi, op->Llo, op->Kp1, op->xThi, op->xTlo, op->Kp1, op->T1f, N1,
                   false, terms, kRoleHeff1);
    }
    mix_f32_to_bf16_rows(ctx, op->T1f, op->T3hi, op->T3lo, op->Mx, op->cl, op->P, op->Q, op->cr, int(op->D2),
                         op->Kp2, NSMI_K_HEFF_MIX);
    {
      ProfScope ps(ctx, NSMI_K_HEFF_GEMM2, op->flops_gemm2, 2.0 * terms * (M2 + N2) * op->Kp2 + 8.0 * M2 * N2, true);
      gemm_bf16_nt(ctx, M2, N2, op->Kp2, op->T3hi, op->T3lo, op->Kp2, op->Rhi, op->Rlo, op->Kp2, y, N2, true, terms,
                   kRoleHeff2);
    }
    return;
  }
  fail(NSMI_ERR_UNSUPPORTED, "H_eff precision not served by this build");
}

namespace nsmi {
void heff_apply_dev(nsmi_ctx* ctx, nsmi_heff* op, const double* x, double* y) {
  heff_apply_impl(ctx, op, x, y, op->precision);
}
int64_t heff_size(const nsmi_heff* op) { return op->n; }
bool heff_noalloc_ok(const nsmi_heff* op) {
  return !op->net && !op->bs && !op->cplx && (op->precision == NSMI_PREC_FP64 || op->precision == NSMI_PREC_FP32);
}
bool heff_is_complex(const nsmi_heff* op) { return op->cplx; }
}  // namespace nsmi

static void heff_release(nsmi_ctx* ctx, nsmi_heff* op) {
  void* bufs[] = {op->Mx, op->T1, op->T3, op->L32, op->R32, op->Lhi, op->Llo, op->Rhi, op->Rlo,
                  op->xThi, op->xTlo, op->T3hi, op->T3lo, op->T1f};
  for (void* b : bufs) scratch_release(ctx, b);
  net_release(ctx, op->net);
  bs_release(ctx, op->bs);
  delete op;
}

namespace nsmi {
nsmi_heff* heff_wrap_net(NetProgram* p) {
  nsmi_heff* op = new nsmi_heff();
  op->net = p;
  op->nsite = 0;
  op->precision = NSMI_PREC_FP64;
  op->cplx = net_is_complex(p);
  op->n = net_size(p);
  return op;
}
nsmi_heff* heff_wrap_bs(BsProgram* p, int64_t n) {
  nsmi_heff* op = new nsmi_heff();
  op->bs = p;
  op->nsite = 0;
  op->precision = NSMI_PREC_FP64;
  op->cplx = false;
  op->n = n;
  return op;
}
BsProgram* heff_bs_program(nsmi_heff* op) { return op ? op->bs : nullptr; }
}  // namespace nsmi

extern "C" {


int nsmi_heff_create(nsmi_ctx* ctx, const nsmi_tensor* L, const nsmi_tensor* W1, const nsmi_tensor* W2,
                     const nsmi_tensor* R, int precision, nsmi_heff** out) {
  if (!ctx || !out) return NSMI_ERR_INVALID;
  nsmi_heff* op = nullptr;
  API_BEGIN(ctx)
  *out = nullptr;
  require(L && R, "heff: L and R are required");
  const bool cplx = L->dtype == NSMI_C128;
  if (!cplx) {
    check_f64(L, "L");
    check_f64(R, "R");
  } else {
    require(R->dtype == NSMI_C128, "heff: L and R must have the same element type");
    if (precision != NSMI_PREC_FP64 && precision != NSMI_PREC_FP32)
      fail(NSMI_ERR_UNSUPPORTED, "heff: complex operators are served in FP64 and FP32");
  }
  check_f64(W1, "W1 (the MPO is real)");
  require(L->rank == 3 && R->rank == 3 && W1->rank == 4, "heff: L, R must be rank 3 and W rank 4");
  require(precision == NSMI_PREC_FP64 || precision == NSMI_PREC_FP32 || precision == NSMI_PREC_BF16X3 ||
              precision == NSMI_PREC_BF16,
          "heff: unknown precision");
  op = new nsmi_heff();
  op->cplx = cplx;
  op->L = L;
  op->R = R;
  op->precision = precision;
  op->cl = L->dims[0];
  op->cr = R->dims[0];
  op->D0 = L->dims[1];
  require(L->dims[2] == op->cl && R->dims[2] == op->cr, "heff: environments must be square in the links");
  require(W1->dims[0] == op->D0 && W1->dims[2] == W1->dims[3], "heff: W1 does not match L");
  const int64_t d1 = W1->dims[2];
  if (W2) {
    check_f64(W2, "W2");
    require(W2->rank == 4 && W2->dims[0] == W1->dims[1] && W2->dims[2] == W2->dims[3], "heff: W2 does not match W1");
    const int64_t Dm = W1->dims[1], d2 = W2->dims[2];
    op->nsite = 2;
    op->D2 = W2->dims[1];
    op->dphys = d1 * d2;
    require(R->dims[1] == op->D2, "heff: R does not match W2");
    op->Q = int(op->D0 * d1 * d2);
    op->P = int(d1 * d2 * op->D2);
    require(op->P <= 64 && op->Q <= 64, "heff: D*d^2 above 64 is not served");
    op->Mx = static_cast<double*>(scratch(ctx, sizeof(double) * op->P * op->Q));
    const int np = op->P * op->Q;
    hipLaunchKernelGGL(k_build_w12, dim3((np + 255) / 256), dim3(256), 0, ctx->stream, dptr(W1), dptr(W2), op->Mx,
                       int(op->D0), int(Dm), int(op->D2), int(d1), int(d2));
    NSMI_LAUNCH_CHECK();
  } else {
    op->nsite = 1;
    op->D2 = W1->dims[1];
    op->dphys = d1;
    require(R->dims[1] == op->D2, "heff: R does not match W");
    op->Q = int(op->D0 * d1);
    op->P = int(d1 * op->D2);
    require(op->P <= 64 && op->Q <= 64, "heff: D*d above 64 is not served");
    op->Mx = static_cast<double*>(scratch(ctx, sizeof(double) * op->P * op->Q));
    build_w1(ctx, dptr(W1), op->Mx, int(op->D0), int(op->D2), int(d1), 0);
  }
  op->n = op->cl * op->dphys * op->cr;
  const bool bf = precision == NSMI_PREC_BF16X3 || precision == NSMI_PREC_BF16;
  const bool two = precision == NSMI_PREC_BF16X3;
  if (!bf) {
    const size_t elt = (cplx ? 2 : 1) * prec_elt(precision);
    op->T1 = scratch(ctx, elt * size_t(op->cl * op->D0 * op->dphys * op->cr));
    op->T3 = scratch(ctx, elt * size_t(op->cl * op->D2 * op->dphys * op->cr));
  } else {
    // planes: L as (cl*D0) x Kp1, theta^T as (dphys*cr) x Kp1, T3 as (cl*dphys) x Kp2, R as cr x Kp2
    op->Kp1 = pad32(op->cl);
    op->Kp2 = pad32(op->D2 * op->cr);
    const size_t nL = size_t(op->cl * op->D0 * op->Kp1), nX = size_t(op->dphys * op->cr * op->Kp1);
    const size_t nT3 = size_t(op->cl * op->dphys * op->Kp2), nR = size_t(op->cr * op->Kp2);
    op->Lhi = static_cast<uint16_t*>(scratch(ctx, 2 * nL));
    op->Rhi = static_cast<uint16_t*>(scratch(ctx, 2 * nR));
    op->xThi = static_cast<uint16_t*>(scratch(ctx, 2 * nX));
    op->T3hi = static_cast<uint16_t*>(scratch(ctx, 2 * nT3));
    if (two) {
      op->Llo = static_cast<uint16_t*>(scratch(ctx, 2 * nL));
      op->Rlo = static_cast<uint16_t*>(scratch(ctx, 2 * nR));
      op->xTlo = static_cast<uint16_t*>(scratch(ctx, 2 * nX));
      op->T3lo = static_cast<uint16_t*>(scratch(ctx, 2 * nT3));
    }
    op->T1f = static_cast<float*>(scratch(ctx, 4 * size_t(op->cl * op->D0 * op->dphys * op->cr)));
    split_bf16_pad(ctx, dptr(L), op->cl * op->D0, op->cl, op->Kp1, op->Lhi, op->Llo, 0);
    split_bf16_pad(ctx, dptr(R), op->cr, op->D2 * op->cr, op->Kp2, op->Rhi, op->Rlo, 0);
    // the K padding of T3 is never written by the mixing kernel: clear it once
    NSMI_HIP(hipMemsetAsync(op->T3hi, 0, 2 * nT3, ctx->stream));
    if (two) NSMI_HIP(hipMemsetAsync(op->T3lo, 0, 2 * nT3, ctx->stream));
  }
  op->flops_gemm1 = 2.0 * double(op->cl * op->D0) * double(op->dphys * op->cr) * double(op->cl);
  op->flops_gemm2 = 2.0 * double(op->cl * op->dphys) * double(op->cr) * double(op->D2 * op->cr);
  op->flops_mix = 2.0 * double(op->cl) * double(op->cr) * op->P * op->Q;
  if (precision == NSMI_PREC_FP32) {
    const int64_t c = cplx ? 2 : 1;  // scalars per element
    op->L32 = static_cast<float*>(scratch(ctx, sizeof(float) * L->numel * c));
    op->R32 = static_cast<float*>(scratch(ctx, sizeof(float) * R->numel * c));
    vec_to_f32(ctx, op->L32, dptr(L), L->numel * c);
    vec_to_f32(ctx, op->R32, dptr(R), R->numel * c);
  }
  *out = op;
  op = nullptr;
  }
  catch (const nsmi::Error& e) {
    if (op) heff_release(ctx, op);
    ctx->err = e.what();
    return e.code;
  }
  catch (const std::exception& e) {
    if (op) heff_release(ctx, op);
    ctx->err = std::string("internal: ") + e.what();
    return NSMI_ERR_INVALID;
  }
  return NSMI_OK;
}

int nsmi_heff_destroy(nsmi_ctx* ctx, nsmi_heff* op) {
  if (!ctx) return NSMI_ERR_INVALID;
  if (!op) return NSMI_OK;
  API_BEGIN(ctx)
  heff_release(ctx, op);
  API_END(ctx)
}

int nsmi_heff_apply(nsmi_ctx* ctx, nsmi_heff* op, const nsmi_tensor* x, nsmi_tensor* y) {
  if (!ctx || !op) return NSMI_ERR_INVALID;
  API_BEGIN(ctx)
  const int dt = op->cplx ? NSMI_C128 : NSMI_F64;
  require(x && y && x->dtype == dt && y->dtype == dt, "heff_apply: x/y element type does not match the operator");
  require(x->numel == op->n && y->numel == op->n, "heff_apply: x/y size does not match the operator");
  require(x->data != y->data, "heff_apply: x and y must not alias");
  heff_apply_impl(ctx, op, static_cast<const double*>(x->data), static_cast<double*>(y->data), op->precision);
  API_END(ctx)
}

int nsmi_heff_rayleigh(nsmi_ctx* ctx, nsmi_heff* op, const nsmi_tensor* x, double* e) {
  if (!ctx || !op || !e) return NSMI_ERR_INVALID;
  API_BEGIN(ctx)
  require(x && x->dtype == (op->cplx ? NSMI_C128 : NSMI_F64), "rayleigh: element type does not match");
  require(x->numel == op->n, "rayleigh: size mismatch");
  // an FP64 apply of a reduced-precision operator needs FP64-sized workspace
  const size_t e64 = op->cplx ? 16 : 8;
  const bool swap = !op->net && !op->bs && op->precision != NSMI_PREC_FP64;
  void* T1 = op->T1;
  void* T3 = op->T3;
  Scratch t1(ctx, swap ? e64 * size_t(op->cl * op->D0 * op->dphys * op->cr) : 8);
  Scratch t3(ctx, swap ? e64 * size_t(op->cl * op->D2 * op->dphys * op->cr) : 8);
  if (swap) {
    op->T1 = t1.p;
    op->T3 = t3.p;
  }
  Scratch ys(ctx, e64 * size_t(op->n));
  try {
    heff_apply_impl(ctx, op, dptr(x), ys.as<double>(), NSMI_PREC_FP64);
  } catch (...) {
    op->T1 = T1;
    op->T3 = T3;
    throw;
  }
  op->T1 = T1;
  op->T3 = T3;
  if (op->cplx) {
    vec_zdot_dev(ctx, dptr(x), ys.as<double>(), op->n, 0);
    vec_dot_dev(ctx, dptr(x), dptr(x), 2 * op->n, 2);
    double r[3];
    read_slots(ctx, 3, r);
    require(r[2] > 0.0, "rayleigh: zero vector");
    *e = r[0] / r[2];
    return NSMI_OK;
  }
  vec_dot_dev(ctx, dptr(x), ys.as<double>(), op->n, 0);
  vec_dot_dev(ctx, dptr(x), dptr(x), op->n, 1);
  double r[2];
  read_slots(ctx, 2, r);
  require(r[1] > 0.0, "rayleigh: zero vector");
  *e = r[0] / r[1];
  API_END(ctx)
}

// ----------------------------------------------------------- environments
int nsmi_env_update(nsmi_ctx* ctx, const nsmi_tensor* E, const nsmi_tensor* A, const nsmi_tensor* W, int side,
                    int precision, nsmi_tensor** out) {
  if (!ctx || !out) return NSMI_ERR_INVALID;
  API_BEGIN(ctx)
  *out = nullptr;
  require(E && A, "env_update: E and A are required");
  const bool cplx = A->dtype == NSMI_C128;
  if (cplx)
    require(E->dtype == NSMI_C128, "env_update: E and A must have the same element type");
  else {
    check_f64(E, "E");
    check_f64(A, "A");
  }
  check_f64(W, "W (the MPO is real)");
  require(E->rank == 3 && A->rank == 3 && W->rank == 4, "env_update: ranks must be E:3, A:3, W:4");
  require(side == 0 || side == 1, "env_update: side must be 0 (left) or 1 (right)");
  if (precision != NSMI_PREC_FP64) fail(NSMI_ERR_UNSUPPORTED, "env_update: environments are computed in FP64");
  const int64_t ca = A->dims[0], d = A->dims[1], cb = A->dims[2];
  require(W->dims[2] == d && W->dims[3] == d, "env_update: W physical dims do not match A");
  if (cplx) {
    const int64_t Dl = W->dims[0], Dr = W->dims[1];
    const double* Ad = static_cast<const double*>(A->data);
    const double* Ed = static_cast<const double*>(E->data);
    nsmi_tensor* res = nullptr;
    if (side == 0) {
      require(E->dims[0] == ca && E->dims[2] == ca && E->dims[1] == Dl, "env_update(left): E does not match A/W");
      const int Q = int(Dl * d), P = int(d * Dr);
      require(P <= 64 && Q <= 64, "env_update: D*d above 64 is not served");
      Scratch dmx(ctx, size_t(P) * Q * 8);
      build_w1(ctx, dptr(W), dmx.as<double>(), int(Dl), int(Dr), int(d), 0);
      const int64_t dims[3] = {cb, Dr, cb};
      res = tensor_new(ctx, NSMI_C128, 3, dims);
      Scratch X(ctx, 16 * size_t(ca * Dl * d * cb)), Y(ctx, 16 * size_t(ca * d * Dr * cb));
      ProfScope ps(ctx, NSMI_K_ENV, 4.0 * (2.0 * ca * Dl * ca * d * cb + 2.0 * cb * Dr * cb * ca * d),
                   16.0 * (E->numel + 2 * A->numel + res->numel));
      gemm_c128(ctx, desc(ca * Dl, d * cb, ca, false, false), Ed, false, Ad, false, X.as<double>(), kRoleEnv);
      mix_f64(ctx, X.as<double>(), Y.as<double>(), dmx.as<double>(), ca, P, Q, 2 * cb, -1);
      gemm_c128(ctx, desc(cb, Dr * cb, ca * d, true, false), Ad, true, Y.as<double>(), false,
                static_cast<double*>(res->data), kRoleEnv);
    } else {
      require(E->dims[0] == cb && E->dims[2] == cb && E->dims[1] == Dr, "env_update(right): E does not match A/W");
      const int Q = int(d * Dr), P = int(Dl * d);
      require(P <= 64 && Q <= 64, "env_update: D*d above 64 is not served");
      Scratch dmx(ctx, size_t(P) * Q * 8);
      build_w1(ctx, dptr(W), dmx.as<double>(), int(Dl), int(Dr), int(d), 1);
      const int64_t dims[3] = {ca, Dl, ca};
      res = tensor_new(ctx, NSMI_C128, 3, dims);
      Scratch X(ctx, 16 * size_t(ca * d * Dr * cb)), Y(ctx, 16 * size_t(ca * Dl * d * cb));
      ProfScope ps(ctx, NSMI_K_ENV, 4.0 * (2.0 * ca * d * cb * Dr * cb + 2.0 * ca * Dl * ca * d * cb),
                   16.0 * (E->numel + 2 * A->numel + res->numel));
      gemm_c128(ctx, desc(ca * d, Dr * cb, cb, false, false), Ad, true, Ed, false, X.as<double>(), kRoleEnv);
      mix_f64(ctx, X.as<double>(), Y.as<double>(), dmx.as<double>(), ca, P, Q, 2 * cb, -1);
      gemm_c128(ctx, desc(ca * Dl, ca, d * cb, false, true), Y.as<double>(), false, Ad, false,
                static_cast<double*>(res->data), kRoleEnv);
    }
    *out = res;
    return NSMI_OK;
  }
  const int64_t Dl = W->dims[0], Dr = W->dims[1];
  nsmi_tensor* res = nullptr;
  if (side == 0) {
    require(E->dims[0] == ca && E->dims[2] == ca && E->dims[1] == Dl, "env_update(left): E does not match A/W");
    const int Q = int(Dl * d), P = int(d * Dr);
    require(P <= 64 && Q <= 64, "env_update: D*d above 64 is not served");
    Scratch dmx(ctx, size_t(P) * Q * 8);  // Mx[(s' w'), (w s)] = W[w, w', s', s]
    build_w1(ctx, dptr(W), dmx.as<double>(), int(Dl), int(Dr), int(d), 0);
    const int64_t dims[3] = {cb, Dr, cb};
    res = tensor_new(ctx, NSMI_F64, 3, dims);
    Scratch X(ctx, 8 * size_t(ca * Dl * d * cb)), Y(ctx, 8 * size_t(ca * d * Dr * cb));
    const double fl = 2.0 * ca * Dl * ca * d * cb + 2.0 * cb * Dr * cb * ca * d;
    ProfScope ps(ctx, NSMI_K_ENV, fl + 2.0 * ca * cb * P * Q, 8.0 * (E->numel + 2 * A->numel + res->numel));
    gemm_f64(ctx, desc(ca * Dl, d * cb, ca, false, false), 1.0, dptr(E), dptr(A), 0.0, X.as<double>(), kRoleEnv);
    mix_f64(ctx, X.as<double>(), Y.as<double>(), dmx.as<double>(), ca, P, Q, cb, -1);
    gemm_f64(ctx, desc(cb, Dr * cb, ca * d, true, false), 1.0, dptr(A), Y.as<double>(), 0.0, dptr(res), kRoleEnv);
  } else {
    require(E->dims[0] == cb && E->dims[2] == cb && E->dims[1] == Dr, "env_update(right): E does not match A/W");
    const int Q = int(d * Dr), P = int(Dl * d);
    require(P <= 64 && Q <= 64, "env_update: D*d above 64 is not served");
    Scratch dmx(ctx, size_t(P) * Q * 8);  // Mx[(w s), (s' v)] = W[w, v, s', s]
    build_w1(ctx, dptr(W), dmx.as<double>(), int(Dl), int(Dr), int(d), 1);
    const int64_t dims[3] = {ca, Dl, ca};
    res = tensor_new(ctx, NSMI_F64, 3, dims);
    Scratch X(ctx, 8 * size_t(ca * d * Dr * cb)), Y(ctx, 8 * size_t(ca * Dl * d * cb));
    const double fl = 2.0 * ca * d * cb * Dr * cb + 2.0 * ca * Dl * ca * d * cb;
    ProfScope ps(ctx, NSMI_K_ENV, fl + 2.0 * ca * cb * P * Q, 8.0 * (E->numel + 2 * A->numel + res->numel));
    gemm_f64(ctx, desc(ca * d, Dr * cb, cb, false, false), 1.0, dptr(A), dptr(E), 0.0, X.as<double>(), kRoleEnv);
    mix_f64(ctx, X.as<double>(), Y.as<double>(), dmx.as<double>(), ca, P, Q, cb, -1);
    gemm_f64(ctx, desc(ca * Dl, ca, d * cb, false, true), 1.0, Y.as<double>(), dptr(A), 0.0, dptr(res), kRoleEnv);
  }
  *out = res;
  API_END(ctx)
}

int nsmi_theta(nsmi_ctx* ctx, const nsmi_tensor* A, const nsmi_tensor* B, nsmi_tensor** theta) {
  if (!ctx || !theta) return NSMI_ERR_INVALID;
  API_BEGIN(ctx)
  *theta = nullptr;
  require(A && B, "theta: A and B are required");
  require(A->rank == 3 && B->rank == 3 && A->dims[2] == B->dims[0], "theta: A[l,s,m] and B[m,s,r] required");
  const int64_t cl = A->dims[0], d1 = A->dims[1], cm = A->dims[2], d2 = B->dims[1], cr = B->dims[2];
  const int64_t dims[4] = {cl, d1, d2, cr};
  if (A->dtype == NSMI_C128 || B->dtype == NSMI_C128) {
    require(A->dtype == B->dtype, "theta: A and B must have the same element type");
    nsmi_tensor* t = tensor_new(ctx, NSMI_C128, 4, dims);
    ProfScope ps(ctx, NSMI_K_THETA, 8.0 * cl * d1 * cm * d2 * cr, 16.0 * (A->numel + B->numel + t->numel));
    gemm_c128(ctx, desc(cl * d1, d2 * cr, cm, false, false), static_cast<const double*>(A->data), false,
              static_cast<const double*>(B->data), false, static_cast<double*>(t->data), kRoleTheta);
    *theta = t;
    return NSMI_OK;
  }
  check_f64(A, "A");
  check_f64(B, "B");
  nsmi_tensor* t = tensor_new(ctx, NSMI_F64, 4, dims);
  ProfScope ps(ctx, NSMI_K_THETA, 2.0 * cl * d1 * cm * d2 * cr, 8.0 * (A->numel + B->numel + t->numel));
  gemm_f64(ctx, desc(cl * d1, d2 * cr, cm, false, false), 1.0, dptr(A), dptr(B), 0.0, dptr(t), kRoleTheta);
  *theta = t;
  API_END(ctx)
}


}  // extern "C"
