// Complex GEMM for the TDVP path: ComplexF64 on v_mfma_f64_16x16x4 and ComplexF32
// on v_mfma_f32_16x16x4 (the FP32 form of tree H_eff contraction programs).
//
// Complex tensors are interleaved (re, im) pairs.  Tiles are staged into LDS as
// separate real and imaginary planes (conjugation applied at staging), and each
// 16x16 output block takes four real MFMAs (small grids: k_zgemm_wave, without LDS tiles):
//   re += ar.br - ai.bi      im += ar.bi + ai.br
// Row-major, op(A) M x K (A stored K x M when transA), op(B) K x N (stored N x K
// when transB); C = op(A) op(B) (no scaling).  Output rows of the f64 MFMA are
// interleaved across lane groups (item r of lane l is row l/16 + 4r); the f32
// MFMA writes row 4(l/16) + r.
#include "internal.h"

namespace nsmi {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

template <typename T> struct ZT;
template <> struct ZT<double> {
  typedef d4 acc;
  typedef d2 pair;
  __device__ static d4 mfma(double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
  __device__ static int row(int kl, int r) { return kl + 4 * r; }
};
template <> struct ZT<float> {
  typedef f4 acc;
  typedef f2 pair;
  __device__ static f4 mfma(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  __device__ static int row(int kl, int r) { return 4 * kl + r; }
};

template <typename T>
struct ZArgs {
  const T* A;
  const T* B;
  T* C;
  int64_t M, N, K, lda, ldb, ldc;  // leading dimensions in complex elements
  int conjA, conjB;
  int tiles_m, tiles_n;
  // network-program steps (MODE 1): A element (m, k) at arow[m] + acol[k] and C element
  // (m, n) at crow[m] + ccol[n] (complex elements) where the tables are given; A and C
  // stored as complex double (a_f64, c_f64) in the FP32 form, converted on the way
  const int64_t *arow = nullptr, *acol = nullptr, *crow = nullptr, *ccol = nullptr;
  int a_f64 = 0, c_f64 = 0;
};

__device__ inline int zxcd_remap(int wg, int nwg) {
  constexpr int kXcd = 8;
  if (nwg < 2 * kXcd || (nwg % kXcd) != 0) return wg;
  return (wg % kXcd) * (nwg / kXcd) + wg / kXcd;
}

// MODE 0: the plain row-major GEMM; MODE 1 (TA = TB = false): a network-program step
// reading A and writing C through the offset tables of ZArgs
template <typename T, int BM, int BN, bool TA, bool TB, int ROLE, int MODE = 0>
__global__ __launch_bounds__(256) void k_zgemm(ZArgs<T> g) {
  typedef typename ZT<T>::acc Acc;
  typedef typename ZT<T>::pair V2;
  constexpr int BK = 8, PAD = 4;
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int FM = WTM / 16, FN = WTN / 16;
  constexpr int EA = BM * BK / 256, EB = BN * BK / 256;
  __shared__ T sAr[2][BK][BM + PAD], sAi[2][BK][BM + PAD];
  __shared__ T sBr[2][BK][BN + PAD], sBi[2][BK][BN + PAD];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int tile = zxcd_remap(blockIdx.x, g.tiles_m * g.tiles_n);
  const int tm = tile / g.tiles_n, tn = tile % g.tiles_n;
  const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
  const T sa = g.conjA ? T(-1) : T(1), sb = g.conjB ? T(-1) : T(1);

  V2 ra[EA > 0 ? EA : 1], rb[EB > 0 ? EB : 1];
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int j = 0; j < EA; ++j) {
      const int e = tid * EA + j;
      const int mm = TA ? (e % BM) : (e / BK);
      const int kk = TA ? (e / BM) : (e % BK);
      const int64_t gm = m0 + mm, gk = k0 + kk;
      V2 v = {T(0), T(0)};
      if constexpr (MODE == 1) {
        if (gm < g.M && gk < g.K) {
          const int64_t off = g.arow ? g.arow[gm] + g.acol[gk] : gm * g.lda + gk;
          if (g.a_f64) {
            const d2 w = *reinterpret_cast<const d2*>(reinterpret_cast<const double*>(g.A) + 2 * off);
            v = V2{T(w.x), T(w.y)};
          } else {
            v = *reinterpret_cast<const V2*>(g.A + 2 * off);
          }
        }
      } else if (gm < g.M && gk < g.K) {
        v = *reinterpret_cast<const V2*>(g.A + 2 * (TA ? gk * g.lda + gm : gm * g.lda + gk));
      }
      ra[j] = v;
    }
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const int e = tid * EB + j;
      const int nn = TB ? (e / BK) : (e % BN);
      const int kk = TB ? (e % BK) : (e / BN);
      const int64_t gn = n0 + nn, gk = k0 + kk;
      V2 v = {T(0), T(0)};
      if (gn < g.N && gk < g.K)
        v = *reinterpret_cast<const V2*>(g.B + 2 * (TB ? gn * g.ldb + gk : gk * g.ldb + gn));
      rb[j] = v;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < EA; ++j) {
      const int e = tid * EA + j;
      const int mm = TA ? (e % BM) : (e / BK);
      const int kk = TA ? (e / BM) : (e % BK);
      sAr[buf][kk][mm] = ra[j].x;
      sAi[buf][kk][mm] = sa * ra[j].y;
    }
#pragma unroll
    for (int j = 0; j < EB; ++j) {
      const int e = tid * EB + j;
      const int nn = TB ? (e / BK) : (e % BN);
      const int kk = TB ? (e % BK) : (e / BN);
      sBr[buf][kk][nn] = rb[j].x;
      sBi[buf][kk][nn] = sb * rb[j].y;
    }
  };

  Acc acr[FM][FN], aci[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      acr[i][j] = Acc{0, 0, 0, 0};
      aci[i][j] = Acc{0, 0, 0, 0};
    }
  const int64_t nk = (g.K + BK - 1) / BK;
  load(0);
  store(0);
  __syncthreads();
  const int kl = lane >> 4, ml = lane & 15;
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int buf = int(kt & 1);
    if (kt + 1 < nk) load((kt + 1) * BK);
#pragma unroll
    for (int ks = 0; ks < BK / 4; ++ks) {
      T ar[FM], ai[FM], br[FN], bi[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        ar[i] = sAr[buf][ks * 4 + kl][wm * WTM + i * 16 + ml];
        ai[i] = sAi[buf][ks * 4 + kl][wm * WTM + i * 16 + ml];
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        br[j] = sBr[buf][ks * 4 + kl][wn * WTN + j * 16 + ml];
        bi[j] = sBi[buf][ks * 4 + kl][wn * WTN + j * 16 + ml];
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          acr[i][j] = ZT<T>::mfma(ar[i], br[j], acr[i][j]);
          acr[i][j] = ZT<T>::mfma(-ai[i], bi[j], acr[i][j]);
          aci[i][j] = ZT<T>::mfma(ar[i], bi[j], aci[i][j]);
          aci[i][j] = ZT<T>::mfma(ai[i], br[j], aci[i][j]);
        }
    }
    if (kt + 1 < nk) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t gm = m0 + wm * WTM + i * 16 + ZT<T>::row(kl, r);
        const int64_t gn = n0 + wn * WTN + j * 16 + ml;
        if (gm < g.M && gn < g.N) {
          V2 v = {acr[i][j][r], aci[i][j][r]};
          if constexpr (MODE == 1) {
            const int64_t off = g.crow ? g.crow[gm] + g.ccol[gn] : gm * g.ldc + gn;
            if (g.c_f64)
              *reinterpret_cast<d2*>(reinterpret_cast<double*>(g.C) + 2 * off) = d2{double(v.x), double(v.y)};
            else
              *reinterpret_cast<V2*>(g.C + 2 * off) = v;
          } else {
            *reinterpret_cast<V2*>(g.C + 2 * (gm * g.ldc + gn)) = v;
          }
        }
      }
}

// The same product for grids too small to fill the chip, where a tile's serial chain of
// slabs (load, barrier, MFMA) is the whole time: one 16 x 16 block of C per
// workgroup, K dealt to its 8 waves in chunks of 16, operands straight from memory into
// the MFMA registers (every element of a block's rows is used once: staging through LDS
// would add a barrier per slab and share nothing), the next chunk's loads in flight, and
// the 8 partial sums added in wave order through LDS.
template <typename T, bool TA, bool TB, int ROLE, int MODE = 0>
__global__ __launch_bounds__(512) void k_zgemm_wave(ZArgs<T> g) {
  typedef typename ZT<T>::acc Acc;
  typedef typename ZT<T>::pair V2;
  constexpr int NW = 8, U = 4;
  __shared__ T part[NW][8][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kl = lane >> 4, ml = lane & 15;
  const int tile = zxcd_remap(blockIdx.x, g.tiles_m * g.tiles_n);
  const int64_t m0 = int64_t(tile / g.tiles_n) * 16, n0 = int64_t(tile % g.tiles_n) * 16;
  // rows and columns past the matrix repeat the last one: they reach only elements of C
  // that are not written
  const int64_t am = min(m0 + ml, g.M - 1), bn = min(n0 + ml, g.N - 1);
  const T sa = g.conjA ? T(-1) : T(1), sb = g.conjB ? T(-1) : T(1);
  const int64_t nch = (g.K + 4 * U - 1) / (4 * U);
  const int64_t ar0 = MODE == 1 && g.arow ? g.arow[am] : am * g.lda;
  V2 a[2][U], b[2][U];
  const auto load = [&](int64_t c, V2 (&xa)[U], V2 (&xb)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = min(c * (4 * U) + u * 4 + kl, g.K - 1);
      if constexpr (MODE == 1) {
        const int64_t off = ar0 + (g.arow ? g.acol[k] : k);
        if (g.a_f64) {
          const d2 w = *reinterpret_cast<const d2*>(reinterpret_cast<const double*>(g.A) + 2 * off);
          xa[u] = V2{T(w.x), T(w.y)};
        } else {
          xa[u] = *reinterpret_cast<const V2*>(g.A + 2 * off);
        }
      } else {
        xa[u] = *reinterpret_cast<const V2*>(g.A + 2 * (TA ? k * g.lda + am : ar0 + k));
      }
      xb[u] = *reinterpret_cast<const V2*>(g.B + 2 * (TB ? bn * g.ldb + k : k * g.ldb + bn));
    }
  };
  Acc acr = Acc{0, 0, 0, 0}, aci = Acc{0, 0, 0, 0};
  const auto mma = [&](int64_t c, const V2 (&xa)[U], const V2 (&xb)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = c * (4 * U) + u * 4 + kl < g.K;
      const T ar = in ? xa[u].x : T(0), ai = in ? sa * xa[u].y : T(0);
      const T br = in ? xb[u].x : T(0), bi = in ? sb * xb[u].y : T(0);
      acr = ZT<T>::mfma(ar, br, acr);
      aci = ZT<T>::mfma(ar, bi, aci);
      acr = ZT<T>::mfma(-ai, bi, acr);
      aci = ZT<T>::mfma(ai, br, aci);
    }
  };
  if (wave < nch) {
    load(wave, a[0], b[0]);
    for (int64_t c = wave; c < nch; c += 2 * NW) {
      load(min(c + NW, nch - 1), a[1], b[1]);
      mma(c, a[0], b[0]);
      if (c + NW >= nch) break;
      load(min(c + 2 * NW, nch - 1), a[0], b[0]);
      mma(c + NW, a[1], b[1]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    part[wave][r][lane] = acr[r];
    part[wave][4 + r][lane] = aci[r];
  }
  __syncthreads();
  if (tid >= 256) return;
  const int r = wave;  // waves 0..3 write item r of every lane
  V2 v = {T(0), T(0)};
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    v.x += part[w][r][lane];
    v.y += part[w][4 + r][lane];
  }
  const int64_t gm = m0 + ZT<T>::row(kl, r), gn = n0 + ml;
  if (gm >= g.M || gn >= g.N) return;
  if constexpr (MODE == 1) {
    const int64_t off = g.crow ? g.crow[gm] + g.ccol[gn] : gm * g.ldc + gn;
    if (g.c_f64)
      *reinterpret_cast<d2*>(reinterpret_cast<double*>(g.C) + 2 * off) = d2{double(v.x), double(v.y)};
    else
      *reinterpret_cast<V2*>(g.C + 2 * off) = v;
  } else {
    *reinterpret_cast<V2*>(g.C + 2 * (gm * g.ldc + gn)) = v;
  }
}

template <typename T, int BM, int BN, int ROLE>
void zlaunch(nsmi_ctx* ctx, const GemmDesc& d, ZArgs<T>& a) {
  a.tiles_m = int((d.M + BM - 1) / BM);
  a.tiles_n = int((d.N + BN - 1) / BN);
  dim3 grid(unsigned(a.tiles_m) * unsigned(a.tiles_n));
#define NSMI_ZGEMM_GO(TA, TB)                                                                  \
  do {                                                                                         \
    if constexpr (BM == 16)                                                                    \
      NSMI_LAUNCH_TIMED(ctx, (k_zgemm_wave<T, TA, TB, ROLE>), grid, dim3(512), a);             \
    else                                                                                       \
      NSMI_LAUNCH_TIMED(ctx, (k_zgemm<T, BM, BN, TA, TB, ROLE>), grid, dim3(256), a);          \
  } while (0)
  if (!d.transA && !d.transB)
    NSMI_ZGEMM_GO(false, false);
  else if (!d.transA && d.transB)
    NSMI_ZGEMM_GO(false, true);
  else if (d.transA && !d.transB)
    NSMI_ZGEMM_GO(true, false);
  else
    NSMI_ZGEMM_GO(true, true);
#undef NSMI_ZGEMM_GO
  NSMI_LAUNCH_CHECK();
}

// k_zgemm_wave where 32 x 32 tiles leave CUs without one and K is more than one of their
// slabs.  Measured (M, N, K; us, wave form / 32 x 32): ComplexF64 240, 60, 300: 6.6 / 20.5;
// 300, 240, 60: 4.4 / 6.7; 800, 200, 1000 (175 tiles): 41 / 62; ComplexF32 400, 100, 500:
// 7.4 / 24.6.  At 256 tiles (512, 512, 512) it is 31 / 36 and, with B transposed, 40 / 36; beyond
// it loses (1000, 800, 200: 40-56 / 38), and with K <= 8 both are one round trip (3.3 / 3.1).
inline bool wave_form(int64_t M, int64_t N, int64_t K) {
  return K > 8 && ((M + 31) / 32) * ((N + 31) / 32) < 256;
}

template <typename T, int ROLE>
void zrole(nsmi_ctx* ctx, const GemmDesc& d, ZArgs<T>& a) {
  const int64_t mid = ((d.M + 63) / 64) * ((d.N + 63) / 64);
  if (wave_form(d.M, d.N, d.K))
    zlaunch<T, 16, 16, ROLE>(ctx, d, a);
  else if (mid >= 256)
    zlaunch<T, 64, 64, ROLE>(ctx, d, a);
  else
    zlaunch<T, 32, 32, ROLE>(ctx, d, a);
}

template <typename T>
void gemm_cplx(nsmi_ctx* ctx, const GemmDesc& d, const T* A, bool conjA, const T* B, bool conjB, T* C, int role) {
  require(d.M >= 0 && d.N >= 0 && d.K >= 0 && d.batch == 1, "zgemm: bad sizes (no batching)");
  if (d.M == 0 || d.N == 0) return;
  ZArgs<T> a{A, B, C, d.M, d.N, d.K, d.lda, d.ldb, d.ldc, conjA ? 1 : 0, conjB ? 1 : 0, 0, 0};
  switch (role) {
    case kRoleHeff1: zrole<T, kRoleHeff1>(ctx, d, a); break;
    case kRoleHeff2: zrole<T, kRoleHeff2>(ctx, d, a); break;
    case kRoleEnv: zrole<T, kRoleEnv>(ctx, d, a); break;
    case kRoleTheta: zrole<T, kRoleTheta>(ctx, d, a); break;
    default: zrole<T, kRoleFact>(ctx, d, a); break;
  }
}

template <typename T>
void gemm_net_t(nsmi_ctx* ctx, const ZNetGemm& z) {
  require(z.M >= 0 && z.N >= 0 && z.K >= 0, "zgemm: bad sizes");
  if (z.M == 0 || z.N == 0) return;
  ZArgs<T> a{static_cast<const T*>(z.A), static_cast<const T*>(z.B), static_cast<T*>(z.C), z.M, z.N, z.K, z.K,
             z.N, z.N, 0, z.conjB ? 1 : 0, 0, 0};
  a.arow = z.arow;
  a.acol = z.acol;
  a.crow = z.crow;
  a.ccol = z.ccol;
  a.a_f64 = z.a_f64 ? 1 : 0;
  a.c_f64 = z.c_f64 ? 1 : 0;
  const int64_t mid = ((z.M + 63) / 64) * ((z.N + 63) / 64);
  if (wave_form(z.M, z.N, z.K)) {
    a.tiles_m = int((z.M + 15) / 16);
    a.tiles_n = int((z.N + 15) / 16);
    NSMI_LAUNCH_TIMED(ctx, (k_zgemm_wave<T, false, false, kRoleHeff2, 1>), dim3(unsigned(a.tiles_m) * a.tiles_n),
                      dim3(512), a);
  } else if (mid >= 256) {
    a.tiles_m = int((z.M + 63) / 64);
    a.tiles_n = int((z.N + 63) / 64);
    NSMI_LAUNCH_TIMED(ctx, (k_zgemm<T, 64, 64, false, false, kRoleHeff2, 1>), dim3(unsigned(a.tiles_m) * a.tiles_n),
                      dim3(256), a);
  } else {
    a.tiles_m = int((z.M + 31) / 32);
    a.tiles_n = int((z.N + 31) / 32);
    NSMI_LAUNCH_TIMED(ctx, (k_zgemm<T, 32, 32, false, false, kRoleHeff2, 1>), dim3(unsigned(a.tiles_m) * a.tiles_n),
                      dim3(256), a);
  }
  NSMI_LAUNCH_CHECK();
}

}  // namespace

void gemm_cplx_net(nsmi_ctx* ctx, bool lo, const ZNetGemm& z) {
  require(lo || (!z.a_f64 && !z.c_f64), "zgemm: complex-double staging is for the FP32 form");
  if (lo)
    gemm_net_t<float>(ctx, z);
  else
    gemm_net_t<double>(ctx, z);
}

void gemm_c128(nsmi_ctx* ctx, const GemmDesc& d, const double* A, bool conjA, const double* B, bool conjB,
               double* C, int role) {
  gemm_cplx<double>(ctx, d, A, conjA, B, conjB, C, role);
}

void gemm_c64(nsmi_ctx* ctx, const GemmDesc& d, const float* A, bool conjA, const float* B, bool conjB, float* C,
              int role) {
  gemm_cplx<float>(ctx, d, A, conjA, B, conjB, C, role);
}

}  // namespace nsmi
