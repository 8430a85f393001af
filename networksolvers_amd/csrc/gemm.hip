// MFMA GEMMs for gfx950 (CDNA4), row-major, strided-batched, with operand
// transposes folded into the global->LDS staging (no separate permute passes).
//
// FP64 / FP32: v_mfma_{f64,f32}_16x16x4 -- 4 waves (2x2; 8 waves as 2x4 for the
// 128 x 128 tile), each wave owns a sub-tile built from 16x16 MFMA blocks; K is
// staged in LDS slabs of 16 (32 for the 32 x 32 tile) with register prefetch two slabs
// ahead (double-buffered LDS, one barrier per slab).  Bound: MFMA issue for large products
// (the 128 x 128 tile is one workgroup per CU and reaches 66 of the 73 TF/s that a large
// FP64 library product does; 4096 x 1024 x 5120: 823 -> 635 us, 5120 x 4096 x 1024: 758 ->
// 661 us with the branch-free loop, the unaligned vector loads, the tile order and the
// tile rule below); for small ones the latency of a slab (852 x 213 x 1065 in FP32: 37 ->
// 13.6 us).  Lane layouts of the 16x16x4 instructions:
//   A operand: lane l holds A[l%16][l/16]    B operand: lane l holds B[l/16][l%16]
//   D (f32):   lane l, item r holds D[4*(l/16)+r][l%16]
//   D (f64):   lane l, item r holds D[l/16+4*r][l%16]
// BF16: v_mfma_f32_16x16x32_bf16 -- A: lane l holds A[l%16][8*(l/16)+j], j<8;
// B: B[8*(l/16)+j][l%16]; D as above.  LDS holds K-contiguous rows so every
// fragment is one 16-byte LDS read.
#include "internal.h"
#include <type_traits>

namespace nsmi {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned short us8 __attribute__((ext_vector_type(8)));

template <typename T> struct Acc;
template <> struct Acc<double> { typedef d4 type; };
template <> struct Acc<float> { typedef f4 type; };

__device__ inline d4 mfma16(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline f4 mfma16(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Row of item r of lane group kl = lane/16 in a 16x16 MFMA result block
// (measured on gfx950): f64 16x16x4 interleaves rows kl + 4r; f32 16x16x4
// and bf16 16x16x32 hold four consecutive rows 4*kl + r.
template <typename T> __device__ inline int out_row(int kl, int r);
template <> __device__ inline int out_row<double>(int kl, int r) { return kl + 4 * r; }
template <> __device__ inline int out_row<float>(int kl, int r) { return 4 * kl + r; }

// T: the MFMA arithmetic type; TBm / TCm: how B and C are stored (a double B is
// rounded to T as it is staged, a double C takes the T accumulator widened), so a
// FP32 product can read an FP64 operand and write an FP64 result without
// conversion passes.
template <typename T, typename TBm = T, typename TCm = T>
struct GemmArgs {
  const T* A;
  const TBm* B;
  TCm* C;
  int64_t M, N, K, lda, ldb, ldc, sA, sB, sC;
  T alpha, beta;
  int tiles_m, tiles_n;
  // split-K: workgroup (tile, s) covers K in [s * kc, s * kc + kc); with part set it
  // writes its raw sum to part[s][M][N] and k_splitk_reduce forms C
  int64_t kc;
  T* part;
};

// XCD-aware tile order: consecutive workgroup ids are dealt round-robin to the 8 XCDs, so
// remap them such that each XCD works on a contiguous band of tiles (the first nwg % 8
// XCDs take one tile more).
__device__ inline int xcd_remap(int wg, int nwg) {
  constexpr int kXcd = 8;
  const int xcd = wg % kXcd;
  return xcd * (nwg / kXcd) + min(xcd, nwg % kXcd) + wg / kXcd;
}
// The band walks blocks of 8 tile rows column by column, so that the tiles an XCD
// has in flight (32 or 64) share as many A rows as B columns in its L2; row by row, each
// tile row read all of B again (5120 x 4096 x 1024: 669 -> 661 us; 32 x 32 tiles, 73 -> 58
// us at 2130 x 639 x 852 transposed).
__device__ inline void tile_of(int tile, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int kTileRows = 8;
  const int grp = min(kTileRows, tiles_m) * tiles_n;  // at most the launch's workgroups
  const int gi = tile / grp, rest = tile % grp;
  const int gh = min(kTileRows, tiles_m - gi * kTileRows);
  tm = gi * kTileRows + rest % gh;
  tn = rest / gh;
}

// Staging of one operand (X = A, rows m; or B, rows n): KC when X is K-contiguous in
// global memory (A not transposed, B transposed).  Then its LDS slab is row-major
// [R][BK + KP] (K contiguous), so the global->LDS copy keeps each thread's run of
// consecutive k contiguous on both sides (no transposing stores, which conflicted on
// the LDS banks), and the MFMA fragments are read as vectors: within a slab the
// k-step ks of lane (row ml, group kl) takes k = kl * (BK / 4) + ks (any fixed
// assignment of the slab's k to the four lane groups gives the same sum, as long as
// A and B use the same one), so a lane's BK / 4 values for the slab are contiguous.
// Otherwise the slab is [BK][R + 4] (row contiguous) and a fragment is one element
// per k-step at row kl * (BK / 4) + ks.  Each thread copies E consecutive elements of
// the slab (along k when KC, along the row otherwise) with 16-byte loads; these need only
// the element's alignment, so odd leading dimensions take them too (a quarter of the
// loads of the element-wise form that such matrices took before, which also tested every
// element's bounds).  A row past the matrix reads the last row instead: it reaches only
// rows (columns) of C that are not written.  Only a slab past K's end (the last) and, for
// a row-contiguous operand, a tile past the last row go element by element.
template <typename T>
struct Vec16 {  // 16 bytes at element alignment
  typedef T type __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};
template <typename T, typename TM, int R, int BK, int NT, bool KC>
struct Stage {
  static constexpr int E = R * BK / NT;
  static constexpr int KP = 16 / int(sizeof(T));       // keeps K-contiguous rows 16-byte aligned
  static constexpr int LD = KC ? BK + KP : R + 4;        // LDS row pitch (elements)
  static constexpr int ROWS = KC ? R : BK;
  // element (row r, k) of the slab -> LDS index
  __device__ static int at(int r, int k) { return KC ? r * LD + k : k * LD + r; }
  // thread's run: first (row, k) of its E consecutive elements
  __device__ static void run(int tid, int& r, int& k) {
    const int e = tid * E;
    if (KC) {
      r = e / BK;
      k = e % BK;
    } else {
      k = e / R;
      r = e % R;
    }
  }
  // the run's place in X, X(row, k) = KC ? X[row * ld + k] : X[k * ld + row]: its address at
  // slab 0 and the step from slab to slab
  struct Src {
    const TM* p;
    int64_t step, gr, gk;
  };
  __device__ static Src source(const TM* __restrict__ X, int64_t ld, int64_t r0, int64_t k0, int64_t rows) {
    int r, k;
    run(threadIdx.x, r, k);
    Src s;
    s.gr = KC ? min(r0 + r, rows - 1) : r0 + r;
    s.gk = k0 + k;
    s.p = KC ? X + s.gr * ld + s.gk : X + s.gk * ld + s.gr;
    s.step = KC ? BK : BK * ld;
    return s;
  }
  // slab kt entirely inside K; INR: the run's rows are inside (always when KC)
  template <bool INR>
  __device__ static void load(const Src& s, int64_t kt, int64_t rows, T (&reg)[E]) {
    const TM* const p = s.p + kt * s.step;
    if constexpr (KC || INR) {
      constexpr int V = 16 / int(sizeof(TM));
      static_assert(E % V == 0, "run length");
#pragma unroll
      for (int v = 0; v < E / V; ++v) {
        const typename Vec16<TM>::type q = *reinterpret_cast<const typename Vec16<TM>::type*>(p + v * V);
#pragma unroll
        for (int j = 0; j < V; ++j) reg[v * V + j] = T(q[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < E; ++j) reg[j] = T(p[min(s.gr + j, rows - 1) - s.gr]);
    }
  }
  // the slab that K ends in (kt * BK + the first slab's k < kend): its elements as they are
  // stored, those past the end repeat the last one; store_last puts zeros there
  __device__ static void load_last(const Src& s, int64_t kt, int64_t rows, int64_t kend, int64_t ld, TM (&raw)[E]) {
    const int64_t k = s.gk + kt * BK;
    const TM* const base = s.p + kt * s.step;
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const int64_t kc = min(KC ? k + j : k, kend - 1);
      raw[j] = KC ? base[kc - k] : base[(kc - k) * ld + (min(s.gr + j, rows - 1) - s.gr)];
    }
  }
  __device__ static void store_last(T* __restrict__ sh, const Src& s, int64_t kt, int64_t kend, const TM (&raw)[E]) {
    const int64_t k = s.gk + kt * BK;
    T reg[E];
#pragma unroll
    for (int j = 0; j < E; ++j) reg[j] = (KC ? k + j : k) < kend ? T(raw[j]) : T(0);
    store(sh, reg);
  }
  __device__ static void store(T* __restrict__ s, const T (&reg)[E]) {
    int r, k;
    run(threadIdx.x, r, k);
#pragma unroll
    for (int j = 0; j < E; ++j) s[KC ? at(r, k + j) : at(r + j, k)] = reg[j];
  }
};

// NW waves: 4 as 2 x 2, or 8 as 2 x 4 (the 128 x 128 tile: half the accumulators per
// wave, so that two waves share each SIMD and hide each other's latency)
template <typename T, typename TBm, typename TCm, int BM, int BN, bool TA, bool TB, int ROLE, int NW>
__global__ __launch_bounds__(64 * NW) void k_gemm_mfma(GemmArgs<T, TBm, TCm> g) {
  // the small tiles run twice as deep a K slice per LDS stage: the products they
  // serve have few tiles and long K, so the per-stage barrier and load latency is
  // what they pay (measured on the FP32 H_eff GEMM2 at 852 x 213 x 1065 with loads one
  // slab ahead: 38.8 us at depth 16, 27.7 us at 32, 30.8 us at 64)
  constexpr int BK = (BM == 32 && BN == 32) ? 32 : 16;
  constexpr int NT = 64 * NW, GM = 2, GN = NW / 2;
  constexpr int WTM = BM / GM, WTN = BN / GN;
  constexpr int FM = WTM / 16, FN = WTN / 16, KS = BK / 4;
  typedef Stage<T, T, BM, BK, NT, !TA> SA;
  typedef Stage<T, TBm, BN, BK, NT, TB> SB;
  typedef typename Acc<T>::type AccT;
  __shared__ __align__(16) T sA[2][SA::ROWS * SA::LD];
  __shared__ __align__(16) T sB[2][SB::ROWS * SB::LD];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / GN, wn = wave % GN;
  const int nwg = g.tiles_m * g.tiles_n;
  const int tile = xcd_remap(blockIdx.x, nwg);
  int tm, tn;
  tile_of(tile, g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
  const int64_t bz = blockIdx.z;
  const int64_t kb = int64_t(blockIdx.y) * g.kc;
  const int64_t ke = min(g.K, kb + g.kc);
  const T* __restrict__ A = g.A + bz * g.sA;
  const TBm* __restrict__ B = g.B + bz * g.sB;
  TCm* __restrict__ C = g.C + bz * g.sC;
  const auto src_a = SA::source(A, g.lda, m0, kb, g.M);
  const auto src_b = SB::source(B, g.ldb, n0, kb, g.N);

  AccT acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = AccT{0, 0, 0, 0};

  const int kl = lane >> 4, ml = lane & 15;
  const auto mma = [&](int buf) {
    // the slab's fragments: lane (ml, kl) at k-step ks holds k = kl * KS + ks
    T af[FM][KS], bf[FN][KS];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = wm * WTM + i * 16 + ml;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) af[i][ks] = sA[buf][SA::at(r, kl * KS + ks)];
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int r = wn * WTN + j * 16 + ml;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) bf[j][ks] = sB[buf][SB::at(r, kl * KS + ks)];
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(af[i][ks], bf[j][ks], acc[i][j]);
  };
  const int64_t nfull = (ke - kb) / BK;  // slabs entirely inside K
  // The whole slabs, loads two slabs ahead (two register sets, two LDS buffers, one barrier
  // per slab).  Past the end the slab index stays at the last one: those loads and
  // stores land in registers and buffers that no later step uses, and the loop has no
  // branches.  The slab that K ends in is loaded with the first ones: loaded after the loop it
  // cost a small product one more round trip (1.5 of 20 us for an environment update at
  // bonds of 20).
  const bool tail = nfull * BK < ke - kb;
  T tail_a[SA::E];
  TBm tail_b[SB::E];
  const auto load_tail = [&]() {
    if (tail) {
      SA::load_last(src_a, nfull, g.M, ke, g.lda, tail_a);
      SB::load_last(src_b, nfull, g.N, ke, g.ldb, tail_b);
    }
  };
  const auto whole = [&](auto in_m, auto in_n) {
    T ra[2][SA::E], rb[2][SB::E];
    const auto load = [&](int64_t kt, T (&xa)[SA::E], T (&xb)[SB::E]) {
      SA::template load<decltype(in_m)::value>(src_a, kt, g.M, xa);
      SB::template load<decltype(in_n)::value>(src_b, kt, g.N, xb);
    };
    const int64_t last = nfull - 1;
    load(0, ra[0], rb[0]);
    load_tail();
    SA::store(sA[0], ra[0]);
    SB::store(sB[0], rb[0]);
    load(min(int64_t(1), last), ra[1], rb[1]);
    __syncthreads();
    const auto step = [&](auto set, int64_t kt) {
      constexpr int S = decltype(set)::value;
      load(min(kt + 2, last), ra[S], rb[S]);
      mma(S);
      SA::store(sA[S ^ 1], ra[S ^ 1]);
      SB::store(sB[S ^ 1], rb[S ^ 1]);
      __syncthreads();
    };
    int64_t kt = 0;
    for (; kt + 1 < nfull; kt += 2) {
      step(std::integral_constant<int, 0>{}, kt);
      step(std::integral_constant<int, 1>{}, kt + 1);
    }
    if (kt < nfull) step(std::integral_constant<int, 0>{}, kt);
  };
  if (nfull > 0) {
    using Yes = std::integral_constant<bool, true>;
    using No = std::integral_constant<bool, false>;
    const bool in_m = !TA || m0 + BM <= g.M, in_n = TB || n0 + BN <= g.N;
    if (in_m && in_n)
      whole(Yes{}, Yes{});
    else
      whole(No{}, No{});
  } else {
    load_tail();
  }
  if (tail) {
    SA::store_last(sA[0], src_a, nfull, ke, tail_a);
    SB::store_last(sB[0], src_b, nfull, ke, tail_b);
    __syncthreads();
    mma(0);
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t gm = m0 + wm * WTM + i * 16 + out_row<T>(kl, r);
        const int64_t gn = n0 + wn * WTN + j * 16 + ml;
        if (BM == 32 && BN == 32 && g.part) {  // only this tile splits K
          if (gm < g.M && gn < g.N) g.part[(int64_t(blockIdx.y) * g.M + gm) * g.N + gn] = acc[i][j][r];
        } else if (gm < g.M && gn < g.N) {
          T v = g.alpha * acc[i][j][r];
          if (g.beta != T(0)) v += g.beta * T(C[gm * g.ldc + gn]);
          C[gm * g.ldc + gn] = TCm(v);
        }
      }
}

// C = alpha * sum_s part[s] + beta * C, the splits added in ascending s (in FP64),
// so the result does not depend on the order in which the split workgroups ran
template <typename T, typename TCm>
__global__ __launch_bounds__(256) void k_splitk_reduce(const T* __restrict__ part, TCm* __restrict__ C, int64_t M,
                                                       int64_t N, int64_t ldc, int S, T alpha, T beta) {
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= M * N) return;
  double acc = 0.0;
  for (int s = 0; s < S; ++s) acc += double(part[int64_t(s) * M * N + e]);
  const int64_t m = e / N, n = e % N;
  double v = double(alpha) * acc;
  if (beta != T(0)) v += double(beta) * double(C[m * ldc + n]);
  C[m * ldc + n] = TCm(v);
}

// The same product for grids too small to fill the chip, where a tile's serial chain of
// slabs (load, barrier, MFMA) is the whole time: one 16 x 16 block of C per workgroup, K
// dealt to its 8 waves in chunks of 16 (lane group kl takes k = 4 kl .. 4 kl + 3 of a chunk: 16-byte
// loads of a K-contiguous operand), operands straight from memory into the MFMA registers
// (every element of a block's rows is used once: LDS would add a barrier per slab and
// share nothing), three chunks in flight per wave, and the 8 partial sums added in wave
// order through LDS.  No partial sums in memory and no second launch, as a split over K has.
template <typename T, typename TM, bool KC>
struct WaveOperand {
  const TM* p;  // element (row, k = 4 kl)
  int64_t ld, k0;
  __device__ WaveOperand(const TM* __restrict__ X, int64_t ld_, int64_t row, int kl)
      : p(KC ? X + row * ld_ + 4 * kl : X + 4 * kl * ld_ + row), ld(ld_), k0(4 * kl) {}
  __device__ void load(int64_t c, T (&reg)[4]) const {
    const TM* const q = p + (KC ? c * 16 : c * 16 * ld);
    if constexpr (KC) {
      constexpr int V = 16 / int(sizeof(TM));
#pragma unroll
      for (int v = 0; v < 4 / V; ++v) {
        const typename Vec16<TM>::type x = *reinterpret_cast<const typename Vec16<TM>::type*>(q + v * V);
#pragma unroll
        for (int j = 0; j < V; ++j) reg[v * V + j] = T(x[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) reg[j] = T(q[j * ld]);
    }
  }
  __device__ void load_last(int64_t c, int64_t K, T (&reg)[4]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t k = c * 16 + k0 + j, kc = min(k, K - 1) - k0;
      const T v = T(p[KC ? kc : kc * ld]);
      reg[j] = k < K ? v : T(0);
    }
  }
};

template <typename T, typename TBm, typename TCm, bool TA, bool TB, int ROLE>
__global__ __launch_bounds__(512) void k_gemm_wave(GemmArgs<T, TBm, TCm> g) {
  typedef typename Acc<T>::type AccT;
  constexpr int NW = 8, D = 3;
  __shared__ T part[NW][4][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kl = lane >> 4, ml = lane & 15;
  int tm, tn;
  tile_of(xcd_remap(blockIdx.x, g.tiles_m * g.tiles_n), g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = int64_t(tm) * 16, n0 = int64_t(tn) * 16, bz = blockIdx.z;
  // rows and columns past the matrix repeat the last one: they reach only elements of C
  // that are not written
  const WaveOperand<T, T, !TA> oa(g.A + bz * g.sA, g.lda, min(m0 + ml, g.M - 1), kl);
  const WaveOperand<T, TBm, TB> ob(g.B + bz * g.sB, g.ldb, min(n0 + ml, g.N - 1), kl);
  AccT acc = AccT{0, 0, 0, 0};
  const auto mma = [&](const T (&a)[4], const T (&b)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = mfma16(a[u], b[u], acc);
  };
  const int64_t nfull = g.K / 16;
  T a[D][4], b[D][4];
  if (wave < nfull) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int64_t c = min(int64_t(wave + d * NW), nfull - 1);
      oa.load(c, a[d]);
      ob.load(c, b[d]);
    }
  }
  for (int64_t c0 = wave; c0 < nfull; c0 += D * NW)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (c0 + d * NW >= nfull) break;
      mma(a[d], b[d]);
      const int64_t c = min(c0 + (d + D) * NW, nfull - 1);
      oa.load(c, a[d]);
      ob.load(c, b[d]);
    }
  if (nfull * 16 < g.K && wave == nfull % NW) {
    oa.load_last(nfull, g.K, a[0]);
    ob.load_last(nfull, g.K, b[0]);
    mma(a[0], b[0]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[wave][r][lane] = acc[r];
  __syncthreads();
  if (tid >= 256) return;
  // waves 0..3 write item r = wave of every lane; as in k_splitk_reduce the partial sums of
  // a split K are added and scaled in FP64 and rounded once, to C's type
  double sum = 0.0;
#pragma unroll
  for (int w = 0; w < NW; ++w) sum += double(part[w][wave][lane]);
  const int64_t gm = m0 + out_row<T>(kl, wave), gn = n0 + ml;
  if (gm >= g.M || gn >= g.N) return;
  TCm* const C = g.C + bz * g.sC;
  double v = double(g.alpha) * sum;
  if (g.beta != T(0)) v += double(g.beta) * double(C[gm * g.ldc + gn]);
  C[gm * g.ldc + gn] = TCm(v);
}

// number of K splits of the 32 x 32 tile: only for single products whose tile grid leaves most
// CUs idle and whose K is long; each split keeps at least four K stages.  (The larger tiles
// are taken from 205 and 448 of them on, where there is nothing to split.)
constexpr int kSplitBk = 32;
inline int splitk_count(const GemmDesc& d, int64_t tiles) {
  if (d.batch != 1 || tiles >= 128) return 1;
  const int64_t stages = (d.K + kSplitBk - 1) / kSplitBk;
  const int64_t by_grid = 512 / tiles, by_k = stages / 4;
  return int(std::max<int64_t>(1, std::min<int64_t>({by_grid, by_k, int64_t(8)})));
}

template <typename T, typename TBm, typename TCm, int BM, int BN, int ROLE>
void launch_tile(nsmi_ctx* ctx, const GemmDesc& d, GemmArgs<T, TBm, TCm>& a) {
  constexpr bool kSplit = BM == 32 && BN == 32;
  a.tiles_m = int((d.M + BM - 1) / BM);
  a.tiles_n = int((d.N + BN - 1) / BN);
  const int S = kSplit ? splitk_count(d, int64_t(a.tiles_m) * a.tiles_n) : 1;
  a.kc = S == 1 ? std::max<int64_t>(d.K, 1) : ((d.K + S - 1) / S + kSplitBk - 1) / kSplitBk * kSplitBk;
  const int splits = int((d.K + a.kc - 1) / a.kc);
  std::unique_ptr<Scratch> part;
  a.part = nullptr;
  if (splits > 1) {
    const size_t need = sizeof(T) * size_t(splits) * size_t(d.M) * size_t(d.N);
    if (ctx->fixed_part) {
      if (need > ctx->fixed_part_bytes)
        fail(NSMI_ERR_INVALID, "gemm: the split-K partial sums need " + std::to_string(need) +
                                   " B, above the no-allocation scratch of " + std::to_string(ctx->fixed_part_bytes) +
                                   " B");
      a.part = static_cast<T*>(ctx->fixed_part);
    } else {
      part.reset(new Scratch(ctx, need));
      a.part = part->as<T>();
    }
  }
  constexpr int NW = (BM == 128 && BN == 128) ? 8 : 4;
  dim3 grid(unsigned(a.tiles_m) * unsigned(a.tiles_n), unsigned(std::max(splits, 1)), unsigned(d.batch));
  dim3 block(64 * NW);
  // with a split the product's timed span runs from the start of the MFMA kernel to
  // the end of the reduction
#define NSMI_GEMM_GO(KER)                                                           \
  do {                                                                              \
    if (a.part) NSMI_LAUNCH_TIMED_FIRST(ctx, KER, grid, block, a);                  \
    else NSMI_LAUNCH_TIMED(ctx, KER, grid, block, a);                               \
  } while (0)
  if (!d.transA && !d.transB)
    NSMI_GEMM_GO((k_gemm_mfma<T, TBm, TCm, BM, BN, false, false, ROLE, NW>));
  else if (!d.transA && d.transB)
    NSMI_GEMM_GO((k_gemm_mfma<T, TBm, TCm, BM, BN, false, true, ROLE, NW>));
  else if (d.transA && !d.transB)
    NSMI_GEMM_GO((k_gemm_mfma<T, TBm, TCm, BM, BN, true, false, ROLE, NW>));
  else
    NSMI_GEMM_GO((k_gemm_mfma<T, TBm, TCm, BM, BN, true, true, ROLE, NW>));
#undef NSMI_GEMM_GO
  NSMI_LAUNCH_CHECK();
  if (a.part) {
    const int64_t n = d.M * d.N;
    NSMI_LAUNCH_TIMED_LAST(ctx, (k_splitk_reduce<T, TCm>), dim3(unsigned((n + 255) / 256)), dim3(256), a.part, a.C,
                           d.M, d.N, d.ldc, splits, a.alpha, a.beta);
    NSMI_LAUNCH_CHECK();
  }
}

template <typename T, typename TBm, typename TCm, int ROLE>
void launch_wave(nsmi_ctx* ctx, const GemmDesc& d, GemmArgs<T, TBm, TCm>& a) {
  a.tiles_m = int((d.M + 15) / 16);
  a.tiles_n = int((d.N + 15) / 16);
  const dim3 grid(unsigned(a.tiles_m) * unsigned(a.tiles_n), 1, unsigned(d.batch)), block(512);
  if (!d.transA && !d.transB)
    NSMI_LAUNCH_TIMED(ctx, (k_gemm_wave<T, TBm, TCm, false, false, ROLE>), grid, block, a);
  else if (!d.transA && d.transB)
    NSMI_LAUNCH_TIMED(ctx, (k_gemm_wave<T, TBm, TCm, false, true, ROLE>), grid, block, a);
  else if (d.transA && !d.transB)
    NSMI_LAUNCH_TIMED(ctx, (k_gemm_wave<T, TBm, TCm, true, false, ROLE>), grid, block, a);
  else
    NSMI_LAUNCH_TIMED(ctx, (k_gemm_wave<T, TBm, TCm, true, true, ROLE>), grid, block, a);
  NSMI_LAUNCH_CHECK();
}

// whether tiles of TS x TS leave at most a fifth of the last round over the 256 CUs (and of
// the edge tiles) unused
template <int TS>
bool tiles_fill(const GemmDesc& d) {
  const int64_t tiles = ((d.M + TS - 1) / TS) * ((d.N + TS - 1) / TS) * d.batch;
  const int64_t rounds = (tiles + 255) / 256;
  return double(d.M) * double(d.N) * double(d.batch) >= 0.8 * (double(TS) * TS * 256.0) * double(rounds);
}

// The 128 x 128 tile (one workgroup per CU in FP64) only where its rounds are full: it
// reaches 66 TF/s at 2048 x 2048 x 1024 (32 x 32: 54-56), loses at 3072 x 3072 x 1024 (75%
// full: 377 us against 345) and at 1536 x 1536 x 1024 (56%: 127 against 93).  Everywhere
// else the 32 x 32 tile, whose deep slabs and many workgroups hide the latency: in FP64 it
// is never behind 64 x 64 by more than the runs differ (1024 x 1024 x 1024: 44 us against
// 50-55; 1536 x 1536 x 1024: 93 against 115-138), which is therefore not built for FP64.
// In FP32 64 x 64 wins from about two full rounds (1536 x 1280 x 1024: 40 us against 45;
// 2176 x 2176 x 1024: 94 against 108) and loses before (1024 x 1024 x 1024: 26 against 24).
// Up to 64 tiles of 32 x 32 the wave form, while K is short enough for its uncoalesced reads
// (512 in FP64, 1024 in FP32); us, wave form / 32 x 32 with its split: FP64 60, 60, 60: 3.5 /
// 4.4; 394, 64, 394: 5.5-6.1 / 8.2; 400, 100, 500: 6.5 / 8.7; FP32 64, 64, 1024: 5.4-7.0 / 7.9;
// 400, 100, 500: 4.4 / 7.6.  It loses at more tiles (FP64 320, 256, 64, 80 tiles: 5.2 / 4.1;
// 384, 384, 384: 11-18 / 8.7) and longer K (FP64 64, 64, 1024: 7.4-11.9 / 9.0; 64, 200, 2048:
// 11-19 / 10.8).
template <typename T, typename TBm, typename TCm, int ROLE>
void launch_role(nsmi_ctx* ctx, const GemmDesc& d, GemmArgs<T, TBm, TCm>& a) {
  if (((d.M + 31) / 32) * ((d.N + 31) / 32) * d.batch <= 64 && d.K <= 4096 / int64_t(sizeof(T)))
    return launch_wave<T, TBm, TCm, ROLE>(ctx, d, a);
  if (tiles_fill<128>(d)) return launch_tile<T, TBm, TCm, 128, 128, ROLE>(ctx, d, a);
  if constexpr (sizeof(T) == 4) {
    const int64_t mid = ((d.M + 63) / 64) * ((d.N + 63) / 64) * d.batch;
    if (mid >= 448 && tiles_fill<64>(d)) return launch_tile<T, TBm, TCm, 64, 64, ROLE>(ctx, d, a);
  }
  launch_tile<T, TBm, TCm, 32, 32, ROLE>(ctx, d, a);
}

template <typename T>
void gemm_generic(nsmi_ctx* ctx, const GemmDesc& d, T alpha, const T* A, const T* B, T beta, T* C, int role) {
  require(d.M >= 0 && d.N >= 0 && d.K >= 0 && d.batch >= 1, "gemm: bad sizes");
  require(d.tiles_ok(), "gemm: too many tiles");
  if (d.M == 0 || d.N == 0) return;
  GemmArgs<T> a{A, B, C, d.M, d.N, d.K, d.lda, d.ldb, d.ldc, d.sA, d.sB, d.sC, alpha, beta, 0, 0, 0, nullptr};
  switch (role) {
    case kRoleHeff1: launch_role<T, T, T, kRoleHeff1>(ctx, d, a); break;
    case kRoleHeff2: launch_role<T, T, T, kRoleHeff2>(ctx, d, a); break;
    case kRoleEnv: launch_role<T, T, T, kRoleEnv>(ctx, d, a); break;
    case kRoleTheta: launch_role<T, T, T, kRoleTheta>(ctx, d, a); break;
    default: launch_role<T, T, T, kRoleFact>(ctx, d, a); break;
  }
}

}  // namespace

bool GemmDesc::tiles_ok() const {
  const int64_t t = ((M + 63) / 64) * ((N + 63) / 64);
  return t < (int64_t(1) << 30) && batch < 65536;
}

void gemm_f64(nsmi_ctx* ctx, const GemmDesc& g, double alpha, const double* A, const double* B, double beta,
              double* C, int role) {
  gemm_generic<double>(ctx, g, alpha, A, B, beta, C, role);
}

void gemm_f32(nsmi_ctx* ctx, const GemmDesc& g, const float* A, const float* B, float* C, int role) {
  gemm_generic<float>(ctx, g, 1.0f, A, B, 0.0f, C, role);
}

void gemm_f32_heff1_bd(nsmi_ctx* ctx, const GemmDesc& d, const float* A, const double* B, float* C) {
  require(d.M >= 0 && d.N >= 0 && d.K >= 0 && d.batch >= 1 && d.tiles_ok(), "gemm: bad sizes");
  if (d.M == 0 || d.N == 0) return;
  GemmArgs<float, double, float> a{A,    B,    C,    d.M,  d.N, d.K, d.lda,  d.ldb,
                                   d.ldc, d.sA, d.sB, d.sC, 1.0f, 0.0f, 0, 0, 0, nullptr};
  launch_role<float, double, float, kRoleHeff1>(ctx, d, a);
}

void gemm_f32_heff2_cd(nsmi_ctx* ctx, const GemmDesc& d, const float* A, const float* B, double* C) {
  require(d.M >= 0 && d.N >= 0 && d.K >= 0 && d.batch >= 1 && d.tiles_ok(), "gemm: bad sizes");
  if (d.M == 0 || d.N == 0) return;
  GemmArgs<float, float, double> a{A,    B,    C,    d.M,  d.N, d.K, d.lda,  d.ldb,
                                   d.ldc, d.sA, d.sB, d.sC, 1.0f, 0.0f, 0, 0, 0, nullptr};
  launch_role<float, float, double, kRoleHeff2>(ctx, d, a);
}

}  // namespace nsmi

// ---------------------------------------------------------------------------
// BF16 MFMA GEMM, "NT" form: C[M x N] = sum_t A_t[M x Kp] . B_t[N x Kp]^T with
// both operands K-contiguous bf16 planes (row pitch Kp, Kp % 32 == 0, padding
// zero).  TERMS == 3 computes Ahi.Bhi + Ahi.Blo + Alo.Bhi (bf16x3 split
// products, FP32 accumulation); TERMS == 1 computes Ahi.Bhi.
// K slab 32 (one MFMA k-step), LDS rows padded to 80 bytes so the 16 lanes of each
// quarter-wave hit 16 distinct 4-bank groups on their 16-byte fragment reads.
// ---------------------------------------------------------------------------
namespace nsmi {
namespace {

struct BfArgs {
  const uint16_t *Ahi, *Alo, *Bhi, *Blo;
  void* C;
  int64_t M, N, Kp, lda, ldb, ldc;
  int tiles_m, tiles_n;
};

typedef unsigned int u4 __attribute__((ext_vector_type(4)));

// TS x TS tiles: 128 with 8 waves (2 x 4, each 64 x 32), 64 with 4 (2 x 2, 32 x 32), 32 with 2
// (1 x 2, 32 x 16); each thread stages one 16-byte chunk per plane and operand in all three
template <int TS, int TERMS, typename TC, int ROLE>
__global__ __launch_bounds__(TS * 4) void k_gemm_bf16_nt(BfArgs g) {
  constexpr int BM = TS, BN = TS, BK = 32, PITCH = BK + 8;  // in bf16 elements
  constexpr int WM = TS == 32 ? 1 : 2, WN = TS == 128 ? 4 : 2, WTM = BM / WM, WTN = BN / WN;
  constexpr int FM = WTM / 16, FN = WTN / 16;
  constexpr int NP = (TERMS == 3) ? 2 : 1;                     // planes per operand
  __shared__ __attribute__((aligned(16))) uint16_t sA[2][NP][BM][PITCH];
  __shared__ __attribute__((aligned(16))) uint16_t sB[2][NP][BN][PITCH];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;
  int tm, tn;
  tile_of(xcd_remap(blockIdx.x, g.tiles_m * g.tiles_n), g.tiles_m, g.tiles_n, tm, tn);
  const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;

  // each thread stages the 16-byte chunk tid % 4 of row tid / 4 of every tile plane
  // (a row's 64 bytes come from four neighbouring lanes).  Rows past M (N) read row
  // M - 1 (N - 1) instead: A's row m only reaches C's row m (B's row n only C's
  // column n), and those are not written, so no zero fill is needed and the K loop
  // has no branches (a branch there makes the compiler copy the accumulators between
  // AGPRs and VGPRs on every step).
  const int lr = tid >> 2, lc = (tid & 3) * 8;
  const int64_t ra_row = min(m0 + lr, g.M - 1), rb_row = min(n0 + lr, g.N - 1);
  const uint16_t* pa[2] = {g.Ahi + ra_row * g.lda + lc, TERMS == 3 ? g.Alo + ra_row * g.lda + lc : nullptr};
  const uint16_t* pb[2] = {g.Bhi + rb_row * g.ldb + lc, TERMS == 3 ? g.Blo + rb_row * g.ldb + lc : nullptr};
  u4 ra[NP], rb[NP];
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      ra[p] = *reinterpret_cast<const u4*>(pa[p] + k0);
      rb[p] = *reinterpret_cast<const u4*>(pb[p] + k0);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      *reinterpret_cast<u4*>(&sA[buf][p][lr][lc]) = ra[p];
      *reinterpret_cast<u4*>(&sB[buf][p][lr][lc]) = rb[p];
    }
  };

  f4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f4{0, 0, 0, 0};

  // two fragment sets in registers: the MFMAs of K-step kt use set kt & 1 while
  // the fragments of step kt + 1 are read from the other LDS buffer
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  bf8 fa[2][NP][FM], fb[2][NP][FN];
  auto frag = [&](auto set_c, int buf) {
    constexpr int S = decltype(set_c)::value;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
        fa[S][p][i] = *reinterpret_cast<const bf8*>(&sA[buf][p][wm * WTM + i * 16 + fr][fk]);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        fb[S][p][j] = *reinterpret_cast<const bf8*>(&sB[buf][p][wn * WTN + j * 16 + fr][fk]);
    }
  };
  auto mma = [&](auto set_c) {
    constexpr int S = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if constexpr (TERMS == 3) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[S][1][i], fb[S][0][j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[S][0][i], fb[S][1][j], acc[i][j], 0, 0, 0);
        }
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[S][0][i], fb[S][0][j], acc[i][j], 0, 0, 0);
      }
  };
  // K-step kt: global loads of slab kt + 2, LDS reads of step kt + 1's fragments
  // (buffer (kt + 1) & 1, stored before the last barrier), MFMAs of step kt, then
  // slab kt + 2 into buffer kt & 1, whose fragments every wave read before that
  // barrier.  Past the end the slab index stays at nk - 1: those loads, stores and
  // fragment reads land in buffers and registers that no later step uses.
  const int64_t nk = g.Kp / BK;
  auto step = [&](auto set_c, int64_t kt) {
    constexpr int S = decltype(set_c)::value;
    const int buf = int(kt & 1);
    load(min(kt + 2, nk - 1) * BK);
    frag(std::integral_constant<int, S ^ 1>{}, buf ^ 1);
    // keeps the scheduler from sinking the reads into the MFMA block (it would
    // trade the overlap for registers) ...
    __builtin_amdgcn_sched_barrier(0);
    mma(set_c);
    // ... and the LDS stores (which wait for the global loads) out of it
    __builtin_amdgcn_sched_barrier(0);
    store(buf);
    __syncthreads();
  };
  load(0);
  store(0);
  load(min(int64_t(1), nk - 1) * BK);
  store(1);
  __syncthreads();
  frag(std::integral_constant<int, 0>{}, 0);
  int64_t kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    step(std::integral_constant<int, 0>{}, kt);
    step(std::integral_constant<int, 1>{}, kt + 1);
  }
  if (kt < nk) mma(std::integral_constant<int, 0>{});
  TC* C = static_cast<TC*>(g.C);
  const int kl = lane >> 4;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t gm = m0 + wm * WTM + i * 16 + 4 * kl + r;  // bf16 16x16x32: rows 4*(l/16)+r
        const int64_t gn = n0 + wn * WTN + j * 16 + fr;
        if (gm < g.M && gn < g.N) C[gm * g.ldc + gn] = TC(acc[i][j][r]);
      }
}

template <int TS, int TERMS, typename TC>
void bf16_role(nsmi_ctx* ctx, int role, BfArgs& a) {
  a.tiles_m = int((a.M + TS - 1) / TS);
  a.tiles_n = int((a.N + TS - 1) / TS);
  const dim3 grid(unsigned(a.tiles_m) * unsigned(a.tiles_n)), block(TS * 4);
  switch (role) {
    case kRoleHeff1: NSMI_LAUNCH_TIMED(ctx, (k_gemm_bf16_nt<TS, TERMS, TC, kRoleHeff1>), grid, block, a); break;
    case kRoleHeff2: NSMI_LAUNCH_TIMED(ctx, (k_gemm_bf16_nt<TS, TERMS, TC, kRoleHeff2>), grid, block, a); break;
    default: NSMI_LAUNCH_TIMED(ctx, (k_gemm_bf16_nt<TS, TERMS, TC, kRoleEnv>), grid, block, a); break;
  }
}

// 128 x 128 (one workgroup per CU) where its rounds over the CUs are full enough: the three-term
// product from 65% (3200 x 800 x 4000, 175 tiles: 106 us, 64 x 64 113; 3500 x 2800 x 700, 616: 65 / 71;
// but 2560 x 2048 x 512, 320: 34 / 29; 2800 x 700 x 3500, 132: 95 / 71), the single-term one from 75%
// (3000 x 2400 x 600, 456: 20 / 26; 3200 x 800 x 4000: 68 / 57).  Below it 64 x 64 while it has a tile
// per CU (2400 x 600 x 3000, 380 tiles: 59 us, 32 x 32 72; 2048 x 512 x 2560, 256: 40 / 43), else
// 32 x 32 (1556 x 421 x 2105, 175 tiles: 29 us, 64 x 64 34, 128 x 128 59; 800 x 200 x 1000: 10 / 14 / 28).
template <int TERMS, typename TC>
void bf16_tile(nsmi_ctx* ctx, int role, BfArgs& a) {
  const int64_t big = ((a.M + 127) / 128) * ((a.N + 127) / 128);
  const bool mid = ((a.M + 63) / 64) * ((a.N + 63) / 64) >= 256;
  if (100 * big >= (TERMS == 3 ? 65 : 75) * 256 * ((big + 255) / 256))
    bf16_role<128, TERMS, TC>(ctx, role, a);
  else if (mid)
    bf16_role<64, TERMS, TC>(ctx, role, a);
  else
    bf16_role<32, TERMS, TC>(ctx, role, a);
}

}  // namespace

void gemm_bf16_nt(nsmi_ctx* ctx, int64_t M, int64_t N, int64_t Kp, const uint16_t* Ahi, const uint16_t* Alo,
                  int64_t lda, const uint16_t* Bhi, const uint16_t* Blo, int64_t ldb, void* C, int64_t ldc,
                  bool c_double, int terms, int role) {
  require(Kp > 0 && Kp % 32 == 0 && lda % 8 == 0 && ldb % 8 == 0,
          "gemm_bf16: K must be positive and padded to 32, rows 16-byte aligned");
  require(terms == 1 || terms == 3, "gemm_bf16: terms must be 1 or 3");
  if (M == 0 || N == 0) return;
  BfArgs a{Ahi, Alo, Bhi, Blo, C, M, N, Kp, lda, ldb, ldc, 0, 0};
  if (terms == 3) {
    if (c_double) bf16_tile<3, double>(ctx, role, a);
    else bf16_tile<3, float>(ctx, role, a);
  } else {
    if (c_double) bf16_tile<1, double>(ctx, role, a);
    else bf16_tile<1, float>(ctx, role, a);
  }
  NSMI_LAUNCH_CHECK();
}

}  // namespace nsmi
