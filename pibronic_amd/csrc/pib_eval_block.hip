// FP64 evaluation with four bead streams per wave on 4 x 4 matrix blocks (A, A_rho <= 16).
//
// Same estimator as k_eval_fp64 (pibronic/pimc/pimc.py:1087-1213 fused; block loops
// :1341-1462) for surface counts whose A x A matrices do not fit one lane's registers. A matrix is
// NB x NB blocks of 4 x 4 (NB = ceil(max(A, A_rho) / 4)); one register pair of the wave holds one
// block of FOUR independent matrices, one per bead stream: lane 16 i + 4 b + j holds element
// (i, j) of stream b. That is the layout of v_mfma_f64_4x4x4_4b_f64 (measured on gfx950):
// results and B operands in it, A operands transposed, so for a symmetric factor
//   (X Y)_IK = sum_J mfma(X_JI, Y_JK):
// every product of the exponential chains in registers with no data movement. Only the blocks
// I <= K of a symmetric product are formed; the others are their transposes, mfma(Z_IK, 1)
// (A operands are read transposed), 7 instead of 8 instructions at NB = 2, 21 instead of 27 at 3.
//
// A stream is a sample (C = 1) or one of C = 2, 4 contiguous bead chunks of a sample (small
// launches). The wave takes four steps of its four streams at a time:
//  * front: the couplings and the O-exponents are contractions over the modes and run on the
//    FP64 matrix cores, v_mfma_f64_16x16x4_f64 with the 16 (stream, step) beads as columns, 16
//    matrix elements (or surfaces) as rows and four modes per instruction; the coefficient
//    operands come from a table laid out in operand order. X = -tau V is handed to the
//    4 x 4 layout through LDS (lower triangles; the reads mirror them).
//  * back: step by step, M = exp(X) by the scaled and squared degree-16 form of the per-lane
//    kernel, and the ring products R^T <- diag(O / S) M R^T of every chain (one, or three with
//    +-dbeta).
// Padding: rows and columns >= A of X are zero and the Taylor identity covers only the leading
// A x A block, so M is zero outside it; padded surfaces have log F = -inf, O = 0.
//
// Measured (MI355X, evaluation of 1e5 samples at A = 8, N = 16, P = 64, us): 1340 against 1650 for the
// per-lane kernel (one wave per SIMD, a third of its vector instructions moves to and from the
// accumulation registers); with +-dbeta 1800 against 5470 for three single-chain passes of that
// kernel. With +-dbeta at A = 12, N = 24, P = 128, 16,384 samples 1480 against 5720 for the
// one-wave-per-sample kernel; at A = 11, N = 17, P = 50, 3,001 samples 130 against 373.
//
// What bounds it: FP64 issue. On gfx950 the FP64 matrix and vector instructions share one pipe
// (timed together they add up exactly: 8 mfma_f64_4x4x4 + 32 v_fma_f64 take 311 cycles per SIMD,
// alone 152 and 174), so the kernel counts instructions of both kinds; per flop the matrix
// instructions are the cheaper ones (18.8 cycles per 4x4x4x4, 70 per 16x16x4, 5.4 per v_fma_f64). Memory
// does not: each step of four beads takes 16 (float offsets) or 32 bytes of a line, so lines come again
// (8.4 GB for 1.07 GB at 262,144 float offsets, 2.1 TB/s with the writes), and the registers below spill 72 to 84 bytes per
// lane at S = 8 (0.28 GB written in that launch, once per wave and four steps, outside the exponential),
// up to 36 at S <= 7, none to 20 at S = 9..12 and 380 to 444 at S = 13..16.
#include "pib_common.hpp"
#include "pib_ctx.hpp"
#include "pib_expm.hpp"
#include "pib_kernels.hpp"

namespace pib {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

// Sizes of the kernel for S surfaces (S = max(A, A_rho, 5)). The coupling matrices' lower-triangle
// elements are numbered off-diagonal first, r (r - 1) / 2 + c, then the diagonal, so that a linear
// coupling without diagonal (the folded models') needs only the first NTL tiles of 16 elements; a
// tile-per-block numbering would hold every diagonal block's off-diagonal elements twice. The
// operands of one mode group are the NL tiles of O-exponents, the tiles of the linear couplings,
// those of the quadratic ones, and the rest of the linear ones, in pairs (one 16-byte load).
template <int S, bool PM>
struct Geo {
  static constexpr int NB = (S + 3) / 4, SETS = PM ? 4 : 2, CH = PM ? 3 : 1;
  static constexpr int NT = (S * (S + 1) / 2 + 15) / 16, NTL = (S * (S - 1) / 2 + 15) / 16;
  static constexpr int NL = (SETS * NB + 3) / 4;
  static constexpr int NO = NL + 2 * NT, pairs = (NO + 1) / 2;
  static constexpr int ldx = 17;  // LDS row of one element: its 16 beads (stream b, step g at 4 b + g)
};

__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ d4 mfma16(double a, double b, const d4& c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// the wave's LDS traffic before this point is complete and visible to all its lanes after it
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x of the other 32-lane half (out1 beside out0), and of the neighbouring 16-lane row
typedef unsigned u2 __attribute__((ext_vector_type(2)));
struct Pair {
  double a, b;
};
__device__ __forceinline__ Pair swap_rows(double x, bool half) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
  const u2 l = half ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                    : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const u2 h = half ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                    : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return Pair{__builtin_bit_cast(double, ((unsigned long long)h[0] << 32) | l[0]),
              __builtin_bit_cast(double, ((unsigned long long)h[1] << 32) | l[1])};
}
// over the four 16-lane rows (the same bits on every row)
__device__ __forceinline__ double rows_sum(double x) {
  Pair p = swap_rows(x, false);
  x = p.a + p.b;
  p = swap_rows(x, true);
  return p.a + p.b;
}
__device__ __forceinline__ double rows_max(double x) {
  Pair p = swap_rows(x, false);
  x = fmax(p.a, p.b);
  p = swap_rows(x, true);
  return fmax(p.a, p.b);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  const int u = __builtin_bit_cast(int, x);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(u, u, CTRL, 0xF, 0xF, false));
}

// Z = X Y + Z for commuting symmetric X, Y and a symmetric Z given by its blocks I <= K
template <int NB>
__device__ __forceinline__ void sym_mul_upper(const double (&X)[NB][NB], const double (&Y)[NB][NB],
                                              double (&Z)[NB][NB]) {
#pragma unroll
  for (int J = 0; J < NB; ++J)
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = I; K < NB; ++K) Z[I][K] = mfma4(X[J][I], Y[J][K], Z[I][K]);
}
// the blocks I > K as the transposes of those above; ident holds the unit block
template <int NB>
__device__ __forceinline__ void mirror(double (&Z)[NB][NB], double ident) {
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = I + 1; K < NB; ++K) Z[K][I] = mfma4(Z[I][K], ident, 0.0);
}
template <int NB>
__device__ __forceinline__ void sym_mul(const double (&X)[NB][NB], const double (&Y)[NB][NB], double ident,
                                        double (&Z)[NB][NB]) {
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = I; K < NB; ++K) Z[I][K] = 0.0;
  sym_mul_upper<NB>(X, Y, Z);
  mirror<NB>(Z, ident);
}

// T = exp(X) of the wave's four symmetric matrices, zero outside the leading n x n block (X is
// scaled in place): Exp16's degree-16 polynomial in four products, scaled and squared. Each stream has
// its own scaling 2^-s and is squared s times (powers of two are exact), so that its bits are the same
// whichever samples share the wave: all are squared up to the wave's smallest count, then those that
// need more. One count for all four loses up to all digits of a sample beside one whose |tau V| is large.
// MI355X, us, one count / own: A = 8, N = 16, P = 64, 1e5 samples 1,327 / 1,340, with +-dbeta 1,797 / 1,800,
// 262,144 of a trained flow (two or three squarings) 3,930 / 4,062; A = 11, N = 17, P = 50, 3,001 samples
// with +-dbeta 128 / 130; A = 16, N = 10, P = 30, 20,000 with +-dbeta 1,091 / 1,110. (Products with a per-lane
// power of two instead of v_ldexp_f64: A = 8 1,373; one loop that selects after every squaring: trained
// flow 4,175.)
// alpha = |X^2|_F^(1/2) needs only its binary exponent: its sum is taken in FP32, of alpha^4 2^-100
// (alpha up to 2^57 without overflow; below 2^-6, where s is 0 anyway, it may vanish).
template <int NB>
__device__ __forceinline__ void expm_block(double (&X)[NB][NB], int n, int i, int j, double ident,
                                           double (&T)[NB][NB]) {
  using E = Exp16;
  double X2[NB][NB], G[NB][NB], F[NB][NB];
  sym_mul<NB>(X, X, ident, X2);
  double nd = 0.0, no = 0.0;
#pragma unroll
  for (int I = 0; I < NB; ++I) {
    nd = fma(X2[I][I], X2[I][I], nd);
#pragma unroll
    for (int K = I + 1; K < NB; ++K) no = fma(X2[I][K], X2[I][K], no);
  }
  float m = (float)fma(0x1p-99, no, 0x1p-100 * nd);
  m += dpp_f<0xB1>(m);  // over the four columns of the stream: quad_perm [1,0,3,2], [2,3,0,1]
  m += dpp_f<0x4E>(m);
  {  // over the four rows
    unsigned u = __builtin_bit_cast(unsigned, m);
    u2 r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    m = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
    u = __builtin_bit_cast(unsigned, m);
    r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    m = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
  }
  // smallest s >= 0 with alpha 2^-s <= theta; a zero matrix gives -inf, a NaN s = 0
  const float sd = fmaf(0.25f, __log2f(m), 25.0f - (float)E::log2_theta);
  int s = 0;
  if (sd > 0.0f) s = sd < 64.0f ? (int)ceilf(sd) : 64;
  // largest and smallest of the four streams' counts: s and 64 - s in one register, row_ror 4, 8
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  auto pmax = [](unsigned x, unsigned y) {
    const us2 p = __builtin_bit_cast(us2, x), q = __builtin_bit_cast(us2, y);
    return __builtin_bit_cast(unsigned, __builtin_elementwise_max(p, q));
  };
  unsigned pk = (unsigned)s | (unsigned)(64 - s) << 16;
  pk = pmax(pk, (unsigned)__builtin_amdgcn_update_dpp((int)pk, (int)pk, 0x124, 0xF, 0xF, false));
  pk = pmax(pk, (unsigned)__builtin_amdgcn_update_dpp((int)pk, (int)pk, 0x128, 0xF, 0xF, false));
  pk = (unsigned)__builtin_amdgcn_readfirstlane((int)pk);
  const int smax = (int)(pk & 0xffffu), smin = 64 - (int)(pk >> 16);
  if (smax) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = 0; K < NB; ++K) {
        X[I][K] = ldexp(X[I][K], -s);
        X2[I][K] = ldexp(X2[I][K], -2 * s);
      }
  }
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      F[I][K] = fma(E::c1, X2[I][K], E::c2 * X[I][K]);
      if (K >= I) G[I][K] = E::c5 * X2[I][K];
    }
  sym_mul_upper<NB>(X2, F, G);  // G = y02 + c5 X2
  mirror<NB>(G, ident);
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      F[I][K] = fma(E::c4, X[I][K], fma(E::d3, X2[I][K], G[I][K]));
      if (K >= I) T[I][K] = fma(E::c6, G[I][K], E::e7 * X2[I][K]);
    }
  sym_mul_upper<NB>(F, G, T);  // T = y12
  mirror<NB>(T, ident);
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      const double x = X[I][K], x2 = X2[I][K], gg = G[I][K], y = T[I][K];
      F[I][K] = fma(E::c8, x2, fma(E::c9, x, y));
      G[I][K] = fma(E::c10, gg, fma(E::c11, x, fma(E::f10, x2, y)));
      if (K >= I) {
        double r = fma(E::c12, y, fma(E::c13, gg, fma(E::g14, x2, x)));
        if (K == I) r += (i == j && 4 * I + i < n) ? 1.0 : 0.0;
        T[I][K] = r;
      }
    }
  sym_mul_upper<NB>(F, G, T);
  mirror<NB>(T, ident);
  for (int k = 0; k < smin; ++k) {
    sym_mul<NB>(T, T, ident, F);
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = 0; K < NB; ++K) T[I][K] = F[I][K];
  }
  for (int k = smin; k < smax; ++k) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = I; K < NB; ++K) F[I][K] = 0.0;
    sym_mul_upper<NB>(T, T, F);
    const bool mine = k < s;
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = I; K < NB; ++K) T[I][K] = mine ? F[I][K] : T[I][K];
    mirror<NB>(T, ident);
  }
}

// R <- the chain of the stream to the right (b + D) after this one, R^T = R'^T R^T, for the
// streams b that are multiples of 2 D
template <int NB, int D>
__device__ __forceinline__ void join(double (&R)[NB][NB], double ident) {
  double W[NB][NB], Z[NB][NB];
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      W[I][K] = mfma4(shfl_down_d(R[I][K], 4 * D), ident, 0.0);  // A operands: transposed blocks
      Z[I][K] = 0.0;
    }
#pragma unroll
  for (int J = 0; J < NB; ++J)
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = 0; K < NB; ++K) Z[I][K] = mfma4(W[I][J], R[J][K], Z[I][K]);
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = 0; K < NB; ++K) R[I][K] = Z[I][K];
}

// Registers: at S <= 8 four waves per SIMD (three with +-dbeta), above two; what they spill stands above.
template <int S, bool PM>
struct BlockOccupancy {
  static constexpr int waves = S <= 8 ? (PM ? 3 : 4) : 2;
};

template <int S, bool PM, bool QF>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(BlockOccupancy<S, PM>::waves)))
k_eval_block(const BlockArgs a) {
  using Z = Geo<S, PM>;
  constexpr int NB = Z::NB, NT = Z::NT, NTL = Z::NTL, NL = Z::NL, SETS = Z::SETS, CH = Z::CH, NQ = SETS * NB;
  __shared__ double ldsV[NT * 16 * Z::ldx];
  __shared__ double ldsO[CH * NB * 64];
  const int lane = threadIdx.x;
  const int row = lane >> 4, n = lane & 15, b = n >> 2, g = n & 3;
  const int C = a.C, N = a.N, P = a.P, K = a.K, NK = (N + 3) / 4;
  const int spw = 4 / C;
  const int64_t first = (int64_t)blockIdx.x * spw;
  const int64_t sample = first + b / C;
  const bool live = sample < a.B;
  const int64_t NP = (int64_t)N * P;
  // the stream's beads [pbeg, pbeg + len)
  const int pbeg = (b % C) * K;
  const int len = live ? max(0, min(K, P - pbeg)) : 0;
  typedef typename std::conditional<QF, CoordOffsetBuf, CoordBuf>::type Loader;
  Loader qb;
  if constexpr (QF)
    qb = CoordOffsetBuf::wave_samples(a.qf, a.qcentre, a.B, NP, first, spw, live ? sample : -1);
  else
    qb = CoordBuf::wave_samples(a.q, a.B, NP, first, spw, live ? sample : -1);
  typedef typename Loader::raw_t raw_t;
  const __amdgpu_buffer_rsrc_t ops =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.ops, (short)0, NK * a.op_pairs * 1024, 0x00020000);

  double Rg[NB][NB], Rp[NB][NB], Rm[NB][NB];
  const double ident = row == g ? 1.0 : 0.0;  // unit block: element (row, g) of stream b
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      Rg[I][J] = I == J ? ident : 0.0;
      if (PM) Rp[I][J] = Rm[I][J] = Rg[I][J];
    }
  double lr[NB], ls = 0.0;  // log-domain products of rho's factors and of the scales
#pragma unroll
  for (int I = 0; I < NB; ++I) lr[I] = 0.0;
  // where the back finds element (4 I + row, 4 J + g) of its stream's first step: padding reads
  // the element after the last, whose coefficients are zero
  int xoff[NB][NB];
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      const int r = max(4 * I + row, 4 * J + g), c = min(4 * I + row, 4 * J + g);
      const int e = r >= S ? S * (S + 1) / 2 : (r == c ? S * (S - 1) / 2 + r : r * (r - 1) / 2 + c);
      xoff[I][J] = e * Z::ldx + 4 * b;
    }

  // mode (clamped) of this lane at mode group kk, and its coordinates at the bead of (stream, step
  // st + g) and at the next bead of the ring
  auto mode_of = [&](int kk) { return min(4 * kk + row, N - 1); };
  auto load_x = [&](int st, int kk, raw_t& x0, raw_t& xn) {
    const int p = st + g < len ? pbeg + st + g : min(pbeg, P - 1);
    const int m = mode_of(kk);
    x0 = qb.load(m, P, p);
    xn = qb.load(m, P, p + 1 == P ? 0 : p + 1);
  };
  // operand k of mode group kk
  struct Ops {
    double o[2 * Z::pairs];
  };
  auto load_ops = [&](int kk, Ops& w) {
    const int base = kk * a.op_pairs * 1024;
#pragma unroll
    for (int i = 0; i < Z::pairs; ++i) {
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      typedef double dd __attribute__((ext_vector_type(2)));
      const dd v = __builtin_bit_cast(dd, (u4)__builtin_amdgcn_raw_buffer_load_b128(ops, lane * 16 + 1024 * i, base, 0));
      w.o[2 * i] = v[0];
      w.o[2 * i + 1] = v[1];
    }
  };
  raw_t x0, xn;
  load_x(0, 0, x0, xn);

  for (int st = 0; st < K; st += 4) {
    const bool valid = st + g < len;
    const bool full = __all(valid);
    // ---------------------------------------------------------------- front
    d4 v[NT], e[NL];
    double t[SETS];
#pragma unroll
    for (int q = 0; q < NT; ++q) v[q] = *(const d4*)(a.energy + 16 * q + 4 * row);
#pragma unroll
    for (int q = 0; q < NL; ++q) e[q] = *(const d4*)(a.k2 + 16 * q + 4 * row);
#pragma unroll
    for (int s = 0; s < SETS; ++s) t[s] = 0.0;
    for (int kk = 0; kk < NK; ++kk) {
      raw_t y0, yn;  // the next group's (or the next steps') coordinates, loaded ahead
      const bool more = kk + 1 < NK;
      load_x(more ? st : st + 4, more ? kk + 1 : 0, y0, yn);
      Ops w;
      load_ops(kk, w);
      const int m = mode_of(kk);
      double x, xb;
      if constexpr (QF) {
        const double c = a.qcentre[m];
        x = c + (double)x0;
        xb = c + (double)xn;
      } else {
        x = x0;
        xb = xn;
      }
      const double* __restrict__ tt = a.tcs + (kk * 4 + row) * 8;
      const double sx = x + xb, dx = x - xb, q2s = fma(x, x, xb * xb), d2 = dx * dx;
#pragma unroll
      for (int s = 0; s < SETS; ++s) t[s] = fma(tt[2 * s + 1], d2, fma(tt[2 * s], q2s, t[s]));
#pragma unroll
      for (int q = 0; q < NL; ++q) e[q] = mfma16(w.o[q], sx, e[q]);
#pragma unroll
      for (int q = 0; q < NTL; ++q) v[q] = mfma16(w.o[NL + q], x, v[q]);
      if (a.quad) {
        const double xx = x * x;
#pragma unroll
        for (int q = 0; q < NT; ++q) v[q] = mfma16(w.o[NL + NTL + q], xx, v[q]);
      }
      if (NT > NTL && a.ldiag) {
#pragma unroll
        for (int q = NTL; q < NT; ++q) v[q] = mfma16(w.o[NL + NT + q], x, v[q]);
      }
      x0 = y0;
      xn = yn;
    }
    if (a.npair) {  // off-diagonal quadratic mode pairs, four per step like the modes
      const int p = valid ? pbeg + st + g : min(pbeg, P - 1);
      for (int kk = 0; 4 * kk < a.npair; ++kk) {
        const int pr = min(4 * kk + row, a.npair - 1);
        const int j1 = a.pair[2 * pr], j2 = a.pair[2 * pr + 1];
        const double f = qb.value_at(j1, P, p) * qb.value_at(j2, P, p);
        const double* __restrict__ ct = a.cpair + kk * NT * 64 + lane;
#pragma unroll
        for (int q = 0; q < NT; ++q) v[q] = mfma16(ct[64 * q], f, v[q]);
      }
    }
    wave_sync();  // the previous steps' reads of X and O are done
#pragma unroll
    for (int q = 0; q < NT; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) ldsV[(16 * q + row + 4 * r) * Z::ldx + n] = a.ntau * v[q][r];
    // O-factors in the log domain (surface 4 I + row of bead n in register I of a set), S_p = max
    // over both models' (pimc.py:1076-1084)
    double lo[NQ], lS = -INFINITY;
#pragma unroll
    for (int s = 0; s < SETS; ++s) t[s] = rows_sum(t[s]);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      lo[q] = fma(-0.5, t[q / NB] + e[q / 4][q % 4], a.lpref[16 * (q / 4) + 4 * row + q % 4]);
      if (q < 2 * NB) lS = fmax(lS, lo[q]);
    }
    lS = a.noscale ? 0.0 : rows_max(lS);
    if (valid) {
#pragma unroll
      for (int I = 0; I < NB; ++I) lr[I] += lo[I] - lS;
      ls += lS;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        const double o = exp(lo[(c + 1) * NB + I] - lS);
        ldsO[(c * NB + I) * 64 + 16 * row + n] = valid ? o : 1.0;  // past the stream's end: a unit step
      }
    if (a.dbg && valid) {
      double* dr = a.dbg + (sample * P + pbeg + st + g) * eval_debug_record(a.A, a.AR);
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        if (4 * I + row < a.AR) dr[4 * I + row] = exp(lo[I]);
        if (4 * I + row < a.A) dr[a.AR + 4 * I + row] = exp(lo[NB + I]);
      }
      if (row == 0) dr[a.AR + a.A] = exp(lS);
    }
    wave_sync();
    // ---------------------------------------------------------------- back
#pragma clang loop unroll(disable)
    for (int step = 0; step < 4; ++step) {
      const bool mine = st + step < len;  // this lane's stream has this step
      if (!full && !__any(mine)) break;
      double M[NB][NB];
      {
        double X[NB][NB];
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J) X[I][J] = ldsV[xoff[I][J] + step];
        if (!full) {
#pragma unroll
          for (int I = 0; I < NB; ++I)
#pragma unroll
            for (int J = 0; J < NB; ++J) X[I][J] = mine ? X[I][J] : 0.0;
        }
        expm_block<NB>(X, a.A, row, g, ident, M);
      }
      if (a.dbg && mine) {
        double* dr = a.dbg + (sample * P + pbeg + st + step) * eval_debug_record(a.A, a.AR) + a.AR + a.A + 1;
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J)
            if (4 * I + row < a.A && 4 * J + g < a.A) dr[(4 * I + row) * a.A + 4 * J + g] = M[I][J];
      }
      // R^T <- diag(O / S) M R^T (pimc.py:1181-1206; M at the base tau for every chain, quirk Q1)
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        double (&R)[NB][NB] = c == 0 ? Rg : (c == 1 ? Rp : Rm);
        double W[NB][NB];
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int J = 0; J < NB; ++J) W[I][J] = 0.0;
#pragma unroll
        for (int L = 0; L < NB; ++L)
#pragma unroll
          for (int I = 0; I < NB; ++I)
#pragma unroll
            for (int J = 0; J < NB; ++J) W[I][J] = mfma4(M[L][I], R[L][J], W[I][J]);
#pragma unroll
        for (int I = 0; I < NB; ++I) {
          const double o = ldsO[(c * NB + I) * 64 + 16 * row + 4 * b + step];
#pragma unroll
          for (int J = 0; J < NB; ++J) R[I][J] = W[I][J] * o;
        }
      }
    }
  }

  // the chains of a sample's streams in order, then the traces; rho and log S over the steps
  // (lanes 1, 2 apart) and the sample's streams
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    double (&R)[NB][NB] = c == 0 ? Rg : (c == 1 ? Rp : Rm);
    if (C >= 2) join<NB, 1>(R, ident);
    if (C == 4) join<NB, 2>(R, ident);
  }
  double tr[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    double (&R)[NB][NB] = c == 0 ? Rg : (c == 1 ? Rp : Rm);
    double s = 0.0;
#pragma unroll
    for (int I = 0; I < NB; ++I) s += R[I][I];
    s = row == g ? s : 0.0;
    s += shfl_xor_d(s, 1);
    s += shfl_xor_d(s, 2);
    tr[c] = rows_sum(s);
  }
  for (int w = 1; w < 4 * C; w <<= 1) {
#pragma unroll
    for (int I = 0; I < NB; ++I) lr[I] += shfl_xor_d(lr[I], w);
    ls += shfl_xor_d(ls, w);
  }
  double rho = 0.0;
#pragma unroll
  for (int I = 0; I < NB; ++I) rho += exp(lr[I]);
  rho = rows_sum(rho);
  if (live && row == 0 && n % (4 * C) == 0) {
    const int64_t os = a.out_stride;
    a.out[OUT_RHO * os + sample] = rho;
    a.out[OUT_G * os + sample] = tr[0];
    if (PM) {
      a.out[OUT_GP * os + sample] = tr[CH > 1 ? 1 : 0];
      a.out[OUT_GM * os + sample] = tr[CH > 1 ? 2 : 0];
    }
    a.out[OUT_LOGS * os + sample] = ls;
  }
}

template <int S>
hipError_t launch_s(int pm, const BlockArgs& a, hipStream_t s) {
  const int spw = 4 / a.C;
  const dim3 grid((unsigned)((a.B + spw - 1) / spw));
  if (a.qf) {
    if constexpr (S == 7 || S == 8) {
      if (pm) return hipErrorInvalidValue;
      hipLaunchKernelGGL((k_eval_block<S, false, true>), grid, dim3(kWave), 0, s, a);
    } else {
      return hipErrorInvalidValue;
    }
  } else if (pm) {
    hipLaunchKernelGGL((k_eval_block<S, true, false>), grid, dim3(kWave), 0, s, a);
  } else if constexpr (S <= 8) {
    hipLaunchKernelGGL((k_eval_block<S, false, false>), grid, dim3(kWave), 0, s, a);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

static hipError_t launch_piece(int pm, const BlockArgs& a, hipStream_t s) {
  switch (a.S) {
#define PIB_CASE(s_) \
  case s_: return launch_s<s_>(pm, a, s);
    PIB_CASE(5) PIB_CASE(6) PIB_CASE(7) PIB_CASE(8) PIB_CASE(9) PIB_CASE(10) PIB_CASE(11) PIB_CASE(12)
    PIB_CASE(13) PIB_CASE(14) PIB_CASE(15) PIB_CASE(16)
#undef PIB_CASE
  }
  return hipErrorInvalidValue;
}

// A launch has fewer than 2^32 threads: 2^24 waves at a time (2^26 samples of one stream each).
hipError_t launch_eval_block(int pm, const BlockArgs& a, hipStream_t s) {
  const int64_t most = (int64_t)(4 / a.C) << 24, NP = (int64_t)a.N * a.P;
  for (int64_t b = 0; b < a.B; b += most) {
    BlockArgs p = a;
    p.B = a.B - b < most ? a.B - b : most;
    if (a.qf) p.qf += b * NP; else p.q += b * NP;
    p.out += b;
    if (a.dbg) p.dbg += b * a.P * eval_debug_record(a.A, a.AR);
    if (hipError_t e = launch_piece(pm, p, s)) return e;
  }
  return hipSuccess;
}

// The constants in the order the kernel's operands read them (BlockArgs), for the plain or the
// +-dbeta kernel.
BlockTables block_tables(const BlockModel& m, bool pm) {
  const int S = block_size(m.A, m.AR), NB = (S + 3) / 4, NK = (m.N + 3) / 4, sets = pm ? 4 : 2;
  const int NT = (S * (S + 1) / 2 + 15) / 16, NTL = (S * (S - 1) / 2 + 15) / 16, NL = (sets * NB + 3) / 4;
  const int npair = (int)m.pairs.size() / 2;
  BlockTables t;
  t.S = S;
  t.op_pairs = (NL + 2 * NT + 1) / 2;
  size_t at = 0;
  auto section = [&](size_t n) {
    const size_t o = at;
    at += (n + 15) & ~(size_t)15;  // 128-byte sections
    return o;
  };
  t.energy = section((size_t)NT * 16);
  t.k2 = section((size_t)NL * 16);
  t.lpref = section((size_t)NL * 16);
  t.tcs = section((size_t)NK * 32);
  t.ops = section((size_t)NK * t.op_pairs * 128);
  t.cpair = section((size_t)((npair + 3) / 4) * NT * 64);
  t.data.assign(at, 0.0);
  double* d = t.data.data();
  const size_t AA = (size_t)m.A * m.A;
  // where row e of operand k of the group of mode j sits
  auto op = [&](int j, int k, int e) -> double& {
    return d[t.ops + (((size_t)(j / 4) * t.op_pairs + k / 2) * 64 + 16 * (j % 4) + e) * 2 + k % 2];
  };
  t.ldiag = 0;
  // elements (r, c), r >= c, from the lower triangle, as eigh(UPLO='L') reads V
  for (int r = 0; r < m.A; ++r)
    for (int c = 0; c <= r; ++c) {
      const int id = r == c ? S * (S - 1) / 2 + r : r * (r - 1) / 2 + c, q = id / 16, e = id % 16;
      const size_t el = (size_t)r * m.A + c;
      d[t.energy + 16 * q + 4 * (e % 4) + e / 4] = m.energy[el];
      for (int j = 0; j < m.N; ++j) {
        const double L = m.linear[j * AA + el];
        op(j, q < NTL ? NL + q : NL + NT + q, e) = L;
        if (q >= NTL && L != 0.0) t.ldiag = 1;
        if (m.qdiag) op(j, NL + NTL + q, e) = m.qdiag[j * AA + el];
      }
      for (int k = 0; k < npair; ++k)
        d[t.cpair + ((size_t)(k / 4) * NT + q) * 64 + 16 * (k % 4) + e] = m.qpair[k * AA + el];
    }
  for (int s = 0; s < sets; ++s) {
    const BlockModel::Set& st = m.set[s];
    for (int I = 0; I < NB; ++I)
      for (int i = 0; i < 4; ++i) {
        const int reg = s * NB + I, surf = 4 * I + i;  // register of the set, its row
        const size_t o = (size_t)(reg / 4) * 16 + 4 * i + reg % 4;
        const bool in = surf < st.A;
        d[t.k2 + o] = in ? st.k2[surf] : 0.0;
        d[t.lpref + o] = in ? st.lpref[surf] : -INFINITY;
        for (int j = 0; in && j < m.N; ++j) op(j, reg / 4, 4 * (reg % 4) + i) = st.lin[(size_t)surf * m.N + j];
      }
    for (int j = 0; j < m.N; ++j) {
      d[t.tcs + (size_t)j * 8 + 2 * s] = st.th[j];
      d[t.tcs + (size_t)j * 8 + 2 * s + 1] = st.cs[j];
    }
  }
  return t;
}

}  // namespace pib
