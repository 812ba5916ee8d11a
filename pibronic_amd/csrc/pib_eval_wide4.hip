// FP64 evaluation for 9 to 12 surfaces without +-dbeta, four samples per wave on 4 x 4 matrix blocks.
//
// The arithmetic of the one-wave-per-sample kernel (pib_eval_wide.hip), operation for operation, so
// the results are the same bits; only where it happens differs:
//  * Matrices are 3 x 3 blocks of 4 x 4, one register pair holding one block of four samples
//    (lane 16 i + 4 b + j: element (i, j) of sample b, the layout of v_mfma_f64_4x4x4_4b_f64; a sum
//    over k is the same chain of fused multiply-adds there and in 16x16x4). A product of 12 x 12
//    matrices is 27 instructions of 19 cycles for four samples, against 3 of 70 cycles on 16 x 16
//    tiles for one. Products are formed whole: the blocks below the diagonal differ from the
//    transposes of those above in their last bits.
//  * Couplings: four steps of the four samples at a time, only the S (S + 1) / 2 elements of the
//    lower triangle (lane 16 b + e: element 16 k + e of sample b, its four steps), handed to the
//    block layout through LDS, whose reads mirror them. The wide kernel forms all 16 x 12. The
//    coefficients of all modes stay in LDS, shared by the work-group's four waves: read from L2 they
//    held the wave longer than the products (2,600 us in all at the size below, with the exponents
//    on the vector unit; 2,320 from LDS).
//  * O-exponents: sums over the modes in mode order, so 16x16x4 instructions with the 16 beads as
//    columns form them; lane 16 i + 4 b + g has surfaces 4 I + i of bead 4 c + g of sample b (a
//    fifth of the loads: 2,320 -> 1,725 us).
//  * Each sample keeps its own squaring count; the wave runs the largest and each sample stops at
//    its own.
//
// Measured (MI355X, A = 12, N = 24, P = 128, 16,384 samples, us): 3,600 in the wide kernel, 1,725 here.
// What bounds it: FP64 issue, as the block kernel (about three quarters of the cycles; two waves per SIMD, by
// registers and LDS, leave the rest exposed).
#include "pib_common.hpp"
#include "pib_expm.hpp"
#include "pib_kernels.hpp"

namespace pib {

namespace {

__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
typedef double d4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ d4 mfma16(double a, double b, const d4& c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
  const long long u = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double rows_sum(double x) {  // (r0 + r1) + (r2 + r3) over the 16-lane rows
  x += shfl_xor_d(x, 16);
  x += shfl_xor_d(x, 32);
  return x;
}

constexpr int NB = 3;
typedef double Mat[NB][NB];

// Z + X Y for a symmetric X
__device__ __forceinline__ void mul(const Mat& X, const Mat& Y, Mat& Z) {
#pragma unroll
  for (int J = 0; J < NB; ++J)
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int K = 0; K < NB; ++K) Z[I][K] = mfma4(X[J][I], Y[J][K], Z[I][K]);
}
__device__ __forceinline__ void mul0(const Mat& X, const Mat& Y, Mat& Z) {
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int K = 0; K < NB; ++K) Z[I][K] = 0.0;
  mul(X, Y, Z);
}

#define PIB_EACH                 \
  _Pragma("unroll") for (int I = 0; I < NB; ++I) \
  _Pragma("unroll") for (int K = 0; K < NB; ++K)

// expm_sym of the wide kernel on the wave's four matrices (x1 = X in, destroyed)
__device__ __forceinline__ void expm4(Mat& x1, int n, int i, int j, Mat& T) {
  using E = Taylor16;
  Mat x2, G, F;
  mul0(x1, x1, x2);
  double n2 = 0.0;
  PIB_EACH n2 = fma(x2[I][K], x2[I][K], n2);
  n2 += dpp_d<0xB1>(n2);  // the four columns, then the four rows of the sample's blocks
  n2 += dpp_d<0x4E>(n2);
  n2 = rows_sum(n2);
  const double sd = 0.25 * log2_coarse(n2) - E::log2_theta;
  int s = 0;
  if (sd > 0.0) s = sd < 64.0 ? (int)ceil(sd) : 64;
  int smax = max(s, __builtin_amdgcn_update_dpp(s, s, 0x124, 0xF, 0xF, false));  // row_ror 4, 8
  smax = max(smax, __builtin_amdgcn_update_dpp(smax, smax, 0x128, 0xF, 0xF, false));
  smax = __builtin_amdgcn_readfirstlane(smax);
  PIB_EACH {
    x1[I][K] = ldexp(x1[I][K], -s);
    x2[I][K] = ldexp(x2[I][K], -2 * s);
    F[I][K] = fma(E::c1, x2[I][K], E::c2 * x1[I][K]);
    G[I][K] = E::c5 * x2[I][K];
  }
  mul(x2, F, G);  // y02 + E::c5 X2
  PIB_EACH {
    F[I][K] = fma(E::c4, x1[I][K], fma(E::d3, x2[I][K], G[I][K]));
    T[I][K] = fma(E::c6, G[I][K], E::e7 * x2[I][K]);
  }
  mul(F, G, T);  // y12
  PIB_EACH {
    const double y = T[I][K], g = G[I][K], a = x1[I][K], b = x2[I][K];
    F[I][K] = fma(E::c8, b, fma(E::c9, a, y));
    G[I][K] = fma(E::c10, g, fma(E::c11, a, fma(E::f10, b, y)));
    T[I][K] = fma(E::c12, y, fma(E::c13, g, fma(E::g14, b, a)));
    if (I == K) T[I][K] += (i == j && 4 * I + i < n) ? 1.0 : 0.0;
  }
  mul(F, G, T);
  for (int k = 0; k < smax; ++k) {
    mul0(T, T, F);
    const bool mine = k < s;
    PIB_EACH T[I][K] = mine ? F[I][K] : T[I][K];
  }
}

// loads by buffer: a per-lane byte offset that stays, a uniform one that moves with the mode
__device__ __forceinline__ double load1(__amdgpu_buffer_rsrc_t r, int lane_off, int off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, off, 0));
}
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef double dd __attribute__((ext_vector_type(2)));
__device__ __forceinline__ dd load2(__amdgpu_buffer_rsrc_t r, int lane_off, int off) {
  return __builtin_bit_cast(dd, (u4)__builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0));
}

constexpr size_t kLds4 = 80 * 1024;  // two work-groups per CU
constexpr int kWaves4 = 4;  // waves per work-group, sharing the coupling table
template <int S>
struct Lds4 {
  static constexpr int tri = S * (S + 1) / 2, NT = (tri + 15) / 16, ldx = 17;
  double V[(NT * 16 + 1) * ldx];  // element e, bead column 4 b + step; the last row zero
  double O[NB * 64];
};
// with the coupling table {L, Qh}[mode][element] of N modes
template <int S>
constexpr size_t lds4_bytes(int N) {
  return kWaves4 * sizeof(Lds4<S>) + (size_t)N * Lds4<S>::tri * sizeof(dd);
}

template <int S>
__global__ void __launch_bounds__(kWave * kWaves4) __attribute__((amdgpu_waves_per_eu(2)))
k_eval_wide4(const EvalArgs a) {
  typedef Lds4<S> L4;
  constexpr int tri = L4::tri, NT = L4::NT, ldx = L4::ldx;
  extern __shared__ __align__(16) unsigned char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  double* ldsV = ((L4*)lds)[wave].V;
  double* ldsO = ((L4*)lds)[wave].O;
  dd* LQ = (dd*)((L4*)lds + kWaves4);
  for (int e = threadIdx.x; e < a.N * tri; e += kWave * kWaves4) {
    const int d = e / tri, k = e - d * tri;
    int r = 0;
    while ((r + 1) * (r + 2) / 2 <= k) ++r;
    const double2 c = a.wide_lq[d * 256 + r * 16 + k - r * (r + 1) / 2];
    LQ[e] = dd{c.x, c.y};
  }
  __syncthreads();
  const int lane = threadIdx.x % kWave;
  const int row = lane >> 4, n = lane & 15, b = n >> 2, g = n & 3;
  const int N = a.N, P = a.P, A = a.A, AR = a.AR;
  const int64_t first = ((int64_t)blockIdx.x * kWaves4 + wave) * 4;
  if (first >= a.B) return;  // whole wave; no work-group barrier follows
  const int64_t NP = (int64_t)N * P;
  const int64_t so = first + b, sv = first + row;  // this lane's sample in the O and V parts
  const CoordBuf qo = CoordBuf::wave_samples(a.q, a.B, NP, first, 4, so < a.B ? so : -1);
  const CoordBuf qv = CoordBuf::wave_samples(a.q, a.B, NP, first, 4, sv < a.B ? sv : -1);
  const ModeRec rec(A, AR);
  const int rl = rec.len();
  const auto tabb = __builtin_amdgcn_make_buffer_rsrc((void*)a.mode_tab, (short)0, N * rl * 8, 0x00020000);
  const OSet sr = a.set[SET_RHO], sw = a.set[SET_VIB];
  const double ntau = -a.tau;

  if (lane < ldx) ldsV[NT * 16 * ldx + lane] = 0.0;
  // element 16 k + n of the lower triangle, r (r + 1) / 2 + c: its number, its place in padded tables
  int le[NT], el[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    const int e = le[k] = min(16 * k + n, tri - 1);
    int r = 0;
    while ((r + 1) * (r + 2) / 2 <= e) ++r;
    el[k] = r * 16 + e - r * (r + 1) / 2;
  }
  int xoff[NB][NB];
  PIB_EACH {
    const int r = max(4 * I + row, 4 * K + g), c = min(4 * I + row, 4 * K + g);
    xoff[I][K] = (r < S ? r * (r + 1) / 2 + c : NT * 16) * ldx + 4 * b;
  }
  Mat R;
  PIB_EACH R[I][K] = (I == K && row == g) ? 1.0 : 0.0;
  int jr[NB], jv[NB];  // this lane's surfaces, clamped
  bool inr[NB], inv_[NB];
  // byte offsets in a mode's record of the exponent operands' coefficients, lane 16 k + i: row i
  const int lin0 = (n < 12 ? rec.lin_rho() + min(n, AR - 1) : rec.lin_vib() + min(n - 12, A - 1)) * 8;
  const int lin1 = (rec.lin_vib() + min(4 + n, A - 1)) * 8;
  const int cst = ((n < 4 ? 0 : 2) + (row & 1)) * 8;
  double rp[NB], smant = 1.0;
  int sexp = 0;
#pragma unroll
  for (int I = 0; I < NB; ++I) {
    const int j = 4 * I + row;
    inr[I] = j < AR;
    inv_[I] = j < A;
    jr[I] = min(j, AR - 1);
    jv[I] = min(j, A - 1);
    rp[I] = 1.0;
  }

  for (int st = 0; st < P; st += 4) {
    const int p = st + g, pc = p < P ? p : P - 1, pn = pc + 1 == P ? 0 : pc + 1;
    const int xo0 = (qo.base + pc) * 8, xon = (qo.base + pn) * 8;
    int xv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) xv[k] = (qv.base + min(st + k, P - 1)) * 8;
    // the couplings; each mode's inputs are loaded while the one before is summed
    struct X4 {
      double x[4];
    };
    auto load_x = [&](int d) {
      X4 m;
#pragma unroll
      for (int k = 0; k < 4; ++k) m.x[k] = load1(qv.rsrc, xv[k], d * P * 8);
      return m;
    };
    double v[NT][4];
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int s = 0; s < 4; ++s) v[k][s] = 0.0;
    {
      X4 cur = load_x(0);
      for (int d = 0; d < N; ++d) {
        const X4 nxt = load_x(min(d + 1, N - 1));
#pragma unroll
        for (int k = 0; k < NT; ++k) {
          const dd c = LQ[d * tri + le[k]];
#pragma unroll
          for (int s = 0; s < 4; ++s) v[k][s] = fma(cur.x[s], fma(c[1], cur.x[s], c[0]), v[k][s]);
        }
        cur = nxt;
      }
    }
    for (int t = 0; t < a.npair; ++t) {  // off-diagonal quadratic mode pairs
      const int j1 = a.pair[2 * t], j2 = a.pair[2 * t + 1];
      double xj[4], xk[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        xj[s] = load1(qv.rsrc, xv[s], j1 * P * 8);
        xk[s] = load1(qv.rsrc, xv[s], j2 * P * 8);
      }
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const double cq = a.wide_qpair[(size_t)t * 256 + el[k]];
#pragma unroll
        for (int s = 0; s < 4; ++s) v[k][s] = fma(xk[s] * cq, xj[s], v[k][s]);
      }
    }
    wave_sync();  // the previous steps' reads of X and O are done
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      const double e = a.wide_e[el[k]];
#pragma unroll
      for (int s = 0; s < 4; ++s) ldsV[(16 * k + n) * ldx + 4 * row + s] = ntau * (v[k][s] + e);
    }
    // The O-exponents (see OSet), then the O-factors and the scale (pimc.py:1076-1084). The sums over
    // the modes are chains of fused multiply-adds in mode order, so 16x16x4 matrix instructions form
    // them, with the 16 beads as columns: four modes of the surfaces' linear parts (rows 4 r + i:
    // register r of lane row i; rho's three, then vib's), two of the parts common to all surfaces
    // (th q2s, csch d2 in turn; rho in register 0 of every row, vib in register 1).
    struct ExpIn {
      double x0, xn, l0, l1, y0[2], yn[2], c[2];
    };
    auto load_exp = [&](int kk) {
      ExpIn m;
      const int d = min(4 * kk + row, N - 1);
      m.x0 = load1(qo.rsrc, xo0 + d * P * 8, 0);
      m.xn = load1(qo.rsrc, xon + d * P * 8, 0);
      m.l0 = load1(tabb, lin0 + d * rl * 8, 0);
      m.l1 = load1(tabb, lin1 + d * rl * 8, 0);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = min(4 * kk + 2 * h + (row >> 1), N - 1);
        m.y0[h] = load1(qo.rsrc, xo0 + e * P * 8, 0);
        m.yn[h] = load1(qo.rsrc, xon + e * P * 8, 0);
        m.c[h] = load1(tabb, cst + e * rl * 8, 0);
      }
      return m;
    };
    d4 e0 = {0.0, 0.0, 0.0, 0.0}, e1 = e0, tt = e0;
    {
      ExpIn cur = load_exp(0);
      for (int kk = 0; 4 * kk < N; ++kk) {
        const ExpIn nxt = load_exp(kk + 1);
        const bool in = 4 * kk + row < N;
        const double sx = in ? cur.x0 + cur.xn : 0.0;
        e0 = mfma16(in ? cur.l0 : 0.0, sx, e0);
        e1 = mfma16(in ? cur.l1 : 0.0, sx, e1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (4 * kk + 2 * h >= N) break;  // uniform
          const bool il = 4 * kk + 2 * h + (row >> 1) < N;
          const double y = cur.y0[h], yn = cur.yn[h], dx = y - yn;
          const double f = row & 1 ? dx * dx : fma(y, y, yn * yn);
          tt = mfma16(il && n < 8 ? cur.c[h] : 0.0, il ? f : 0.0, tt);
        }
        cur = nxt;
      }
    }
    const double tr = tt[0], tv = tt[1];
    const double er[NB] = {e0[0], e0[1], e0[2]}, ev[NB] = {e0[3], e1[0], e1[1]};
    double Or[NB], Ov[NB], mx = 0.0;  // a padded surface's O is 0
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      Or[I] = inr[I] ? exp(-0.5 * ((tr + er[I]) + sr.k2[jr[I]])) * sr.pref[jr[I]] : 0.0;
      Ov[I] = inv_[I] ? exp(-0.5 * ((tv + ev[I]) + sw.k2[jv[I]])) * sw.pref[jv[I]] : 0.0;
      mx = fmax(mx, fmax(Or[I], Ov[I]));
    }
    mx = fmax(mx, shfl_xor_d(mx, 16));
    mx = fmax(mx, shfl_xor_d(mx, 32));
    const double sc = a.noscale ? 1.0 : mx, inv = 1.0 / sc;
#pragma unroll
    for (int I = 0; I < NB; ++I) ldsO[I * 64 + 16 * row + n] = Ov[I] * inv;
    if (p < P) {
#pragma unroll
      for (int I = 0; I < NB; ++I) rp[I] *= Or[I] * inv;
      int e;
      smant = frexp(smant * sc, &e);
      sexp += e;
    }
    wave_sync();
    const int nb = min(4, P - st);
#pragma clang loop unroll(disable)
    for (int s = 0; s < nb; ++s) {
      Mat M, W;
      PIB_EACH W[I][K] = ldsV[xoff[I][K] + s];
      expm4(W, A, row, g, M);
      mul0(M, R, W);
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        const double o = ldsO[I * 64 + 16 * row + 4 * b + s];
#pragma unroll
        for (int K = 0; K < NB; ++K) R[I][K] = W[I][K] * o;
      }
    }
  }

  double tg = row == g ? (R[0][0] + R[1][1]) + R[2][2] : 0.0;
  tg += shfl_xor_d(tg, 1);
  tg += shfl_xor_d(tg, 2);
  tg = rows_sum(tg);
  double ls = log(smant) + (double)sexp * 0.69314718055994530942, rho = 0.0;
#pragma unroll
  for (int I = 0; I < NB; ++I) {
    rp[I] *= shfl_xor_d(rp[I], 1);
    rp[I] *= shfl_xor_d(rp[I], 2);
    const double q = rows_sum(inr[I] ? rp[I] : 0.0);
    rho = I ? rho + q : q;
  }
  ls += shfl_xor_d(ls, 1);
  ls += shfl_xor_d(ls, 2);
  if (so < a.B && row == 0 && g == 0) {
    const int64_t os = a.out_stride;
    a.out[OUT_RHO * os + so] = rho;
    a.out[OUT_G * os + so] = tg;
    a.out[OUT_LOGS * os + so] = ls;
  }
}

}  // namespace

template <int S>
static hipError_t launch_s4(const EvalArgs& a, hipStream_t s) {
  static unsigned long long lds_set = 0;
  if (hipError_t e = ensure_dynamic_lds((const void*)k_eval_wide4<S>, kLds4, lds_set)) return e;
  const int64_t groups = (a.B + 4 * kWaves4 - 1) / (4 * kWaves4);
  if (groups > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_eval_wide4<S>, dim3((unsigned)groups), dim3(kWave * kWaves4), lds4_bytes<S>(a.N), s, a);
  return hipGetLastError();
}

// Below 11 samples per CU the chip is not full of these longer waves, and the coupling table has to
// leave room for two work-groups per CU. MI355X, us, wide / this, A N P samples: 10 8 64 2,048
// 159 / 197, 3,000 218 / 199, 8,300 597 / 469, 12,000 806 / 479; 12 24 128 2,000 509 / 571,
// 3,000 680 / 573, 16,384 3,600 / 1,725; 9 3 12 2,816 45 / 41, 1e5 1,182 / 742; 11 24 60 50,000
// 5,211 / 2,937. With 13 surfaces and more a product is 64 instructions here and the 4 of the wide kernel
// are no more cycles. Rows of fewer than seven beads leave steps empty and need more waves: 12 3 3 2,816
// 14.9 / 16.5, 11 3 5 2,816 1.07 of the wide kernel's time, 5,000 1.01, 10,000 0.83.
bool wide4_supported(const EvalArgs& a, int num_cu) {
  if (a.P < 7 && a.B < (int64_t)num_cu * 20) return false;
  if (a.dbg || (int64_t)a.N * a.P >= (1 << 25) || a.B < (int64_t)num_cu * 11) return false;
  switch (a.A > a.AR ? a.A : a.AR) {
    case 9: return lds4_bytes<9>(a.N) <= kLds4;
    case 10: return lds4_bytes<10>(a.N) <= kLds4;
    case 11: return lds4_bytes<11>(a.N) <= kLds4;
    case 12: return lds4_bytes<12>(a.N) <= kLds4;
  }
  return false;
}

hipError_t launch_eval_wide4(const EvalArgs& a, hipStream_t s) {
  switch (a.A > a.AR ? a.A : a.AR) {
    case 9: return launch_s4<9>(a, s);
    case 10: return launch_s4<10>(a, s);
    case 11: return launch_s4<11>(a, s);
    case 12: return launch_s4<12>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pib
