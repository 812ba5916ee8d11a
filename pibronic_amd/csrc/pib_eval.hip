// FP64 per-sample evaluation of the PIMC estimator (one launch per block of samples).
//
// Replaces the body of block_compute / block_compute_pm after the coordinate transform
// (pibronic/pimc/pimc.py:1366-1381, 1421-1449): build_o_matrix (:1087-1129),
// build_scaling_factors + scale_o_matrices (:1062-1084), build_denominator (:1132-1136),
// diagonalize_coupling_matrix (:1139-1174) and build_numerator (:1177-1213), fused.
//
// Mapping (gfx950, wave64): G lanes cooperate on one sample, 64/G samples per wave. Lane g
// owns the contiguous bead chunk [g*K, min((g+1)*K, P)). Per bead it forms the diagonal
// O-factors of every temperature set, the residual coupling V in registers, M = exp(-tau V)
// directly (a scaled and squared polynomial, per lane, A x A in registers; the
// reference's eigendecomposition serves only to form M) and multiplies M * diag(O_vib / S_p)
// into its running ring product. The G partial products are
// then combined by a log2(G)-level ordered tree of A x A products over cross-lane moves
// (chunk 0 * chunk 1 * ... keeps the reference's left-to-right order).
//
// Numerics: the O-matrix exponent sum_j coth (x1^2 + x2^2) - 2 csch x1 x2 (x1, x2 the shifted
// coordinates of beads p, p+1) is evaluated as
//   sum_j th (x^2 + x'^2) + csch (x - x')^2 + lin_a (x + x') + k2_a,   th = coth - csch,
// which needs one FMA per surface and mode instead of nine operations. The reference's
// expression cancels when tau*omega is small (coth*x^2 ~ 1e3 against a result ~1e1); this
// form does not, so it sits about 100x closer to the exact value of the same rounded
// constants, and the O-factors differ from the reference's by the reference's own rounding
// (<= 1e-11 relative at A=12, N=24, P=128; ~1e-13 at the small workloads). V is built from
// the unshifted coordinates (the reference's shift/unshift leaves an ulp of drift in q,
// which moves V by ~1e-16). Linear algebra (V, M, ring) uses explicit fma().
#include <type_traits>

#include "pib_common.hpp"
#include "pib_expm.hpp"
#include "pib_kernels.hpp"

namespace pib {

// ---------------------------------------------------------------------------------------
// M = exp(X) for a symmetric A x A matrix held in one lane's registers, X = -tau V.
//
// The reference forms M = U diag(exp(-tau lambda)) U^T from eigh(V) (pimc.py:1167-1187); M is
// the only consumer of the decomposition, so it is computed directly: scaling and squaring of a
// polynomial (pib_expm.hpp), in one of two evaluation forms (expm_lane picks one per kernel).
// Every intermediate is a polynomial in X, hence symmetric, so products form the upper triangle
// only. s differs between lanes; the squaring loop runs the wave's largest count.
// Z = X Y + d I for commuting symmetric X, Y (Z symmetric; Z must not alias X or Y)
template <int A>
__device__ __forceinline__ void sym_prod_lane(const double (&X)[A][A], const double (&Y)[A][A], double d,
                                              double (&Z)[A][A]) {
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      double s = (i == k) ? fma(X[i][0], Y[0][k], d) : X[i][0] * Y[0][k];
#pragma unroll
      for (int c = 1; c < A; ++c) s = fma(X[i][c], Y[c][k], s);
      Z[i][k] = s;
      Z[k][i] = s;
    }
}

// T <- T^(2^s) for a symmetric T. Two squarings per iteration (T -> Z -> T), so that no
// register copy follows each one; an odd count ends with one squaring and a copy. s differs
// between lanes; the loop runs the wave's largest count.
template <int A>
__device__ __forceinline__ void square_times(double (&T)[A][A], int s) {
  double Z[A][A];
  for (int k = 0; k + 1 < s; k += 2) {
    sym_prod_lane<A>(T, T, 0.0, Z);
    sym_prod_lane<A>(Z, Z, 0.0, T);
  }
  if (s & 1) {
    sym_prod_lane<A>(T, T, 0.0, Z);
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int j = 0; j < A; ++j) T[i][j] = Z[i][j];
  }
}

// Exp8's degree-8 polynomial in three matrix products (Horner's rule takes seven). Y's product is
// taken as two dot products per entry (X2 X2 and X2 X) so that no fourth matrix is live beside X,
// X2 and Y; the three factors of the last product then replace X, X2 and Y entry by entry.
// alpha = |X^2|_F^(1/2), a tighter bound on the spectral radius of a symmetric X than |X|_F (the
// root of the largest of sum lambda^4), from X2, which the polynomial needs anyway. The terms
// beyond I + X + X^2/2 are small against the result, so the form rounds like Horner's rule.
template <int A>
__device__ __forceinline__ void expm_lane_s8(double (&X)[A][A], double (&T)[A][A]) {
  using E = Exp8;
  double X2[A][A];
  sym_prod_lane<A>(X, X, 0.0, X2);
  double n2 = 0.0;
#pragma unroll
  for (int i = 0; i < A; ++i) {
    n2 = fma(X2[i][i], X2[i][i], n2);
#pragma unroll
    for (int k = i + 1; k < A; ++k) n2 = fma(2.0 * X2[i][k], X2[i][k], n2);
  }
  // smallest s >= 0 with |X^2|_F^(1/2) 2^-s <= theta; a zero matrix gives -inf, NaN s = 0
  const double sd = 0.25 * log2_coarse(n2) - E::log2_theta;
  int s = 0;
  if (sd > 0.0) s = sd < 64.0 ? (int)ceil(sd) : 64;
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      X[i][k] = ldexp(X[i][k], -s);
      X[k][i] = X[i][k];
      X2[i][k] = ldexp(X2[i][k], -2 * s);
      X2[k][i] = X2[i][k];
    }
  // T <- Y = c1 X2 X2 + c2 X2 X (symmetric: polynomials in X commute)
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      double a = X2[i][0] * X2[0][k], b = X2[i][0] * X[0][k];
#pragma unroll
      for (int c = 1; c < A; ++c) {
        a = fma(X2[i][c], X2[c][k], a);
        b = fma(X2[i][c], X[c][k], b);
      }
      T[i][k] = fma(E::c1, a, E::c2 * b);
      T[k][i] = T[i][k];
    }
  // factors in place: X <- Y + c3 X2 + c4 X, X2 <- Y + c5 X2, T <- c6 Y + c7 X2 + X + I
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      const double x = X[i][k], x2 = X2[i][k], y = T[i][k];
      double w = fma(E::c6, y, fma(E::c7, x2, x));
      if (i == k) w += 1.0;
      X[i][k] = fma(E::c3, x2, fma(E::c4, x, y));
      X[k][i] = X[i][k];
      X2[i][k] = fma(E::c5, x2, y);
      X2[k][i] = X2[i][k];
      T[i][k] = w;
      T[k][i] = w;
    }
  // T <- X X2 + T: each output entry reads only its own entry of T
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      double acc = T[i][k];
#pragma unroll
      for (int c = 0; c < A; ++c) acc = fma(X[i][c], X2[c][k], acc);
      T[i][k] = acc;
      T[k][i] = acc;
    }
  square_times<A>(T, s);
}

// Exp16's degree-16 polynomial in four products. To keep four matrices live at most, y02 is held
// as G = y02 + c5 X2 (the second factor of y12's product; the later terms in y02 are rewritten in G
// and X2), and y12's first factor is formed one row at a time. alpha as in the degree-8 form; on
// the A = 4, 6 and 8 workload matrices a wave needs no squaring (Taylor coefficients: 0.5-1.0).
template <int A>
__device__ __forceinline__ void expm_lane_s16(double (&X)[A][A], double (&T)[A][A]) {
  using E = Exp16;
  double X2[A][A], Gm[A][A];
  sym_prod_lane<A>(X, X, 0.0, X2);
  double n2 = 0.0;
#pragma unroll
  for (int i = 0; i < A; ++i) {
    n2 = fma(X2[i][i], X2[i][i], n2);
#pragma unroll
    for (int k = i + 1; k < A; ++k) n2 = fma(2.0 * X2[i][k], X2[i][k], n2);
  }
  const double sd = 0.25 * log2_coarse(n2) - E::log2_theta;
  int s = 0;
  if (sd > 0.0) s = sd < 64.0 ? (int)ceil(sd) : 64;
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      X[i][k] = ldexp(X[i][k], -s);
      X[k][i] = X[i][k];
      X2[i][k] = ldexp(X2[i][k], -2 * s);
      X2[k][i] = X2[i][k];
    }
  // T <- c1 X2 + c2 X; G <- X2 T + c5 X2
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      T[i][k] = fma(E::c1, X2[i][k], E::c2 * X[i][k]);
      T[k][i] = T[i][k];
    }
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      double acc = E::c5 * X2[i][k];
#pragma unroll
      for (int c = 0; c < A; ++c) acc = fma(X2[i][c], T[c][k], acc);
      Gm[i][k] = acc;
      Gm[k][i] = acc;
    }
  // T <- y12 = F G + c6 G + e7 X2, F = G + d3 X2 + c4 X taken one row at a time
#pragma unroll
  for (int i = 0; i < A; ++i) {
    double f[A];
#pragma unroll
    for (int c = 0; c < A; ++c) f[c] = fma(E::c4, X[i][c], fma(E::d3, X2[i][c], Gm[i][c]));
#pragma unroll
    for (int k = i; k < A; ++k) {
      double acc = fma(E::c6, Gm[i][k], E::e7 * X2[i][k]);
#pragma unroll
      for (int c = 0; c < A; ++c) acc = fma(f[c], Gm[c][k], acc);
      T[i][k] = acc;
      T[k][i] = acc;
    }
  }
  // factors in place: X <- y12 + c8 X2 + c9 X, X2 <- y12 + c10 G + c11 X + f10 X2,
  // T <- c12 y12 + c13 G + g14 X2 + X + I
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      const double x = X[i][k], x2 = X2[i][k], g = Gm[i][k], y = T[i][k];
      double r = fma(E::c12, y, fma(E::c13, g, fma(E::g14, x2, x)));
      if (i == k) r += 1.0;
      X[i][k] = fma(E::c8, x2, fma(E::c9, x, y));
      X[k][i] = X[i][k];
      X2[i][k] = fma(E::c10, g, fma(E::c11, x, fma(E::f10, x2, y)));
      X2[k][i] = X2[i][k];
      T[i][k] = r;
      T[k][i] = r;
    }
  // T <- X X2 + T: each output entry reads only its own entry of T
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = i; k < A; ++k) {
      double acc = T[i][k];
#pragma unroll
      for (int c = 0; c < A; ++c) acc = fma(X[i][c], X2[c][k], acc);
      T[i][k] = acc;
      T[k][i] = acc;
    }
  square_times<A>(T, s);
}

// Which form each kernel uses: four products at degree 16, except at A = 6 without +-dbeta, whose
// kernel holds two waves per SIMD in 256 VGPRs and spills with four live matrices: degree 8 in
// three products there. Measured on MI355X (eval us, 1e5 samples, P = 64, N = 2 A; Taylor
// polynomials of the same forms / these): A = 4 282 / 271, A = 7 1214 / 1177; A = 6 at P = 128
// 1352 / 1294; with +-dbeta A = 4 437 (degree 12 in five products) / 408, A = 5 942 / 906 and A = 6
// 1454 / 1387 (degree 8).
template <int A, bool PM>
__device__ __forceinline__ void expm_lane(double (&X)[A][A], double (&T)[A][A]) {
  if constexpr (!PM && A == 6)
    expm_lane_s8<A>(X, T);
  else
    expm_lane_s16<A>(X, T);
}

// FOLD (EvalArgs.fold): rho's exponents equal vib's, and no linear coupling has a diagonal; both
// hold bit for bit for a coupled model folded by the host and its own surface diagonal as rho.
// Skipping those products leaves the results' bits alone; measured on MI355X (us, 1e5 samples, A = 4,
// N = 8, P = 64): sampler, evaluation and sums 382 -> 364, evaluation with +-dbeta 409 -> 395; FP32 at
// A = 6, N = 12, P = 128, 50,000 samples 414 -> 398.
template <int A, int AR, bool PM, bool QD, bool FOLD, class Q>
__device__ __forceinline__ void mode_terms(const_as<double>* tab, const Q& qs, int N,
                                           int P, int p, int pn, double& tr, double& tv, double& tp,
                                           double& tm, double (&er)[AR], double (&ev)[A], double (&ep)[A],
                                           double (&em)[A], double (&v)[A][A]) {
  constexpr ModeRec R(A, AR);
  // one mode's terms from its coordinates x0 (bead p) and xn (bead pn)
  auto mode = [&](int j, double x0, double xn) {
    const_as<double>* t = tab + j * R.len();
    const double sx = x0 + xn, dx = x0 - xn;
    const double q2s = fma(x0, x0, xn * xn), d2 = dx * dx;
    if (!FOLD) tr = fma(t[1], d2, fma(t[0], q2s, tr));
    tv = fma(t[3], d2, fma(t[2], q2s, tv));
    if (PM) {
      tp = fma(t[R.pm() + 1], d2, fma(t[R.pm() + 0], q2s, tp));
      tm = fma(t[R.pm() + 3], d2, fma(t[R.pm() + 2], q2s, tm));
    }
#pragma unroll
    for (int a = 0; a < AR; ++a)
      if (!FOLD) er[a] = fma(t[R.lin_rho() + a], sx, er[a]);
#pragma unroll
    for (int a = 0; a < A; ++a) {
      ev[a] = fma(t[R.lin_vib() + a], sx, ev[a]);
      if (PM) {
        ep[a] = fma(t[R.lin_plus() + a], sx, ep[a]);
        em[a] = fma(t[R.lin_minus() + a], sx, em[a]);
      }
    }
    // one scalar operand per FMA (a VALU op reads at most one SGPR pair)
    const double xx = x0 * x0;
#pragma unroll
    for (int b = 0, e = 0; b < A; ++b)
#pragma unroll
      for (int c = 0; c <= b; ++c, ++e) {
        if (!FOLD || c < b) v[b][c] = fma(t[R.lin_q() + e], x0, v[b][c]);
        if (QD) v[b][c] = fma(t[R.quad() + e], xx, v[b][c]);
      }
  };
  // Eight modes per iteration in two halves of four: the coordinates of one half are loaded
  // while the other half's arithmetic runs, four modes ahead of their use, into registers that
  // are free by then (a copy of a value still in flight would wait for its load). The modes are
  // taken in groups of four: modes past N read the zero records the table is padded with (and
  // the last mode's coordinates again). The loop body is straight-line code, which keeps the
  // compiler's wait counts exact (with a branch per mode it waited for every load in flight at
  // the top of each iteration).
  // (the loader's raw values are carried between iterations; the coordinate is formed at use)
  typedef typename Q::raw_t raw_t;
  auto ld4 = [&](int j, raw_t (&x)[4][2]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int jj = j + k < N ? j + k : N - 1;
      x[k][0] = qs.load(jj, P, p);
      x[k][1] = qs.load(jj, P, pn);
    }
  };
  // modes past N read the centre of mode N - 1 (offset loader) with a zero record: nothing added
  auto use = [&](int j, const raw_t (&x)[2]) {
    const int jj = j < N ? j : N - 1;
    mode(j, qs.value(jj, x[0]), qs.value(jj, x[1]));
  };
  const int N4 = (N + 3) & ~3;
  raw_t xa[4][2], xb[4][2];
  ld4(0, xa);
  int j = 0;
  for (; j + 8 <= N4; j += 8) {
    ld4(j + 4, xb);
#pragma unroll
    for (int k = 0; k < 4; ++k) use(j + k, xa[k]);
    ld4(j + 8, xa);
#pragma unroll
    for (int k = 0; k < 4; ++k) use(j + 4 + k, xb[k]);
  }
  if (j < N4) {
#pragma unroll
    for (int k = 0; k < 4; ++k) use(j + k, xa[k]);
  }
}

// Occupancy: for A <= 4 the VGPR budget is capped at 256 (two waves per SIMD): the plain
// kernel needs 128 (four waves), the +-dbeta kernel's three ring states need ~200, and a cap
// of 168 made it spill (0.78 against 0.59 ms at A = 4, N = 8, P = 64, 1e5 samples, measured on
// MI355X). A = 5, 6 without +-dbeta are held to 256 as well (the persistent batched kernel
// otherwise takes 268 at A = 6 and drops to one wave per SIMD). Larger A, and the +-dbeta
// kernels of A > 4, keep the default budget (512 with the accumulation registers).
template <int A, bool PM>
struct EvalOccupancy {
  static constexpr int waves = (A <= 4 || (A <= 6 && !PM)) ? 2 : 1;
};

// The samples of one wave: wave w evaluates samples [w * 64/G, (w + 1) * 64/G) of `args`.
// QF: coordinates as float offsets from a per-mode centre (args.qf, args.qcentre).
template <int A, int AR, bool PM, bool DBG, bool FOLD, bool QF = false>
__device__ __forceinline__ void eval_wave(const EvalArgs& args, int64_t wave) {
  static_assert(!FOLD || A == AR, "FOLD: rho has the coupled model's surfaces");
  const int lane = threadIdx.x & (kWave - 1);
  const int G = args.G, K = args.K, N = args.N, P = args.P;
  const int gl = lane & (G - 1);
  const int spw = kWave / G;
  const int64_t sample = wave * spw + lane / G;
  const bool live = sample < args.B;
  const int64_t NP = (int64_t)N * P;
  typedef typename std::conditional<QF, CoordOffsetBuf, CoordBuf>::type Loader;
  Loader qb;
  if constexpr (QF)
    qb = CoordOffsetBuf::wave_samples(args.qf, args.qcentre, args.B, NP, wave * spw, spw, live ? sample : -1);
  else
    qb = CoordBuf::wave_samples(args.q, args.B, NP, wave * spw, spw, live ? sample : -1);

  // read-only constants through the constant address space: scalar loads
  struct RO {
    const_as<double>* k2;
    const_as<double>* lpref;
  };
  const RO sr{as_const(args.set[SET_RHO].k2), as_const(args.set[SET_RHO].lpref)};
  const RO sv{as_const(args.set[SET_VIB].k2), as_const(args.set[SET_VIB].lpref)};
  const RO sp{as_const(args.set[SET_VIB_PLUS].k2), as_const(args.set[SET_VIB_PLUS].lpref)};
  const RO sm{as_const(args.set[SET_VIB_MINUS].k2), as_const(args.set[SET_VIB_MINUS].lpref)};
  const_as<double>* Ev = as_const(args.energy);
  const double* __restrict__ Qd = args.qdiag;
  const_as<int>* pairs = as_const(args.pair);
  const_as<double>* qpair = as_const(args.qpair);

  double Ng[A][A], Np[A][A], Nm[A][A];
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int k = 0; k < A; ++k) {
      Ng[i][k] = (i == k) ? 1.0 : 0.0;
      if (PM) { Np[i][k] = Ng[i][k]; Nm[i][k] = Ng[i][k]; }
    }
  // log-domain products: lr[a] = sum_p log(O_rho,a(p) / S_p), ls = sum_p log S_p
  double lr[AR];
#pragma unroll
  for (int a = 0; a < AR; ++a) lr[a] = 0.0;
  double ls = 0.0;

  const int pbeg = gl * K;
  const int pend = live ? min(pbeg + K, P) : pbeg;
  for (int p = pbeg; p < pend; ++p) {
    const int pn = (p + 1 == P) ? 0 : p + 1;
    // O-matrix exponents (pimc.py:1087-1129) in the expanded cancellation-free form of OSet:
    // the surface-independent parts t* once per mode, one FMA per surface and mode
    double er[AR], ev[A], ep[A], em[A], v[A][A];
    double tr = 0.0, tv = 0.0, tp = 0.0, tm = 0.0;
#pragma unroll
    for (int a = 0; a < AR; ++a) er[a] = 0.0;
#pragma unroll
    for (int a = 0; a < A; ++a) {
      ev[a] = 0.0;
      ep[a] = 0.0;
      em[a] = 0.0;
#pragma unroll
      for (int c = 0; c <= a; ++c) v[a][c] = 0.0;
    }
    if (Qd)
      mode_terms<A, AR, PM, true, FOLD>(as_const(args.mode_tab), qb, N, P, p, pn, tr, tv, tp, tm, er, ev, ep, em, v);
    else
      mode_terms<A, AR, PM, false, FOLD>(as_const(args.mode_tab), qb, N, P, p, pn, tr, tv, tp, tm, er, ev, ep, em, v);
    // off-diagonal quadratic mode pairs (j != k)
    for (int t = 0; t < args.npair; ++t) {
      const int jj = pairs[2 * t], kk = pairs[2 * t + 1];
      const double xj = qb.value(jj, qb.load(jj, P, p)), xk = qb.value(kk, qb.load(kk, P, p));
      const_as<double>* Qh = qpair + (int64_t)t * A * A;
#pragma unroll
      for (int b = 0; b < A; ++b)
#pragma unroll
        for (int c = 0; c <= b; ++c) v[b][c] = fma(xk * Qh[b * A + c], xj, v[b][c]);
    }

    // O-factors and the per-bead scaling S_p = max over both O's (pimc.py:1076-1084), in the
    // log domain: log O_a = log F_a - e_a / 2, log S_p = max; rho's factors never leave it,
    // so per bead only the vib O-factors (and M's eigenvalues) need an exponential
    double lOr[AR], lOv[A], lOp[A], lOm[A];
    double lS = -INFINITY;
#pragma unroll
    for (int a = 0; a < AR; ++a) {
      if constexpr (FOLD)
        lOr[a] = fma(-0.5, (tv + ev[a]) + sv.k2[a], sr.lpref[a]);
      else
        lOr[a] = fma(-0.5, (tr + er[a]) + sr.k2[a], sr.lpref[a]);
      lS = fmax(lS, lOr[a]);
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
      lOv[a] = fma(-0.5, (tv + ev[a]) + sv.k2[a], sv.lpref[a]);
      lS = fmax(lS, lOv[a]);
      if (PM) lOp[a] = fma(-0.5, (tp + ep[a]) + sp.k2[a], sp.lpref[a]);
      if (PM) lOm[a] = fma(-0.5, (tm + em[a]) + sm.k2[a], sm.lpref[a]);
    }
    if (args.noscale) lS = 0.0;

    // coupling matrix -> M = exp(-tau V) (pimc.py:1167-1187)
    double M[A][A];
    {
      double X[A][A];
#pragma unroll
      for (int b = 0; b < A; ++b)
#pragma unroll
        for (int c = 0; c <= b; ++c) {
          X[b][c] = -args.tau * (v[b][c] + Ev[b * A + c]);
          X[c][b] = X[b][c];
        }
      expm_lane<A, PM>(X, M);
    }

    if (DBG) {
      const int rec = eval_debug_record(A, AR);
      double* dr = args.dbg + ((int64_t)sample * P + p) * rec;
#pragma unroll
      for (int a = 0; a < AR; ++a) dr[a] = exp(lOr[a]);
#pragma unroll
      for (int a = 0; a < A; ++a) dr[AR + a] = exp(lOv[a]);
      dr[AR + A] = exp(lS);
#pragma unroll
      for (int c = 0; c < A; ++c)
#pragma unroll
        for (int e = 0; e < A; ++e) dr[AR + A + 1 + c * A + e] = M[c][e];
    }

    // scale (pimc.py:1062-1066, 1445, 1448), then accumulate rho and the ring products
    double Ov[A], Op[A], Om[A];
#pragma unroll
    for (int a = 0; a < AR; ++a) lr[a] += lOr[a] - lS;
#pragma unroll
    for (int a = 0; a < A; ++a) {
      Ov[a] = exp(lOv[a] - lS);
      if (PM) {
        Op[a] = exp(lOp[a] - lS);
        Om[a] = exp(lOm[a] - lS);
      }
    }
    ls += lS;
#pragma unroll
    for (int i = 0; i < A; ++i) {
      double rg[A], rpl[A], rmi[A];
#pragma unroll
      for (int c = 0; c < A; ++c) {
        rg[c] = Ng[i][c];
        if (PM) { rpl[c] = Np[i][c]; rmi[c] = Nm[i][c]; }
      }
#pragma unroll
      for (int k = 0; k < A; ++k) {
        double s = rg[0] * M[0][k];
#pragma unroll
        for (int c = 1; c < A; ++c) s = fma(rg[c], M[c][k], s);
        Ng[i][k] = s * Ov[k];
        if (PM) {
          double sp_ = rpl[0] * M[0][k], sm_ = rmi[0] * M[0][k];
#pragma unroll
          for (int c = 1; c < A; ++c) {
            sp_ = fma(rpl[c], M[c][k], sp_);
            sm_ = fma(rmi[c], M[c][k], sm_);
          }
          Np[i][k] = sp_ * Op[k];
          Nm[i][k] = sm_ * Om[k];
        }
      }
    }
  }

  // ordered tree over the G lanes of a sample: lane g (g % 2s == 0) absorbs lane g + s
  for (int s = 1; s < G; s <<= 1) {
    const bool leader = (gl & (2 * s - 1)) == 0;
    double o[A][A];
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
      for (int k = 0; k < A; ++k) o[i][k] = shfl_down_d(Ng[i][k], s);
    if (leader) {
#pragma unroll
      for (int i = 0; i < A; ++i) {
        double r[A];
#pragma unroll
        for (int c = 0; c < A; ++c) r[c] = Ng[i][c];
#pragma unroll
        for (int k = 0; k < A; ++k) {
          double acc = r[0] * o[0][k];
#pragma unroll
          for (int c = 1; c < A; ++c) acc = fma(r[c], o[c][k], acc);
          Ng[i][k] = acc;
        }
      }
    }
    if (PM) {
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        double (&X)[A][A] = (w == 0) ? Np : Nm;
#pragma unroll
        for (int i = 0; i < A; ++i)
#pragma unroll
          for (int k = 0; k < A; ++k) o[i][k] = shfl_down_d(X[i][k], s);
        if (leader) {
#pragma unroll
          for (int i = 0; i < A; ++i) {
            double r[A];
#pragma unroll
            for (int c = 0; c < A; ++c) r[c] = X[i][c];
#pragma unroll
            for (int k = 0; k < A; ++k) {
              double acc = r[0] * o[0][k];
#pragma unroll
              for (int c = 1; c < A; ++c) acc = fma(r[c], o[c][k], acc);
              X[i][k] = acc;
            }
          }
        }
      }
    }
#pragma unroll
    for (int a = 0; a < AR; ++a) {
      const double t = shfl_down_d(lr[a], s);
      if (leader) lr[a] += t;
    }
    const double tl = shfl_down_d(ls, s);
    if (leader) ls += tl;
  }

  if (live && gl == 0) {
    const int64_t st = args.out_stride;
    double rho = exp(lr[0]);
#pragma unroll
    for (int a = 1; a < AR; ++a) rho += exp(lr[a]);
    double g = Ng[0][0];
#pragma unroll
    for (int i = 1; i < A; ++i) g += Ng[i][i];
    args.out[OUT_RHO * st + sample] = rho;
    args.out[OUT_G * st + sample] = g;
    if (PM) {
      double gp = Np[0][0], gm = Nm[0][0];
#pragma unroll
      for (int i = 1; i < A; ++i) { gp += Np[i][i]; gm += Nm[i][i]; }
      args.out[OUT_GP * st + sample] = gp;
      args.out[OUT_GM * st + sample] = gm;
    }
    args.out[OUT_LOGS * st + sample] = ls;
  }
}

template <int A, int AR, bool PM, bool DBG, bool FOLD = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EvalOccupancy<A, PM>::waves)))
k_eval_fp64(const EvalArgs args) {
  eval_wave<A, AR, PM, DBG, FOLD>(args, ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave);
}

// the same on float offsets from a per-mode centre (pib_eval_block_flow_offsets)
template <int A, bool FOLD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EvalOccupancy<A, false>::waves)))
k_eval_fp64_offsets(const EvalArgs args) {
  eval_wave<A, A, false, false, FOLD, true>(args, ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave);
}

LaneProb lane_prob(const EvalArgs& a) {
  LaneProb p{};
  p.q = a.q;
  p.out = a.out;
  p.out_stride = a.out_stride;
  p.B = a.B;
  p.N = a.N;
  p.P = a.P;
  p.G = a.G;
  p.K = a.K;
  p.npair = a.npair;
  p.noscale = a.noscale;
  p.tau = a.tau;
  p.mode_tab = a.mode_tab;
  p.energy = a.energy;
  p.qdiag = a.qdiag;
  p.pair = a.pair;
  p.qpair = a.qpair;
  for (int k = 0; k < NUM_SETS; ++k) {
    p.k2[k] = a.set[k].k2;
    p.lpref[k] = a.set[k].lpref;
  }
  return p;
}

// Persistent batched launch: many blocks of samples (temperatures with different P, models
// with the same surface counts) in one grid. Each wave repeatedly takes the next tile
// (problem, first wave, wave count) from a device counter until the tile list is exhausted;
// the host orders tiles by decreasing cost, so the long ones start first. Every wave reaches
// the exit once the counter passes the tile count. The problems' arguments come by value in
// the kernel arguments (scalar registers), as in the stand-alone launch.
template <int A, int AR, bool PM, bool FOLD = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EvalOccupancy<A, PM>::waves)))
k_eval_batched(const LaneProbs probs, const BatchTile* __restrict__ tiles, int ntiles, int* counter) {
  const int lane = threadIdx.x & (kWave - 1);
  for (;;) {
    int t = 0;
    if (lane == 0) t = atomicAdd(counter, 1);
    t = __builtin_amdgcn_readfirstlane(__shfl(t, 0, kWave));
    if (t >= ntiles) break;
    const int pi = __builtin_amdgcn_readfirstlane(tiles[t].prob);
    const int64_t w0 = __builtin_amdgcn_readfirstlane(tiles[t].wave0);
    const int nw = __builtin_amdgcn_readfirstlane(tiles[t].nwaves);
    const LaneProb& d = probs.p[pi];
    EvalArgs a{};
    a.q = d.q;
    a.out = d.out;
    a.out_stride = d.out_stride;
    a.B = d.B;
    a.N = d.N;
    a.P = d.P;
    a.G = d.G;
    a.K = d.K;
    a.npair = d.npair;
    a.noscale = d.noscale;
    a.tau = d.tau;
    a.mode_tab = d.mode_tab;
    a.energy = d.energy;
    a.qdiag = d.qdiag;
    a.pair = d.pair;
    a.qpair = d.qpair;
    a.dbg = nullptr;
#pragma unroll
    for (int k = 0; k < NUM_SETS; ++k) {
      a.set[k].k2 = d.k2[k];
      a.set[k].lpref = d.lpref[k];
    }
    for (int64_t w = w0; w < w0 + nw; ++w) eval_wave<A, AR, PM, false, FOLD>(a, w);
  }
}

// ---------------------------------------------------------------------------------------
// Sizes with folded instances: up to four surfaces. MI355X, us, general / folded, A N P samples: 2 10 40 1e5
// 116.5 / 109.5, 3 10 40 1e5 149 / 143 and with +-dbeta 239 / 201, 4 8 64 1e5 267 / 258 and 402 / 391; the
// wider ones lose by their schedule what the exponents save: 5 17 56 4,000 39 / 46, 5 10 64 1e5
// 433 / 426 and 902 / 929, 6 12 64 3,000 39.2 / 40.5 and 1e5 1,383 / 1,410 with +-dbeta, 7 14 64 1e5
// 1,176 / 1,211.
template <int A, int AR>
constexpr bool folds = A == AR && A <= 4;

template <int A, int AR>
static hipError_t launch_a(int pm, const EvalArgs& a, hipStream_t s) {
  const int spw = kWave / a.G;
  const int64_t waves = (a.B + spw - 1) / spw;
  const int threads = 256;
  const dim3 grid((unsigned)((waves * kWave + threads - 1) / threads));
  const bool dbg = a.dbg != nullptr;
  // q is read straight from global memory. Staging each wave's samples through LDS (one
  // coalesced copy) removes the ~2.5x re-fetch of q seen in FETCH_SIZE, but measured 3-13%
  // slower on MI355X: the copy prologue adds latency and the LDS it needs costs occupancy,
  // while this kernel is bound by dependent FP64 arithmetic, not by memory.
  const EvalArgs& b = a;
  const size_t lds = 0;
  if (pm) {
    // from A = 7 on +-dbeta runs in the block kernel (three ring chains beside the exponential do
    // not fit in one lane's registers)
    if constexpr (A < 7) {
      if (dbg)
        hipLaunchKernelGGL((k_eval_fp64<A, AR, true, true>), grid, dim3(threads), lds, s, b);
      else if (folds<A, AR> && a.fold)
        hipLaunchKernelGGL((k_eval_fp64<A, AR, true, false, folds<A, AR>>), grid, dim3(threads), lds, s, b);
      else
        hipLaunchKernelGGL((k_eval_fp64<A, AR, true, false>), grid, dim3(threads), lds, s, b);
    } else {
      return hipErrorInvalidValue;
    }
  } else if (dbg)
    hipLaunchKernelGGL((k_eval_fp64<A, AR, false, true>), grid, dim3(threads), lds, s, b);
  else if (folds<A, AR> && a.fold)
    hipLaunchKernelGGL((k_eval_fp64<A, AR, false, false, folds<A, AR>>), grid, dim3(threads), lds, s, b);
  else
    hipLaunchKernelGGL((k_eval_fp64<A, AR, false, false>), grid, dim3(threads), lds, s, b);
  return hipGetLastError();
}

template <int A, int AR>
static hipError_t launch_batched_a(int pm, const LaneProbs& probs, const BatchTile* tiles, int ntiles,
                                   int* counter, int waves, hipStream_t s) {
  const dim3 grid((unsigned)((waves + 3) / 4));
  // the persistent kernel gains by folding at every size (sixteen temperatures of A = 6, us: 3,943 / 3,855)
  const bool fold = A == AR && probs.fold;
  if (pm && fold)
    hipLaunchKernelGGL((k_eval_batched<A, AR, true, A == AR>), grid, dim3(256), 0, s, probs, tiles, ntiles, counter);
  else if (pm)
    hipLaunchKernelGGL((k_eval_batched<A, AR, true>), grid, dim3(256), 0, s, probs, tiles, ntiles, counter);
  else if (fold)
    hipLaunchKernelGGL((k_eval_batched<A, AR, false, A == AR>), grid, dim3(256), 0, s, probs, tiles, ntiles, counter);
  else
    hipLaunchKernelGGL((k_eval_batched<A, AR, false>), grid, dim3(256), 0, s, probs, tiles, ntiles, counter);
  return hipGetLastError();
}

#define PIB_EVAL_CASES(X) \
  X(1, 1) X(2, 2) X(3, 3) X(4, 4) X(5, 5) X(6, 6) X(7, 7) X(8, 8) \
  X(2, 1) X(2, 4) X(2, 8) X(4, 2) X(4, 8)

bool eval_supported(int A, int AR) {
#define PIB_CASE(a_, ar_) if (A == a_ && AR == ar_) return true;
  PIB_EVAL_CASES(PIB_CASE)
#undef PIB_CASE
  return false;
}

hipError_t launch_eval_fp64(int A, int AR, int pm, const EvalArgs& a, hipStream_t s) {
  // A = 8 runs in the block kernel; here only its persistent batched form is compiled
#define PIB_CASE(a_, ar_) \
  if constexpr (a_ < 8)   \
    if (A == a_ && AR == ar_) return launch_a<a_, ar_>(pm, a, s);
  PIB_EVAL_CASES(PIB_CASE)
#undef PIB_CASE
  return hipErrorInvalidValue;
}

template <int A>
static hipError_t launch_offsets_a(const EvalArgs& a, hipStream_t s) {
  const int spw = kWave / a.G;
  const int64_t waves = (a.B + spw - 1) / spw;
  const int threads = 256;
  const dim3 grid((unsigned)((waves * kWave + threads - 1) / threads));
  if (folds<A, A> && a.fold)
    hipLaunchKernelGGL((k_eval_fp64_offsets<A, folds<A, A>>), grid, dim3(threads), 0, s, a);
  else
    hipLaunchKernelGGL((k_eval_fp64_offsets<A, false>), grid, dim3(threads), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_eval_fp64_offsets(int A, const EvalArgs& a, hipStream_t s) {
  switch (A) {
    case 1: return launch_offsets_a<1>(a, s);
    case 2: return launch_offsets_a<2>(a, s);
    case 3: return launch_offsets_a<3>(a, s);
    case 4: return launch_offsets_a<4>(a, s);
    case 5: return launch_offsets_a<5>(a, s);
    case 6: return launch_offsets_a<6>(a, s);
    case 7: return launch_offsets_a<7>(a, s);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_eval_batched(int A, int AR, int pm, const LaneProbs& probs, const BatchTile* tiles,
                               int ntiles, int* counter, int waves, hipStream_t s) {
#define PIB_CASE(a_, ar_) \
  if (A == a_ && AR == ar_) return launch_batched_a<a_, ar_>(pm, probs, tiles, ntiles, counter, waves, s);
  PIB_EVAL_CASES(PIB_CASE)
#undef PIB_CASE
  return hipErrorInvalidValue;
}

}  // namespace pib
