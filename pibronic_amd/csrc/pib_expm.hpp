// Polynomials of the evaluation kernels' M = exp(X), X = -tau V (symmetric): X is scaled by 2^-s
// so that a bound on its spectral radius is at most theta, the polynomial is evaluated in few
// matrix products and squared s times. For a symmetric X the 2-norm error of a polynomial in X is
// its largest scalar error over the eigenvalues, so the polynomials are fitted to the interval
// [-theta, theta] instead of being expanded at 0: each is the minimax approximation (Remez
// exchange at 60 digits) of e^x in relative error among the polynomials of its evaluation form
// with p(0) = p'(0) = 1 (X = 0 gives exactly I), and theta is the largest interval on which that
// error stays below the unit roundoff. Against the Taylor polynomials of the same forms theta
// doubles, one squaring less per exponential: 0.676 -> 1.35 at degree 16, 0.049 -> 0.122 at degree
// 8. (The FP32 kernel keeps its Taylor polynomial.)
#pragma once

namespace pib {

// Degree 16 in four products, after the "15+" evaluation form of Sastre (J. Sastre, "Efficient
// evaluation of matrix polynomials", Linear Algebra Appl. 539 (2018) 229-250), written in
// G = y02 + c5 X2 (so that four matrices are live at most):
//   G = X2 (c1 X2 + c2 X) + c5 X2,
//   Y = (G + d3 X2 + c4 X) G + c6 G + e7 X2,
//   T = (Y + c8 X2 + c9 X)(Y + c10 G + c11 X + f10 X2) + c12 Y + c13 G + g14 X2 + X + I.
// The coefficients give the x^2..x^15 terms of the minimax polynomial whose x^16 term is the
// form's own (c1^4). Rounded one by one to FP64 they would err by 9 u on the interval (terms of ten
// times the sum cancel); these are neighbouring doubles chosen together, 0.91 u.
struct Exp16 {
  static constexpr double log2_theta = 0.432959407;  // log2(1.35)
  static constexpr double c1 = -0.0003993090734898885, c2 = -0.0030127123599242166;
  static constexpr double c5 = -0.03196414960327262, d3 = 0.040815806089214327, c4 = -0.39545222026856774;
  static constexpr double c6 = -0.01103790340919103, e7 = 0.2604228996754721, c8 = -0.23508956851678042;
  static constexpr double c9 = -0.05344609448196047, c10 = -5.750618097503602, c11 = 2.232586953282441;
  static constexpr double f10 = -0.18381361717989209, c12 = 10.5094951224409, c13 = 3.2977060818395096;
  static constexpr double g14 = -2.0158897007186147;
};

// Degree 8 in three products (Sastre 2018), chosen the same way:
//   Y = X2 (c1 X2 + c2 X),  T = (Y + c3 X2 + c4 X)(Y + c5 X2) + c6 Y + c7 X2 + X + I
struct Exp8 {
  static constexpr double log2_theta = -3.03504695;  // log2(0.122), error 0.87 u
  static constexpr double c1 = 0.004978946898829842, c2 = 0.019933608254570908, c3 = 0.07662448691586549;
  static constexpr double c4 = 0.8764144687047127, c5 = 0.12252216956947627, c6 = 2.9741963303388514;
  static constexpr double c7 = 0.5000000000000101;
};

// The degree-16 form with the Taylor polynomial through X^15 (the one-wave-per-sample kernel and its
// four-sample form), theta_15+ = 0.67642
struct Taylor16 {
  static constexpr double c1 = -4.01876161020103546293293287596e-4, c2 = -2.94553144027968298047549126357e-3;
  static constexpr double c3 = 8.70906657683767596765346131523e-3, c4 = -4.01756844067356780152362494573e-1;
  static constexpr double c5 = -3.23076288812231208197540935626e-2, c6 = 2.33731940471157926649827413344e-2;
  static constexpr double c7 = 2.61492797729811710806033238185e-1, c8 = -2.38107037387098722469262858218e-1;
  static constexpr double c9 = -4.1302763659297829110328428344e-2, c10 = -5.79236170707326052179805145605e0;
  static constexpr double c11 = 2.22420917249637356119032703879e0, c12 = 1.04080173523135436461532671084e1;
  static constexpr double c13 = 3.03012340073871230596564458406e0, c14 = -2.12975559049643578453357460382e0;
  static constexpr double d3 = c3 - c5, e7 = c7 - c6 * c5, f10 = -c10 * c5, g14 = c14 - c13 * c5;
  static constexpr double log2_theta = -0.5640051;
};

}  // namespace pib
