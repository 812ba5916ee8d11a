"""The polynomials of pib_expm.hpp: the constants as compiled, read from the header, expanded
exactly and compared with e^x, and their matrix forms against eigh.

A symmetric X's polynomial errs, in the 2-norm, by its largest scalar error over the eigenvalues,
so the truncation bound is |p(x) - e^x| <= u e^x on [-theta, theta], u the unit roundoff of the
kernel's format (FP64). The matrix forms are restated in NumPy as the kernels evaluate them and checked normwise: |M - M_eigh|_max <= 16 (2^s + 16) max(1, |X|_2) u |M|_max,
as for the other forms (tests/test_expm_form.py): each squaring doubles the relative error, and
eigh's own M carries errors of order |X|_2 u."""
import os
import re
from fractions import Fraction

import numpy as np
import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pibronic_amd", "csrc", "pib_expm.hpp")
U64 = 2.0 ** -53


def _coefficients(struct):
    text = open(HEADER).read()
    body = text[text.index(f"struct {struct} {{"):]
    body = body[:body.index("};")]
    return {k: np.float64(v) for k, v in re.findall(r"\b([cdefg]\d+|log2_theta) = (-?[\d.]+(?:e-?\d+)?)", body)}


def _mul(a, b):
    r = [Fraction(0)] * (len(a) + len(b) - 1)
    for i, x in enumerate(a):
        for j, y in enumerate(b):
            r[i + j] += x * y
    return r


def _sum(*terms):
    n = max(len(p) for _, p in terms)
    return [sum((Fraction(c) * (p[i] if i < len(p) else 0) for c, p in terms), Fraction(0)) for i in range(n)]


X, X2, ONE = [Fraction(0), Fraction(1)], [Fraction(0), Fraction(0), Fraction(1)], [Fraction(1)]


def _exact(struct):
    c = {k: Fraction(float(v)) for k, v in _coefficients(struct).items()}
    if struct == "Exp16":
        G = _sum((1, _mul(X2, _sum((c["c1"], X2), (c["c2"], X)))), (c["c5"], X2))
        Y = _sum((1, _mul(_sum((1, G), (c["d3"], X2), (c["c4"], X)), G)), (c["c6"], G), (c["e7"], X2))
        return _sum((1, _mul(_sum((1, Y), (c["c8"], X2), (c["c9"], X)),
                             _sum((1, Y), (c["c10"], G), (c["c11"], X), (c["f10"], X2)))),
                    (c["c12"], Y), (c["c13"], G), (c["g14"], X2), (1, X), (1, ONE))
    Y = _mul(X2, _sum((c["c1"], X2), (c["c2"], X)))
    return _sum((1, _mul(_sum((1, Y), (c["c3"], X2), (c["c4"], X)), _sum((1, Y), (c["c5"], X2)))), (c["c6"], Y),
                (c["c7"], X2), (1, X), (1, ONE))


@pytest.mark.parametrize("struct,theta,u", [("Exp16", 1.35, U64), ("Exp8", 0.122, U64)])
def test_truncation_stays_below_the_unit_roundoff(struct, theta, u):
    """On 801 points of [-theta, theta], for the constants as rounded to the format. theta is the
    header's."""
    assert abs(2.0 ** float(_coefficients(struct)["log2_theta"]) / theta - 1.0) < 1e-6
    p = _exact(struct)
    assert p[0] == 1 and p[1] == 1
    worst = 0.0
    for i in range(-400, 401):
        x = Fraction(theta) * i / 400
        e, term = Fraction(0), Fraction(1)
        for k in range(1, 40):
            e += term
            term *= x / k
        v = Fraction(0)
        for ck in reversed(p):
            v = v * x + ck
        worst = max(worst, abs(float((v - e) / e)))
    print(struct, "largest relative error / u", worst / u)
    assert worst <= u


def _expm(struct, X, dtype):
    c = _coefficients(struct)
    I = np.eye(X.shape[-1], dtype=dtype)
    X2 = X @ X
    alpha = np.sqrt(np.linalg.norm(X2, axis=(-2, -1)))
    with np.errstate(divide="ignore"):
        s = np.maximum(0, np.ceil(np.log2(alpha) - float(c["log2_theta"]))).astype(int)
    f = np.ldexp(dtype(1), -s)[..., None, None].astype(dtype)
    x, x2 = X * f, X2 * f * f
    g = {k: dtype(v) for k, v in c.items()}
    if struct == "Exp16":
        G = x2 @ (g["c1"] * x2 + g["c2"] * x) + g["c5"] * x2
        Y = (G + g["d3"] * x2 + g["c4"] * x) @ G + g["c6"] * G + g["e7"] * x2
        T = ((Y + g["c8"] * x2 + g["c9"] * x) @ (Y + g["c10"] * G + g["c11"] * x + g["f10"] * x2)
             + g["c12"] * Y + g["c13"] * G + g["g14"] * x2 + x + I)
    else:
        Y = x2 @ (g["c1"] * x2 + g["c2"] * x)
        T = (Y + g["c3"] * x2 + g["c4"] * x) @ (Y + g["c5"] * x2) + g["c6"] * Y + g["c7"] * x2 + x + I
    for k in range(int(s.max())):
        T = np.where((s > k)[..., None, None], T @ T, T)
    return T, s


@pytest.mark.parametrize("struct,dtype,u,most", [("Exp16", np.float64, U64, 2), ("Exp8", np.float64, U64, 2)])
@pytest.mark.parametrize("n", [1, 4, 6, 8, 12])
def test_matrix_forms_against_eigh(struct, dtype, u, most, n):
    rng = np.random.default_rng(n)
    for norm in 10.0 ** np.arange(-3, most + 0.5, 0.5):
        Z = rng.normal(size=(200, n, n))
        Z = 0.5 * (Z + Z.transpose(0, 2, 1))
        Z *= (norm / np.abs(np.linalg.eigvalsh(Z)).max(axis=1))[:, None, None]
        Z = Z.astype(dtype)
        lam, U = np.linalg.eigh(Z.astype(np.float64))
        want = (U * np.exp(lam)[:, None, :]) @ U.transpose(0, 2, 1)
        got, s = _expm(struct, Z, dtype)
        err = np.max(np.abs(got - want), axis=(1, 2)) / np.max(np.abs(want), axis=(1, 2))
        assert np.all(err <= 16 * (2.0 ** s + 16) * max(1.0, norm) * u), (norm, err.max())
    zero, _ = _expm(struct, np.zeros((1, n, n), dtype=dtype), dtype)
    assert np.array_equal(zero[0], np.eye(n))
