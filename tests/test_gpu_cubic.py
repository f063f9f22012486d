"""Root 0 of the reference's cubic on the device (one step op per call), over
every branch of the closed form, against the oracle's.  Two correct FP64
evaluations differ by what their roundings move the root: the bound follows
the relative rounding of g and h (a few eps of the terms they sum) through
the branch's cube roots or its arc cosine, for the two sides together."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _bound(a, b, c, d):
    """Difference that the roundings of one evaluation may cause, twice."""
    if a == 0.0:
        if b == 0.0:
            return 8 * EPS * abs(d / c)
        disc = c * c - 4 * b * d
        ed = 8 * EPS * (c * c + abs(4 * b * d))
        er = min(ed / (2 * np.sqrt(disc)), np.sqrt(ed)) if disc > 0 else 0.0
        return 2 * (er + 4 * EPS * (abs(c) + np.sqrt(abs(disc)))) / abs(2 * b)
    f = (3 * c / a - b * b / (a * a)) / 3
    g = (2 * b**3 / a**3 - 9 * b * c / a**2 + 27 * d / a) / 27
    h = g * g / 4 + f**3 / 27
    ef = 8 * EPS * (abs(3 * c / a) + b * b / (a * a)) / 3
    eg = 8 * EPS * (abs(2 * b**3 / a**3) + abs(9 * b * c / a**2) + abs(27 * d / a)) / 27
    eF = f * f * ef / 9 + 8 * EPS * abs(f**3) / 27
    eh = abs(g) * eg / 2 + eF + 8 * EPS * g * g / 4
    shift = abs(b / (3 * a))

    def cube(x, e):      # |cbrt(x') - cbrt(x)| for |x' - x| <= e, and its own rounding
        lip = e / (3 * (abs(x) - e) ** (2 / 3)) if abs(x) > e else np.inf
        return min(lip, 1.6 * e ** (1 / 3)) + 4 * EPS * abs(x) ** (1 / 3)

    if h <= 0:
        i = np.sqrt(max(g * g / 4 - h, 0.0))
        ei = min(eh / i, np.sqrt(eh)) if i > 0 else np.sqrt(eh)
        x = min(1.0, abs(g / (2 * i))) if i > 0 else 1.0
        ex = (eg / 2 + ei * x) / i + 4 * EPS if i > 0 else 0.0
        ek = min(ex / np.sqrt(1 - x * x), np.sqrt(2 * ex) * 1.6) if x < 1 else np.sqrt(2 * ex) * 1.6
        j = i ** (1 / 3)
        return 2 * (2 * (j * (ek / 3 + 8 * EPS) + cube(i, ei)) + 8 * EPS * shift)
    sh = np.sqrt(h)
    es = min(eh / (2 * sh), np.sqrt(eh)) + 2 * EPS * sh
    e = eg / 2 + es + 4 * EPS * (abs(g) + sh)
    return 2 * (cube(-g / 2 + sh, e) + cube(-g / 2 - sh, e) + 8 * EPS * shift)


@pytest.mark.parametrize("a,b,c", [
    (0.09, 1.5, 6.25),          # the Kerr slab's shape: positive, monotone over the range
    (0.09, -0.9, 3.1),
    (2.0, -6.0, 3.0),           # three real roots for middle d
    (1.0, 0.0, -7.0),
    (-1.0, 2.0, 5.0),
    (1.0, 0.0, 0.0),            # triple root at d = 0 only: f = 0
    (1.0, -6.0, 12.0),          # triple root at d = -8
    (1.0, 0.0, 4.0),
    (0.0, 2.0, -3.0),           # quadratic, both signs of the discriminant
    (0.0, 0.0, 3.0),            # linear
])
def test_cubic_root_branches(a, b, c):
    from fdtd_pic_amd.single_step import run_op
    from oracle.cubic import root0_1728
    d = np.concatenate([np.linspace(-9.0, 0.0, 181), -10.0 ** np.linspace(-10, 6, 161)])
    D = np.sqrt(-d)
    d = -(np.abs(D) * np.abs(D))            # the operand the op forms
    got = run_op(7, [np.zeros_like(D), D], (a, b, c, 1.0), ((0, D.size), (0, 0)))[0]
    ref = np.array([root0_1728(a, b, c, x) for x in d])
    tol = np.array([_bound(a, b, c, x) if abs(x) > 1e-8 else 0.0 for x in d])
    worst = int(np.argmax(np.abs(got - ref) - tol))
    assert np.all(np.abs(got - ref) <= tol), (d[worst], got[worst], ref[worst], tol[worst])
    assert np.all(got[np.abs(d) <= 1e-8] == 0.0)
