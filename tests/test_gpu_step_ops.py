"""The single step functions' device call (fdtd_step_op) against the same
expression in numpy, bit for bit: one range, two ranges, ranges of one cell,
ranges that touch the arrays' ends or are empty, arrays of different lengths,
growing and shrinking calls through one context.  Cells outside the ranges
keep their values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ranges", [
    (3, ((1, 2), (0, 0))), (3, ((0, 0), (1, 3))), (40, ((1, 20), (20, 40))), (300, ((1, 25), (275, 300))),
    (300, ((1, 300), (0, 0))), (300, ((5, 5), (9, 8))), (70001, ((1, 70001), (0, 0))), (250001, ((2, 120000), (125000, 250001))), (700, ((1, 257), (443, 700)))])
def test_ranges(n, ranges):
    from fdtd_pic_amd.single_step import run_op
    rng = np.random.default_rng(n)
    x = [rng.normal(size=n + (k == 3)) for k in range(6)]
    E, psi, H, b, c, Cb = [v.copy() for v in x]
    for lo, hi in ranges:
        s = np.arange(lo, max(hi, lo))
        psi[s] = b[s] * psi[s] + c[s] * (H[s] - H[s - 1])
        E[s] = E[s] - Cb[s] * psi[s]
    got = run_op(2, [v.copy() for v in x], (), ranges)
    assert np.array_equal(got[0], E) and np.array_equal(got[1], psi)
    for k in range(2, 6):
        assert np.array_equal(got[k], x[k])
    D, H, P = x[0], x[2], x[4]
    out = run_op(13, [D.copy(), x[1].copy(), H, P], (0.3, 1.7, 2.9), ranges)
    wD, wE = D.copy(), x[1].copy()
    for lo, hi in ranges:
        s = np.arange(lo, max(hi, lo))
        wD[s] = D[s] + (H[s] - H[s - 1]) * 0.3 / 1.7
        wE[s] = (wD[s] - P[s]) / 2.9
    assert np.array_equal(out[0], wD) and np.array_equal(out[1], wE)
