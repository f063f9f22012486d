"""The drop-in's set-up functions work on whole arrays: against the per-cell
and per-step loops they stand for, bit for bit, over edge sizes (no CPML, one
cell, a CPML as wide as the grid, one side only; no steps, a sine that never
starts or never ends)."""
from types import SimpleNamespace as NS

import numpy as np
import pytest

import BaseFDTD11 as B

KEYS = ("eLoss_CPML Ca Cb Cc sigma_Ex C1 C2 C3 mLoss_CPML "
        "den_Hydz den_Exdz kappa_Hy kappa_Ex").split()


def _strip(n, W):
    return list(range(0, W)) + list(range(n - 1, n - W, -1))


def _den(n, W, jj, m, p, kappa):
    den = np.zeros(n)
    for j in range(n):
        if j <= W and m:
            den[j] = 1 / kappa[j]
        elif j >= n - W and p:
            den[j] = 1 / kappa[jj]
            jj -= 1
        else:
            den[j] = 1.0
    return den


@pytest.mark.parametrize("n,W", [(1, 0), (1, 1), (2, 1), (9, 4), (10, 5), (40, 0), (40, 1), (40, 20), (300, 20)])
@pytest.mark.parametrize("m,p", [(True, True), (True, False), (False, True), (False, False)])
def test_strip_coefficients(n, W, m, p):
    rng = np.random.default_rng(n * 100 + W)
    C = NS(**{k: rng.uniform(1, 2, n) for k in KEYS})
    V = NS(Hy=np.zeros(n), plasmaFreqE=1e9, gammaE=1e7, UpExHcompsCo=rng.normal(size=n), UpExMat=rng.normal(size=n))
    P = NS(pmlWidth=W, CPMLXm=m, CPMLXp=p, delT=1.7e-12, permit_0=8.85e-12, permea_0=1.25e-6)
    want = NS(**{k: getattr(C, k).copy() for k in KEYS})
    beta = (0.5 * V.plasmaFreqE * V.plasmaFreqE * P.permit_0 * P.delT) / (1 + 0.5 * V.gammaE * P.delT)
    for z in _strip(n, W):
        want.eLoss_CPML[z] = (C.sigma_Ex[z] * P.delT) / (2 * P.permit_0)
        want.Ca[z] = (2 * P.permit_0 - beta * P.delT) / (2 * P.permit_0 + beta * P.delT)
        want.Cb[z] = V.UpExHcompsCo[z] * V.UpExMat[z]
        want.Cc[z] = P.delT / ((1 + want.eLoss_CPML[z]) * P.permit_0)
        want.C1[z], want.C2[z] = 1, P.delT / P.permea_0
        want.C3[z] = P.delT / ((1 + C.mLoss_CPML[z]) * P.permea_0)
    try:
        want.den_Hydz = _den(n, W, W, m, p, C.kappa_Hy)
        want.den_Exdz = _den(n, W, W - 1, m, p, C.kappa_Ex)
    except IndexError:          # a CPML as wide as the grid: the mirror cell W does not exist
        with pytest.raises(IndexError):
            B.denominators(V, P, C, None)
        return
    B.CPML_Ex_Update_Coef(V, P, C, None)
    B.CPML_Hy_Update_Coef(V, P, C, None)
    B.denominators(V, P, C, None)
    for k in KEYS:
        assert np.array_equal(getattr(C, k), getattr(want, k)), k


@pytest.mark.parametrize("steps,periods", [(0, 3), (1, 0), (1, 3), (500, 0), (500, 2), (500, 10000)])
def test_smooth_turn_on(steps, periods):
    P = NS(c0=2.99792458e8, freq_in=9e9, dz=1.1e-4, courantNo=0.7, timeSteps=steps, delT=2.5e-13,
           period=1 / 9e9, Periods=periods)
    for freq in (0, 7.2e9):
        ppw = P.c0 / ((freq or P.freq_in) * P.dz)
        E, H = [], []
        for t in range(steps):
            live = t * P.delT < P.period * periods
            E.append(float(np.sin(2.0 * np.pi / ppw * (P.courantNo * t))) if live else 0)
            H.append(float(np.sin(2.0 * np.pi / ppw * (P.courantNo * (t + 1)))) if live else 0)
        got = B.SmoothTurnOn(None, P, freq)
        assert got == (E, H)
        assert [type(x) for x in got[0] + got[1]] == [type(x) for x in E + H]
