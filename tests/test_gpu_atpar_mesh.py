"""ATPAR's radial part at mesh lengths around the pieces that the kernels work
in (64 points, even and odd counts, the shortest mesh), against the same
formulas in extended precision (outwin.f:20-112, atpar.f:212-289, rint13.f).

Tolerance: every mesh point adds a few rounding errors to the recurrence and a
sum, so the functions are good to 8 n eps of their size, and the slope of u / r
at the mesh's end r_n, a difference of u' / r and u / r^2, to that of either
term; the energy derivative is the difference of two functions times
0.25 / 2e-3."""
from __future__ import annotations

import os
import sys

import numpy as np
import pytest

from conftest import Fixture, PKG, REPO

pytestmark = pytest.mark.gpu
L = PKG.lapw1
sys.path.insert(0, os.path.join(REPO, "tests"))
from test_gpu_atpar import _radial  # noqa: E402

X = np.longdouble


def _outwin(rel, v, ro, dh, n, eh, l, z):
    c = 2 * X(137.0359895) if rel else X(1e10)
    f, h, r1 = X(l) * (l + 1), X(8) / 3, X(1) / 9
    if z < 0.9:
        s, sf, f0 = X(l + 1), X(l), X(l) / c
    else:
        aa = 2 * z / c
        s = sf = np.sqrt(f + 1 - aa * aa)
        f0 = (s - 1) / aa
    r = ro * np.exp(dh * np.arange(n).astype(X))
    a, b = np.zeros(n, X), np.zeros(n, X)
    a[:3], b[:3] = r[:3] ** s, r[:3] ** sf * f0
    da, db = list(dh * a[:3] * s), list(dh * b[:3] * sf)
    phi = (2 * eh - 2 * v / r) * dh * r / c
    u = dh * r * c + phi
    y = -f * dh * dh / u + phi
    det = X(64) / 9 - dh * dh + u * y
    for k in range(3, n):
        p = a[k - 1] * h + r1 * da[0] - 5 * r1 * da[1] + 19 * r1 * da[2]
        q = b[k - 1] * h + r1 * db[0] - 5 * r1 * db[1] + 19 * r1 * db[2]
        a[k] = (p * (h + dh) + q * u[k]) / det[k]
        b[k] = (q * (h - dh) - p * y[k]) / det[k]
        da = [da[1], da[2], u[k] * b[k] + dh * a[k]]
        db = [db[1], db[2], -dh * b[k] - y[k] * a[k]]
    val = a[-1] / r[-1]
    return a, b * c / 2, val, (da[2] / (dh * r[-1]) - val) / r[-1]


def _rint13(ro, dx, n, f):
    r = ro * np.exp(dx * np.arange(n).astype(X))
    k0 = 2 - n % 2
    w = np.zeros(n, X)
    w[k0:n - 1:2], w[k0 + 1:n - 1:2] = 4, 2
    w[n - 1] = 1
    w *= r * dx / 3
    w[k0 - 1] += dx * r[k0 - 1] / 3
    w[0] += ro / 3
    if k0 > 1:
        w[0] += dx * ro / 2
        w[k0 - 1] += dx * r[k0 - 1] / 2
    return (w * f).sum()


@pytest.mark.parametrize("n", [5, 6, 63, 64, 65, 66, 67, 128, 129, 323, 640])
def test_mesh_lengths(n):
    fx = Fixture("c1_fcc")
    rad = _radial(fx)
    vr = np.array(rad["vr"])[:n]
    jrj = np.full(np.atleast_1d(rad["jrj"]).shape, n, np.int32)
    ro, dh = (np.atleast_1d(rad[k]).astype(float) for k in ("ro", "dh"))
    rn = ro * np.exp(dh * (n - 1))  # where the mesh ends
    ctx = L.Lapw1(fx.run())
    out = ctx.atpar(rel=rad["rel"], jrj=jrj, ro=ro, dh=dh, zz=rad["zz"], vr=vr, vlm=None)
    ctx.close()
    c2 = 1 / X(137.0359895) ** 2 if rad["rel"] else X(1e-22)
    de = X(2e-3)
    di = X(0.25) / de
    for l in (0, 1, 4, int(fx.run_arrays["LTOP"]) - 1):
        ei = X(out["e"][l, 0]) / 2
        fs = [_outwin(rad["rel"], vr[:, 0].astype(X), X(ro[0]), X(dh[0]), n, e, l, X(rad["zz"][0]))
              for e in (ei - de, ei + de, ei)]
        t = [1 / np.sqrt(_rint13(X(ro[0]), X(dh[0]), n, f[0] ** 2 + c2 * f[1] ** 2)) for f in fs]
        a, b = t[2] * fs[2][0], t[2] * fs[2][1]
        ae, be = (di * (t[1] * fs[1][i] - t[0] * fs[0][i]) for i in (0, 1))
        tr = -_rint13(X(ro[0]), X(dh[0]), n, a * ae + c2 * b * be)
        p, dp = t[2] * fs[2][2], t[2] * fs[2][3]
        pe, dpe = (di * (t[1] * fs[1][i] - t[0] * fs[0][i]) + tr * t[2] * fs[2][i] for i in (2, 3))
        eps = 8 * n * np.finfo(float).eps
        assert abs(out["p"][l, 0] - p) <= eps * abs(p)
        assert abs(out["dp"][l, 0] - dp) <= eps * (abs(dp) + abs(p) / rn[0])
        assert abs(out["pe"][l, 0] - pe) <= 4 * di * eps * abs(p)
        assert abs(out["dpe"][l, 0] - dpe) <= 4 * di * eps * (abs(dp) + abs(p) / rn[0])
        # the integral of a square whose values err by 4 di eps of the function's
        pei = _rint13(X(ro[0]), X(dh[0]), n, (ae + tr * a) ** 2 + c2 * (be + tr * b) ** 2)
        assert abs(out["pei"][l, 0] - pei) <= 8 * di * eps * np.sqrt(abs(pei)) + (4 * di * eps) ** 2
