"""ATPAR's local-orbital functions and its integrals with the non-spherical
potential at mesh lengths around the pieces that the kernels work in, against
the same formulas in extended precision (outwin.f:20-112, atpar.f:212-330,
atpar.f:489-552, rint13.f), for cells with local orbitals of several l and
types with one, two and none.

Tolerance, as in test_gpu_atpar_mesh: a function is good to 8 n eps of its
norm, an energy derivative to that times 4 (0.25 / 2e-3) of the function's norm
(1). An integral of f V g errs by |V|max (df |g| + |f| dg) with the norms |f|
and |g| (Cauchy and Schwarz), and by the n eps of its own sum, which is below."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import Fixture, PKG
from test_gpu_atpar import _radial
from test_gpu_atpar_mesh import X, _outwin, _rint13

pytestmark = pytest.mark.gpu
L = PKG.lapw1


@pytest.mark.parametrize("name", ["lo_mult2", "lo_cplx"])
@pytest.mark.parametrize("n", [5, 6, 63, 64, 65, 67, 128, 129, 640, 781])
def test_orbitals_and_integrals(name, n):
    fx = Fixture(name)
    rad, arr = _radial(fx), fx.run_arrays
    vr, vlm = np.array(rad["vr"])[:n], np.array(rad["vlm"])[:n]
    nat = vr.shape[1]
    ro, dh = (np.atleast_1d(rad[k]).astype(float) for k in ("ro", "dh"))
    ctx = L.Lapw1(fx.run())
    out = ctx.atpar(rel=rad["rel"], jrj=np.full(nat, n, np.int32), ro=ro, dh=dh, zz=rad["zz"], vr=vr, vlm=vlm)
    ctx.close()
    c2 = 1 / X(137.0359895) ** 2 if rad["rel"] else X(1e-22)
    de = X(2e-3)
    di = X(0.25) / de
    eps = 8 * n * np.finfo(float).eps
    loor, ilo = np.asarray(arr["LOOR"]).astype(bool), np.asarray(arr["ILO"])
    count = [0, 0, 0]
    for a in range(nat):
        r0, dx, v = X(ro[a]), X(dh[a]), vr[:, a].astype(X)
        rn = ro[a] * np.exp(dh[a] * (n - 1))

        def integral(f, g, w=1):
            return _rint13(r0, dx, n, (f[0] * g[0] + c2 * f[1] * g[1]) * w)

        def function(e, l):
            f = _outwin(rad["rel"], v, r0, dx, n, e, l, X(rad["zz"][a]))
            return [t / np.sqrt(integral(f, f)) for t in f]

        u, ue, lo = {}, {}, {}
        for l in range(5):
            ei = X(out["e"][l, a]) / 2
            f1, f2, u[l] = (function(e, l) for e in (ei - de, ei + de, ei))
            d = [di * (f2[i] - f1[i]) for i in (0, 1)]
            tr = -integral(u[l], d)
            ue[l] = [d[i] + tr * u[l][i] for i in (0, 1)]
            if l < 4 and loor[l, a]:
                lo[l] = function(X(arr["ELO"][l, ilo[l, a] - 1, a]) / 2, l)
        # (function, its error, its norm)
        size = {"u": (u, eps, lambda l: 1), "e": (ue, 4 * di * eps, lambda l: np.sqrt(integral(ue[l], ue[l]))),
                "o": (lo, eps, lambda l: 1)}

        def check(got, p, lp, q, lq, w=1):
            (f, df, nf), (g, dg, ng) = size[p], size[q]
            tol = np.max(np.abs(w)) * (df * ng(lq) + nf(lp) * dg + df * dg)
            assert abs(got - integral(f[lp], g[lq], w)) <= tol, (a, p, lp, q, lq)

        for l in lo:
            assert abs(out["plo"][l, a] - lo[l][2]) <= eps * abs(lo[l][2])
            assert abs(out["dplo"][l, a] - lo[l][3]) <= eps * (abs(lo[l][3]) + abs(lo[l][2]) / rn)
            check(out["pi12lo"][l, a], "u", l, "o", l)
            check(out["pe12lo"][l, a], "e", l, "o", l)
            count[0] += 1
        for k, key, p, q in ((1, "vns1", "u", "u"), (1, "vns2", "e", "e"), (1, "vns3", "u", "e"),
                             (2, "vns1lo", "o", "u"), (2, "vns2lo", "o", "e"), (2, "vns3lo", "o", "o")):
            t = out[key][..., a]
            for l0, lm, lp in zip(*np.nonzero(t)):
                check(t[l0, lm, lp], p, l0, q, lp, vlm[:, lm, a].astype(X))
                count[k] += 1
    assert min(count) > 0, count
