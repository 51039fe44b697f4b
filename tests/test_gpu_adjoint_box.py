"""Box gradient of the band energy (k_adj_warp_grad) at orders where its split
matters: 16 slices of the pairs' first index, four at a time, 64 box entries a
block.  c1_fcc has empty slices and slices shorter than four, rs8 and
c4_ortho8 remainders in each slice; no box is a multiple of 64 entries.

The reference is the same sum on the host over the returned vectors.  A box
entry adds at most nv products Gamma, so any order of the additions agrees to
nv eps times the sum of their moduli; Gamma itself, a product over ne vectors,
to ne eps times sum_n f_n |z(I,n)||z(J,n)|.  The bound is the sum of the two."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import Fixture, PKG

pytestmark = pytest.mark.gpu
L = PKG.lapw1


@pytest.mark.parametrize("name", ["c1_fcc", "rs8", "c4_ortho8"])
def test_box_gradient_matches_host_sum(name):
    fx = Fixture(name)
    kd, basis = fx.k(0), fx.basis(0)
    ctx = L.Lapw1(L.RunData(fx.run_arrays, fx.is_complex))
    ctx.set_basis(basis)
    ctx.calkpt(float(kd["EL"]), float(kd["EU"]), int(kd["NUME"]))
    ev, z = ctx.get_eig()
    f = np.linspace(2.0, 0.1, len(ev))
    _, g = ctx.adjoint_warp(f)
    ctx.close()
    nv, half = basis.nv, [s // 2 for s in g.shape]
    kzz, zz = basis.kzz[:, :nv].T.astype(np.int64), z[:nv, :]
    gam = (zz * f) @ zz.conj().T
    mod = (np.abs(zz) * f) @ np.abs(zz).T
    ref, size = np.zeros(g.shape, np.complex128), np.zeros(g.shape)
    for i in range(nv):
        q = kzz[: i + 1] - kzz[i]
        t = q + half
        ok = np.all((t >= 0) & (t < g.shape), axis=1)
        v = 2.0 * gam[i, : i + 1].conj()
        v[i] = gam[i, i].real
        at = tuple(t[ok].T)
        np.add.at(ref, at, v[ok] if fx.is_complex else v[ok].real)
        np.add.at(size, at, 2.0 * mod[i, : i + 1][ok])
    assert np.all(np.abs(g - ref) <= (nv + len(ev) + 8) * np.finfo(float).eps * size)
