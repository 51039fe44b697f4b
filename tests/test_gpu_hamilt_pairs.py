"""HAMILT's pair loop with the rows around the tiles that its kernel works in
(64 rows by 2 or 4 columns a wave, four waves a block), against the CPU oracle
on bases cut to that many plane waves.

Tolerance: an entry is a sum over at most 13 l and the atoms (8 at most here)
of four products, each factor good to a few eps and P_l to 13: below 1000
terms of rounding, 1000 eps of the largest entry."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from conftest import Fixture, PKG
from test_gpu_hns_rows import _cut

pytestmark = pytest.mark.gpu
L = PKG.lapw1


@pytest.mark.parametrize("name,nv", [("c1_fcc", 1), ("c1_fcc", 2), ("c1_fcc", 31), ("c1_fcc", 33), ("mgo", 15), ("mgo", 16),
                                     ("mgo", 17), ("mgo", 63), ("mgo", 64), ("mgo", 65), ("lo_cplx", 15), ("lo_cplx", 17),
                                     ("lo_cplx", 32), ("lo_cplx", 97), ("lo_mult2", 65), ("rs8", 48), ("rs8", 129)])
def test_rows_around_the_tiles(name, nv):
    fx = Fixture(name)
    run, b = fx.run(), _cut(fx.basis(0), nv)
    hs, hd, al, bl = O.hamilt(run, b)
    ctx = L.Lapw1(run)
    ctx.set_basis(b)
    ctx.hamilt()
    got, gd = ctx.get_hs()
    ctx.close()
    eps = 1000 * np.finfo(float).eps
    assert np.max(np.abs(np.triu(got) - np.triu(hs))) <= eps * np.max(np.abs(np.triu(hs)))
    assert np.max(np.abs(np.tril(got, -1) - np.tril(hs, -1)), initial=0.0) <= eps * max(np.max(np.abs(hd)), np.max(np.abs(hs)))
    assert np.max(np.abs(gd - hd)) <= eps * np.max(np.abs(hd))
