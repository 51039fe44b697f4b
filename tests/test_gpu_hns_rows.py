"""HNS with the rows around the blocks that its operand kernel works in (64
rows, the last of them with local orbitals), against the CPU oracle on bases
cut to that many plane waves.

Tolerance: an entry is a sum of 4 sum(LINDEX) products of factors that are
sums of 75 terms themselves, all below 1000 terms of rounding each: 1000 eps
of the largest entry."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from conftest import Fixture, PKG

pytestmark = pytest.mark.gpu
L = PKG.lapw1


def _cut(b, nv):
    keep = np.r_[np.arange(nv), np.arange(b.nv, b.n)]
    return L.Basis(nv, b.nlo, b.kzz[:, keep], b.xk[keep], b.yk[keep], b.zk[keep], b.rk[keep])


@pytest.mark.parametrize("name,nv", [("c1_fcc", 1), ("c1_fcc", 17), ("mgo", 58), ("mgo", 59), ("mgo", 60), ("mgo", 64),
                                     ("mgo", 127), ("lo_cplx", 47), ("lo_cplx", 55), ("lo_cplx", 64), ("lo_cplx", 128),
                                     ("rs8", 95), ("rs8", 96), ("rs8", 161)])
def test_rows_around_the_blocks(name, nv):
    fx = Fixture(name)
    run, b = fx.run(), _cut(fx.basis(0), nv)
    hs, hd, al, bl = O.hamilt(run, b)
    hs, hd = O.swap_diag(hs, hd)
    ref = O.hns(run, b, al, bl, hs)
    ctx = L.Lapw1(run)
    ctx.set_basis(b)
    ctx.hamilt()
    ctx.swap_diag()
    before, _ = ctx.get_hs()
    ctx.hns()
    got, _ = ctx.get_hs()
    ctx.close()
    add, want = got - before, ref - hs
    assert np.max(np.abs(np.tril(add) - np.tril(want))) <= 1000 * np.finfo(float).eps * np.max(np.abs(ref))
    assert np.array_equal(np.triu(got, 1), np.triu(before, 1))
