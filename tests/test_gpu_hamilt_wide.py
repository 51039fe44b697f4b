"""HAMILT's pair loop with four columns a wave in the complex build, which bases
from 2560 plane waves on take: a hundred-atom cell cut to plane-wave counts
around that line and around the tiles, compared with the CPU oracle on the same
cell with some of these plane waves (an entry depends on its own two plane waves
only): the first and last ones, some in the middle and a random choice.

Tolerance: an entry is a sum over at most 13 l and 100 atoms of four products,
each factor good to a few eps and P_l to 13: below 10^4 terms of rounding, 10^4
eps of the largest entry."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as O
from conftest import Fixture, PKG
from test_gpu_hns_rows import _cut

pytestmark = [pytest.mark.gpu, pytest.mark.big]
L = PKG.lapw1

NVS = (2559, 2560, 2561, 2563, 2576, 2625)


@pytest.fixture(scope="module")
def cell():
    fx = Fixture("c3_lowsym100")
    run, b = fx.run(), _cut(fx.basis(0), max(NVS))
    rng = np.random.default_rng(17)
    pick = np.r_[:66, 1270:1290, 2490:max(NVS), rng.choice(np.arange(66, 2490), 60, replace=False)]
    pick = np.unique(pick)
    keep = np.r_[pick, np.arange(b.nv, b.n)]
    part = L.Basis(len(pick), b.nlo, b.kzz[:, keep], b.xk[keep], b.yk[keep], b.zk[keep], b.rk[keep])
    hs, hd, _, _ = O.hamilt(run, part)
    return run, b, pick, hs, hd


@pytest.mark.parametrize("nv", NVS)
def test_four_columns_a_wave(cell, nv):
    run, b, pick, hs, hd = cell
    ctx = L.Lapw1(run)
    ctx.set_basis(_cut(b, nv))
    ctx.hamilt()
    got, gd = ctx.get_hs()
    ctx.close()
    have = pick < nv
    mine = np.r_[pick[have], nv + np.arange(b.nlo)]
    ref = np.r_[np.nonzero(have)[0], len(pick) + np.arange(b.nlo)]
    got, gd, hs, hd = got[np.ix_(mine, mine)], gd[mine], hs[np.ix_(ref, ref)], hd[ref]
    eps = 1e4 * np.finfo(float).eps
    assert np.max(np.abs(np.triu(got) - np.triu(hs))) <= eps * np.max(np.abs(np.triu(hs)))
    assert np.max(np.abs(np.tril(got, -1) - np.tril(hs, -1))) <= eps * max(np.max(np.abs(hd)), np.max(np.abs(hs)))
    assert np.max(np.abs(gd - hd)) <= eps * np.max(np.abs(hd))
