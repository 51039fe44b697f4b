"""w2k_seclr4_noalloc up to its largest order: every order up to
W2K_NOALLOC_MAXN = 768 fits the scratch with all its vectors, in both builds.
Complex 705 is the first order whose workspaces pass 128 MiB.  Same kernels
and same matrix as w2k_seclr4, compared as in test_zz_no_alloc."""
from __future__ import annotations

import pytest

import test_zz_no_alloc as T
from conftest import Fixture, PKG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,n", [("c1_fcc", 768), ("lo_cplx", 704), ("lo_cplx", 705), ("lo_cplx", 768)])
def test_largest_orders_fit(name, n):
    fx = Fixture(name)
    run = fx.run()
    hs, hd = T._pack(*T._pencil(n, fx.is_complex, n))
    ref = T._regular(run, hs, hd, 1.0, 0.0, n)
    ctx = PKG.lapw1.Lapw1(run)
    T._compare(T._noalloc(ctx, hs, hd, 1.0, 0.0, n), ref, hs, hd)
    ctx.close()
