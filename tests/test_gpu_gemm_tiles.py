"""The order of the output tiles (strips of eight tile columns, an eighth of
them per XCD, none outside a triangle) at sizes around the strips, and slabs
that end inside the operands, against numpy.

Tolerance: an entry is a sum of k products, k eps of the largest of
sum |a| |b| bounds its rounding in any order."""
from __future__ import annotations

import numpy as np
import pytest

import test_gpu_assembly as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("tri", [0, 1, 2])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (64, 65, 17), (512, 512, 16), (513, 513, 15), (1025, 1025, 33),
                                   (577, 130, 20), (130, 577, 20), (1100, 520, 31), (520, 1100, 1)])
def test_tile_order(m, n, k, tri, variant):
    rng = np.random.default_rng(m + 3 * n + 5 * k + tri)
    a, b, c = rng.standard_normal((m, k)), rng.standard_normal((n, k)), rng.standard_normal((m, n))
    got = A._dgemm_tiles("N", "T", m, n, k, 0.7, a, b, -1.3, c, tri, 0, 0, variant)
    want = 0.7 * a @ b.T - 1.3 * c
    i, j = np.indices((m, n))
    inside = np.ones((m, n), bool) if tri == 0 else i >= j if tri == 1 else i <= j
    bound = (k + 2) * np.finfo(float).eps * np.max(np.abs(a) @ np.abs(b).T + 2 * np.abs(c))
    assert np.max(np.abs(got - want)[inside]) <= bound
    assert np.array_equal(got[~inside], c[~inside])
