"""The Cholesky block kernels (factor and inverse of a 64 x 64 block by 16 x 16
pieces) at orders around the pieces and the blocks, through the generalised
eigenproblem with an ill-scaled overlap, against LAPACK.

Tolerance: the standard form's backward error is of order n eps times
kappa(S) |H| / |S|; S = D (I + E) D with |E| <= 1/4 and D of 1 to 2 has
kappa below 8, so that eigenvalues agree to 64 n eps of the largest."""
from __future__ import annotations

import numpy as np
import pytest
import scipy.linalg as sla

from test_gpu_seclr4 import _run_pencil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 128, 129])
def test_block_orders(n, cplx):
    rng = np.random.default_rng(7 * n + cplx)

    def hermitian():
        a = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
        return (a + a.conj().T) / 2

    H, E = hermitian(), hermitian()
    d = rng.uniform(1.0, 2.0, n)
    S = np.eye(n) + E / (4 * max(np.linalg.norm(E, 2), 1.0))
    S = d[:, None] * S * d[None, :]
    ref = sla.eigh(H, S, eigvals_only=True)
    ne, nb, ev, z = _run_pencil(H, S, ref[-1] + 1.0, ref[0] - 1.0, n)
    tol = 64 * n * np.finfo(float).eps
    assert ne == n and nb == 0
    assert np.max(np.abs(ev - ref)) <= tol * np.max(np.abs(ref))
    assert np.max(np.abs(z.conj().T @ S @ z - np.eye(n))) <= max(tol, 1e-12)
