"""The two-stage tridiagonalisation (twostage.hip) at the sizes where its parts
change: below one band, panels of fewer rows than columns, sweeps that end on
a block's first or last row, one to several work-groups per panel, and
matrices whose panels vanish (diagonal), are rank-deficient (few plane waves
coupled) or need no first stage (banded).  S is the identity, so that the
eigenproblem is H's own.

Tolerances: both stages are products of Householder reflectors, whose
backward error grows at most linearly in their number: 8 n eps |H| for the
eigenvalues, and for the vectors 8 n eps (orthogonality) and ten times that
relative to |H| (residual), neither below 1e-12.  The low-rank kind has
eigenvalues of multiplicity five and more: its vectors are held to the 1e-10
of the other degenerate spectra's tests, since inverse iteration's nearly
parallel vectors of one eigenvalue, once made orthogonal, carry up to 1e-11
of eigenvectors far away (with the column-by-column reduction too); its
eigenvalues are held to the bound above."""
from __future__ import annotations

import numpy as np
import pytest
import scipy.linalg as sla

from conftest import EMU
from test_gpu_seclr4 import _run_pencil

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 31, 32, 33, 34, 35, 63, 64, 65, 66, 96, 97, 98, 129, 161, 289, 290, 321]


def _matrix(n, kind, cplx):
    rng = np.random.default_rng(1000 * n + cplx)
    H = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
    H = (H + H.conj().T) / 2
    if kind == "banded":
        H = np.triu(np.tril(H, 32), -32)
    elif kind == "diagonal":
        H = np.diag(np.sort(rng.standard_normal(n))).astype(H.dtype)
    elif kind == "low rank":
        X = H[:, :3]
        H = np.diag(np.repeat(np.arange((n + 7) // 8), 8)[:n] + 0.0) + X @ X.conj().T / n
    return H


@pytest.mark.parametrize("cplx", [0, 1])
@pytest.mark.parametrize("kind", ["dense", "banded", "diagonal", "low rank"])
@pytest.mark.parametrize("n", SIZES + [600])
def test_two_stage_edges(n, kind, cplx):
    if EMU and (n > 300 or (n > 100 and kind != "dense")):
        pytest.skip("too large for the CPU emulation")
    H = _matrix(n, kind, cplx)
    ne, nb, ev, z = _run_pencil(H, np.eye(n, dtype=H.dtype), 1.0, 0.0, n)
    scale, tol = np.linalg.norm(H, 2), 8 * n * np.finfo(float).eps
    assert ne == n and nb == 0
    assert np.max(np.abs(ev - sla.eigvalsh(H))) <= tol * scale
    vtol = 1e-10 if kind == "low rank" else max(tol, 1e-12)
    assert np.max(np.abs(z.conj().T @ z - np.eye(n))) <= vtol
    assert np.max(np.abs(H @ z - z * ev)) <= 10 * vtol * max(scale, 1.0)
