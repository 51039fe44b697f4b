"""The application of Q2 in ranges of sweep groups (twostage.hip): all groups at
once and as few at a time as the workspace can be made to hold
(W2K_TEST_Q2_OPERANDS doubles of operands, never less than the longest group)
do the same operations in the same order, so that eigenvectors agree bit for
bit: at one group, at orders around a group's 32 sweeps, and with the two sets
of columns that many real vectors take."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import EMU
from test_gpu_seclr4 import _run_pencil

pytestmark = pytest.mark.gpu

BLOCK = 4096  # operands of a block, doubles per plane


@pytest.mark.parametrize("n,nume,cplx", [(2, 2, 0), (33, 33, 1), (34, 34, 0), (65, 65, 1), (66, 5, 0), (161, 161, 0),
                                         (162, 33, 1), (290, 17, 0), (1100, 600, 0), (1100, 600, 1)])
def test_ranges_agree_bit_for_bit(n, nume, cplx, monkeypatch):
    if EMU and n > 300:
        pytest.skip("too large for the CPU emulation")
    rng = np.random.default_rng(3 * n + cplx)
    H = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
    H = (H + H.conj().T) / 2
    S = np.eye(n, dtype=H.dtype)
    ne, nb, ev, z = _run_pencil(H, S, 1.0, 0.0, nume)
    assert ne == nume
    groups = (n + 30) // 32
    for ops in (0, (groups + 2) * BLOCK * (2 if cplx else 1)):
        monkeypatch.setenv("W2K_TEST_Q2_OPERANDS", str(ops))
        _, _, ev2, z2 = _run_pencil(H, S, 1.0, 0.0, nume)
        assert np.array_equal(ev, ev2) and np.array_equal(z, z2), ops
