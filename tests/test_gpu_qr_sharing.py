"""The panel QR of the two-stage tridiagonalisation with fewer work-groups than
blocks of rows, as when the others find no room beside other streams' work: they
share the blocks, whose columns then go through memory, and take the same sums
in the same order. So eigenvalues and vectors agree bit for bit with those of
panels that have a work-group for each block. Orders of several blocks with a
ragged last one; W2K_TEST_QR_GROUPS sets how many work-groups share."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import EMU
from test_gpu_seclr4 import _run_pencil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cplx", [(289, 0), (290, 1), (877, 0), (877, 1), (1380, 0)])
def test_shared_panels_agree_bit_for_bit(n, cplx, monkeypatch):
    if EMU and n > 300:
        pytest.skip("too large for the CPU emulation")
    rng = np.random.default_rng(5 * n + cplx)
    H = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
    H = (H + H.conj().T) / 2
    S = np.eye(n, dtype=H.dtype)
    ne, nb, ev, z = _run_pencil(H, S, 1.0, 0.0, 40)
    assert ne == 40
    assert np.max(np.abs(ev - np.linalg.eigvalsh(H)[:40])) <= 8 * n * np.finfo(float).eps * np.linalg.norm(H, 2)
    blocks = (n - 32 + 255) // 256
    for groups in sorted({1, 2, 3, blocks - 1}):
        monkeypatch.setenv("W2K_TEST_QR_GROUPS", str(max(groups, 1)))
        _, _, ev2, z2 = _run_pencil(H, S, 1.0, 0.0, 40)
        assert np.array_equal(ev, ev2) and np.array_equal(z, z2), groups
