"""The library's kernels on the CPU (tests/cpuemu) with the waves of a
work-group far apart: each wave runs to its next barrier before the next one
starts, in either order (W2K_EMU_WAVES).  A schedule is one that the device
may take, so that results must not depend on it; LDS that one wave reads and
another overwrites with no barrier between gives wrong numbers here every time,
where on the device the waves' usual pace hides it.

The child solves generalised eigenproblems with S far from the identity
(Cholesky blocks and their inverses, the two-stage tridiagonalisation, the
cluster orthogonalisation's Gram blocks) and runs k-points of both builds.

Tolerances: as test_gpu_chol_leaf (64 n eps relative, kappa(S) below 8) and
1e-10 Ry against the reference."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from test_cpuemu import HERE, emu_lib  # noqa: F401  (fixture)

CHILD = r"""
import sys
import numpy as np
import scipy.linalg as sla
sys.path.insert(0, {tests!r})
from conftest import Fixture, PKG
L = PKG.lapw1
L._LIB = L.load_library(path={lib!r})
from test_gpu_seclr4 import _run_pencil

bad = 0
for n, cplx in [(16, 0), (17, 1), (64, 0), (64, 1), (80, 1), (129, 0)]:
    rng = np.random.default_rng(11 * n + cplx)
    def hermitian():
        a = rng.standard_normal((n, n)) + (1j * rng.standard_normal((n, n)) if cplx else 0.0)
        return (a + a.conj().T) / 2
    E = hermitian()
    H = np.diag(np.repeat(np.arange(n), 4)[:n] + 0.0) if n == 64 else hermitian()  # clusters of four
    d = rng.uniform(1.0, 2.0, n)
    S = np.eye(n) + E / (4 * np.linalg.norm(E, 2))
    S = (d[:, None] * S * d[None, :]).astype(E.dtype)
    if n == 64:
        C = np.linalg.cholesky(S)
        H = C @ H @ C.conj().T
        H = (H + H.conj().T) / 2
    ref = sla.eigh(H, S, eigvals_only=True)
    ne, nb, ev, z = _run_pencil(H, S, ref[-1] + 1.0, ref[0] - 1.0, n)
    tol = 64 * n * np.finfo(float).eps
    de = float(np.max(np.abs(ev - ref)) / np.max(np.abs(ref))) if ne == n else -1.0
    do = float(np.max(np.abs(z.conj().T @ S @ z - np.eye(n)))) if ne == n else -1.0
    print(n, cplx, ne, de, do, flush=True)
    if not (ne == n and de <= tol and do <= 1e-10):
        bad += 1
for name in ["c1_fcc", "lo_cplx"]:
    fx = Fixture(name)
    kd = fx.k(0)
    ctx = L.Lapw1(fx.run())
    ctx.set_basis(fx.basis(0))
    ne, nb = ctx.calkpt(float(kd["EL"]), float(kd["EU"]), int(kd["NUME"]))
    ev, z = ctx.get_eig()
    ctx.close()
    de = float(np.max(np.abs(ev - kd["EIGVAL"]))) if ne == int(kd["NE"]) else -1.0
    print(name, ne, nb, de, flush=True)
    if not (ne == int(kd["NE"]) and nb == int(kd["NBELW"]) and de < 1e-10):
        bad += 1
assert bad == 0, bad
print("CHILD OK", flush=True)
"""


@pytest.mark.parametrize("order", ["up", "down"])
def test_results_do_not_depend_on_the_waves_pace(emu_lib, order):  # noqa: F811
    code = CHILD.format(tests=HERE, lib=emu_lib)
    env = dict(os.environ, W2K_EMU_WAVES=order)
    r = subprocess.run([sys.executable, "-c", code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       timeout=900)
    out = r.stdout.decode(errors="replace")
    assert r.returncode == 0 and "CHILD OK" in out, out[-4000:]
