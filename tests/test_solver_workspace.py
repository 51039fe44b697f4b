"""Device memory that SECLR4 takes: beside four matrices of order n, the
eigenvectors, the inverse iteration's factors (five planes of n x m and the
pivots) and what grows with n alone, not more than a fixed amount at any order.

The number is the library's own (the workspace that w2k_seclr4_noalloc says an
order beyond its limit would need), asked of the CPU build; no solve runs.
What grows with n alone (panels, band, sums) is below 3000 elements a row, the
fixed pieces (split-K partial products, operands of Q2) below 1.25 GiB."""
from __future__ import annotations

import os
import subprocess
import sys

import pytest

from test_cpuemu import HERE, emu_lib  # noqa: F401  (fixture)

CHILD = r"""
import ctypes, re, sys
import numpy as np
sys.path.insert(0, {tests!r})
from conftest import Fixture, PKG
L = PKG.lapw1
L._LIB = L.load_library(path={lib!r})
for name, z in [("c1_fcc", 1), ("lo_cplx", 2)]:
    ctx = L.Lapw1(Fixture(name).run())
    f = ctx.lib.w2k_seclr4_noalloc
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_double, ctypes.c_double,
                  ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    one = np.zeros(1)
    i1, i2 = ctypes.c_int(0), ctypes.c_int(0)
    for n, m in [(769, 769), (2000, 200), (5951, 1190), (12447, 1200), (40000, 4000), (46000, 10)]:
        rc = f(ctx.ctx, n, one.ctypes.data, one.ctypes.data, 1.0, 0.0, m, ctypes.addressof(i1), ctypes.addressof(i2),
               one.ctypes.data, one.ctypes.data, n)
        text = ctx.lib.w2k_last_error().decode()
        need, scratch = map(int, re.search(r"needs (\d+) bytes .* holds (\d+) bytes", text).groups())
        print(name, n, m, need, scratch, flush=True)
        assert rc == -1 and scratch == 128 << 20, text
        least = 8 * (z * (4 * n * n + n * m) + 5.5 * (n + 2) * m)
        assert need <= least + 8 * z * 3000 * n + 1.25 * 2**30, (n, m, need / least)
    ctx.close()
print("CHILD OK", flush=True)
"""


def test_no_more_than_the_matrices_and_a_fixed_amount(emu_lib):  # noqa: F811
    r = subprocess.run([sys.executable, "-c", CHILD.format(tests=HERE, lib=emu_lib)], env=dict(os.environ),
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=600)
    out = r.stdout.decode(errors="replace")
    assert r.returncode == 0 and "CHILD OK" in out, out[-4000:]
