"""The calls that a user of the library makes, over the range of cells it is used on.

A case is one of
  kpoint   one k-point of an SCF iteration: the basis handed over, HAMILT, HNS and SECLR4 on the device, the
           eigenvalues fetched, and the interstitial band density that lapw2 forms from the vectors;
  coors    the same with the basis generated on the device (COORS and LOPW) instead of handed over;
  adjoint  a k-point with its band-energy gradients (interstitial box, non-spherical integrals);
  bands    a band-structure run: a list of k-points in one batched call, eigenvalues only;
  solve    SECLR4 alone on host matrices, as the Fortran drop-in calls it;
  matrix   HAMILT and HNS alone, for a caller that keeps its own eigensolver: HS and HSDIAG on the device;
  atpar    the radial functions and non-spherical integrals of one SCF iteration.

The cells are the ones of tests/golden (one to a hundred atoms, real and complex, with and without local orbitals) at
plane-wave cut-offs from well below to somewhat above their own; the seed makes another potential on the same cell, as
the iterations of an SCF run do.  SECLR4's vectors are determined up to a phase, or a rotation among equal
eigenvalues, and close ones are ill-conditioned one by one, so what is returned of them is what lapw2 and the gradients
make of all of them, with occupations that are smooth in the energy: the whole density or gradient, which every vector
enters and which has one value.
"""
from __future__ import annotations

import ctypes
import functools
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(maxsize=None)
def _lapw1():
    name = "hack_wein2k_amd"
    if name not in sys.modules:
        pkg = os.path.join(ROOT, "hack-wein2k_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(pkg, "__init__.py"),
                                                      submodule_search_locations=[pkg])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name].lapw1


@functools.lru_cache(maxsize=None)
def _cell(name):
    """(run arrays, complex build?) of a cell of tests/golden."""
    with np.load(os.path.join(ROOT, "tests", "golden", name + ".npz"), allow_pickle=False) as z:
        return {k[4:]: z[k] for k in z.files if k.startswith("run/")}, bool(int(z["meta/complex"]))


def listed():
    return [
        # a one-atom metal at the smallest basis, basis generation included: latency and launches
        dict(name="coors fcc", kind="coors", cell="c1_fcc", rkm=1.0, sx=0.21, sy=0.09, sz=0.37, frac=0.4, split=0),
        # a two-atom oxide with local orbitals, the size of the program's own example
        dict(name="kpoint mgo", kind="kpoint", cell="mgo", rkm=1.0, sx=0.25, sy=0.25, sz=0.0, frac=0.2, split=0),
        # three atoms without inversion (complex matrices), local orbitals, a general k-point
        dict(name="kpoint 3 atoms complex", kind="kpoint", cell="lo_cplx", rkm=1.0, sx=0.13, sy=0.22, sz=0.41, frac=0.2,
             split=0),
        # the drop-in's eigensolve of a host matrix, odd order
        dict(name="solve real 731", kind="solve", n=731, complex=False, frac=0.12),
        # a band-structure path of an eight-atom cell at a modest cut-off
        dict(name="bands ortho8 16 k", kind="bands", cell="c4_ortho8", rkm=0.7, nk=16, sx=0.0, sy=0.0, sz=0.0, ex=0.5,
             ey=0.5, ez=0.5, frac=0.15, split=0),
        # an ordinary cell: eight atoms, complex, one general k-point
        dict(name="kpoint ortho8", kind="kpoint", cell="c4_ortho8", rkm=1.0, sx=0.31, sy=0.12, sz=0.27, frac=0.1,
             split=0),
        # gradients of the band energy of a sixteen-atom cell (real, N about 3000)
        dict(name="adjoint cubic16", kind="adjoint", cell="c5_cubic16", rkm=1.0, sx=0.25, sy=0.75, sz=0.25,
             frac=0.05, split=0),
        # assembly only, a hundred atoms
        dict(name="matrix lowsym100", kind="matrix", cell="c3_lowsym100", rkm=0.66, sx=0.12, sy=0.37, sz=0.25,
             split=0),
        # the 64-atom supercell at Gamma (real, high symmetry, many equal eigenvalues)
        dict(name="kpoint rs64", kind="kpoint", cell="c2_rs64", rkm=1.0, sx=0.0, sy=0.0, sz=0.0, frac=0.2,
             split=0),
        # a hundred atoms, complex, HNS in split precision
        dict(name="kpoint lowsym100 mid", kind="kpoint", cell="c3_lowsym100", rkm=0.8, sx=0.12, sy=0.37, sz=0.25,
             frac=0.2, split=4),
        # the largest: a hundred atoms, complex, every product in 64 bits
        dict(name="kpoint lowsym100 large", kind="kpoint", cell="c3_lowsym100", rkm=0.955, sx=0.12, sy=0.37, sz=0.25,
             frac=0.2, split=0),
        # radial functions and integrals of the 64 atoms of the supercell
        dict(name="atpar rs64", kind="atpar", cell="c2_rs64"),
    ]


# cut-offs per cell, relative to the cell's own, that draw() spreads over
_RANGE = {"c1_fcc": (0.9, 1.6), "mgo": (0.75, 1.25), "lo_cplx": (0.8, 1.4), "rs8": (0.8, 1.5), "c4_ortho8": (0.5, 1.1),
          "c5_cubic16": (0.5, 1.1), "c2_rs64": (0.45, 1.0), "c3_lowsym100": (0.6, 0.9)}


def draw(rng):
    kind = rng.choice(["kpoint", "kpoint", "kpoint", "coors", "adjoint", "bands", "solve", "matrix", "atpar"])
    if kind == "solve":
        return dict(kind=kind, n=int(round(math.exp(rng.uniform(math.log(40), math.log(1100))))),
                    complex=rng.random() < 0.5, frac=round(rng.uniform(0.05, 0.3), 3))
    if kind == "atpar":
        return dict(kind=kind, cell=rng.choice(["c1_fcc", "lo_cplx", "rs8", "c4_ortho8", "c5_cubic16", "c2_rs64"]),
                    tilt=round(rng.uniform(-0.01, 0.01), 5))
    cells = {"kpoint": list(_RANGE), "matrix": list(_RANGE), "bands": ["c1_fcc", "mgo", "lo_cplx", "rs8", "c4_ortho8"],
             "coors": ["c1_fcc", "mgo", "lo_cplx", "rs8", "c4_ortho8"],
             "adjoint": ["c1_fcc", "lo_cplx", "rs8", "c4_ortho8", "c5_cubic16"]}[kind]
    cell = rng.choice(cells)
    lo, hi = _RANGE[cell]
    c = dict(kind=kind, cell=cell, rkm=round(math.exp(rng.uniform(math.log(lo), math.log(hi))), 4))
    for a in ("sx", "sy", "sz"):
        c[a] = round(rng.uniform(-0.5, 0.5), 4)
    if kind == "bands":
        c.update(nk=rng.randint(2, 24), ex=round(rng.uniform(-0.5, 0.5), 4), ey=round(rng.uniform(-0.5, 0.5), 4),
                 ez=round(rng.uniform(-0.5, 0.5), 4))
    if kind != "matrix":
        c["frac"] = round(rng.uniform(0.05, 0.25), 3)
    c["split"] = rng.choice([0, 0, 0, 4, 5])
    return c


# ------------------------------------------------------------------ inputs
def _run_arrays(cell, rng):
    """The cell's run with a potential of this seed: the warped box and the non-spherical integrals scaled by a per cent
    or two, as from one SCF iteration to the next."""
    d, cplx = _cell(cell)
    d = dict(d)
    d["WARP"] = np.asarray(d["WARP"]) * (1.0 + 0.02 * rng.standard_normal())
    for k in ("VNS1", "VNS2", "VNS3", "VNS1LO", "VNS2LO", "VNS3LO"):
        d[k] = np.asarray(d[k]) * (1.0 + 0.02 * rng.standard_normal())
    return d, cplx


def _lattice(d, rkm):
    return _lapw1().Lattice.make(d["BR2"], d["PIA"], int(d["ORTHO"]), int(d["CXZ"]), float(d["RKM"]) * rkm)


def _sphere(n):
    """The n shortest vectors of the simple cubic lattice (ties in a fixed order)."""
    m = 2
    while (4.0 / 3.0) * math.pi * m ** 3 < 1.5 * n + 60:
        m += 1
    g = np.array([(x, y, z) for x in range(-m, m + 1) for y in range(-m, m + 1) for z in range(-m, m + 1)])
    return g[np.lexsort((g[:, 2], g[:, 1], g[:, 0], np.sum(g * g, axis=1)))][:n]


def _pencil(case, seed):
    """H and S (whole matrices) of a plane-wave kind: H = L (k^2 + V) L^H with a potential that falls off away from
    the diagonal, S = L L^H with overlaps of a few tenths."""
    rng = np.random.default_rng([seed, 7])
    n, cplx = case["n"], case["complex"]

    def noise():
        a = rng.standard_normal((n, n))
        return a + 1j * rng.standard_normal((n, n)) if cplx else a

    g = _sphere(n)
    k2 = 9.0 * np.sum(g * g, axis=1) / max(1, int(np.max(np.sum(g * g, axis=1))))
    i = np.arange(n)
    v = 0.4 * noise() / (1.0 + np.abs(i[:, None] - i[None, :]) / 4.0)
    h0 = np.diag(k2) + 0.5 * (v + v.conj().T)
    low = np.eye(n) + np.tril(0.5 / math.sqrt(n) * noise(), -1)
    h, s = low @ h0 @ low.conj().T, low @ low.conj().T
    return 0.5 * (h + h.conj().T), 0.5 * (s + s.conj().T), g


def _box(g):
    return int(np.max(np.abs(g))) + 1


def _count(case):
    return max(4, int(round(case["frac"] * case["n"])))


def prepare(case, seed):
    L = _lapw1()
    rng = np.random.default_rng([seed, 3])
    kind = case["kind"]
    st = {"case": case}
    if kind == "solve":
        h, s, g = _pencil(case, seed)
        n, w = case["n"], _box(g)
        d, _ = _cell("c1_fcc")  # the run that the context needs; HAMILT is not called
        d = dict(d, WARP1=w, WARP2=w, WARP3=w, WARP=np.zeros((2 * w + 1,) * 3, np.complex128))
        st["ctx"] = L.Lapw1(L.RunData(d, case["complex"]))
        length = np.sqrt(np.sum(g * g, axis=1).astype(np.float64))
        st["ctx"].set_basis(L.Basis(n, 0, g.T, g[:, 0], g[:, 1], g[:, 2], length))
        # S above the diagonal, H below it (conjugated), diag(S) apart
        st["hs"] = np.asfortranarray(np.triu(s, 1) + np.tril(h.conj(), -1) + np.diag(np.diag(h)))
        st["hsdiag"] = np.ascontiguousarray(np.diag(s))
        st["nume"] = _count(case)
        return st
    if kind == "atpar":
        d, cplx = _cell(case["cell"])
        st["ctx"] = L.Lapw1(L.RunData(d, cplx))
        scale = 1.0 + case.get("tilt", 0.0) + 0.01 * rng.standard_normal()
        st["args"] = [int(d["REL"]), np.atleast_1d(d["JRJ"]), np.atleast_1d(d["RO"]), np.atleast_1d(d["DH"]),
                      *_charges(d, scale)]
        return st
    d, cplx = _run_arrays(case["cell"], rng)
    st["ctx"] = ctx = L.Lapw1(L.RunData(d, cplx))
    if case["split"]:
        ctx.set_split_precision(case["split"])
    lat = _lattice(d, case["rkm"])
    if kind == "bands":
        t = np.linspace(0.0, 1.0, case["nk"])
        st["bases"] = [ctx.coors(lat, *(case[s] + x * (case[e] - case[s]) for s, e in
                                        (("sx", "ex"), ("sy", "ey"), ("sz", "ez")))) for x in t]
        st["nume"] = max(4, int(case["frac"] * min(b.n for b in st["bases"])))
        return st
    st["lat"] = lat
    st["basis"] = ctx.coors(lat, case["sx"], case["sy"], case["sz"])
    if kind != "matrix":
        st["nume"] = max(4, int(case["frac"] * st["basis"].n))
    return st


def _charges(d, scale):
    """Nuclear charges, r V00(r) and V_LM(r) of the cell, the electrons' part of the potential scaled."""
    vr = np.asarray(d["VR"], np.float64)
    vr = vr.reshape(vr.shape[0], -1, order="F")
    z = np.round(np.abs(vr[0])) if np.max(np.abs(vr[0])) >= 1.0 else np.ones(vr.shape[1])
    vlm = np.asarray(d["VLM"], np.float64)
    vlm = vlm.reshape(vlm.shape[0], vlm.shape[1], -1, order="F")
    return z, np.asfortranarray(-z + scale * (vr + z)), np.asfortranarray(scale * vlm)


# ------------------------------------------------------------------ passes
# the window holds everything: the number of eigenpairs is set by NUME
_EL, _EU = -50.0, 1.0e4


def _levels(ctx):
    """EIGVAL of the last k-point, without the vectors."""
    ev = np.zeros(ctx.ne)
    ctx._chk("w2k_get_eig", ctx.lib.w2k_get_eig(ctx.ctx, ev.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), None,
                                                ctx.basis.n))
    return ev


def _occupations(ev):
    """Fermi function around the middle of the window, zero to rounding at its top."""
    mu = ev[len(ev) // 2]
    x = (ev - mu) / max((ev[-1] - mu) / 36.0, 1e-3)
    return 1.0 / (1.0 + np.exp(np.minimum(x, 500.0)))


class _OnDevice:
    """Doubles of the context's own memory, for torch, which keeps this object and so the context alive."""

    def __init__(self, ctx, ptr, shape):
        self.ctx = ctx
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f8", "version": 3}


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "atpar":
        return ctx.atpar(*state["args"])
    if kind == "bands":
        got = ctx.calkpt_batched(state["bases"], _EL, _EU, state["nume"], vectors=False)
        return {"levels": np.stack([ev for _, _, ev, _ in got])}
    if kind == "solve":
        ctx.put_hs(state["hs"], state["hsdiag"])
        ctx.seclr4(_EL, _EU, state["nume"])
        ev = _levels(ctx)
        return {"levels": ev, "density": ctx.density_interstitial(_occupations(ev))}
    if kind == "coors":
        ctx.coors(state["lat"], case["sx"], case["sy"], case["sz"])
    else:
        ctx.set_basis(state["basis"])
    if kind == "matrix":
        ctx.hamilt()
        ctx.swap_diag()
        ctx.hns()
        hs, hd = ctypes.c_void_p(), ctypes.c_void_p()
        ctx._chk("w2k_device_buffers", ctx.lib.w2k_device_buffers(ctx.ctx, ctypes.byref(hs), ctypes.byref(hd), None,
                                                                  None))
        ctx.sync()
        n, w = state["basis"].n, 2 if ctx.run.is_complex else 1
        return {"hs": torch.as_tensor(_OnDevice(ctx, hs.value, (n, n * w)), device="cuda"),
                "hsdiag": torch.as_tensor(_OnDevice(ctx, hd.value, (n * w,)), device="cuda")}
    ctx.calkpt(_EL, _EU, state["nume"])
    ev = _levels(ctx)
    f = _occupations(ev)
    if kind == "adjoint":
        energy, warp = ctx.adjoint_warp(f)
        return {"levels": ev, "energy": energy, "warp": warp, **ctx.adjoint_vns(f)}
    return {"levels": ev, "density": ctx.density_interstitial(f)}


# ------------------------------------------------------------------ what a pass cannot do without
def _order(case):
    """(plane waves, local orbitals) of the case's basis, from the volume of its sphere."""
    d, _ = _cell(case["cell"])
    return int((float(d["RKM"]) * case["rkm"]) ** 3 / (6.0 * math.pi ** 2 * float(d["VI"]))), int(d["NLO"])


def work(case):
    kind = case["kind"]
    if kind == "solve":
        n, z = case["n"], 4 if case["complex"] else 1
        m = _count(case)
        flops = z * (2.0 * n ** 3 / 3 + 2.0 * n ** 3 + 4.0 * n ** 3 / 3 + 4.0 * n * n * m)
        return {"bytes": 8.0 * (2 if case["complex"] else 1) * (n * n + n * m), "flops": flops}
    d, cplx = _cell(case["cell"])
    nat, lt = int(d["NDF"]), int(d["LTOP"])
    if kind == "atpar":
        jrid, lm = np.shape(d["VLM"])[:2]
        types = int(d["NAT"])
        return {"bytes": 8.0 * types * jrid * (1 + lm), "flops": types * jrid * (lt * 3 * 40.0 + lm * 25 * 9 * 4.0)}
    nv, nlo = _order(case)
    n = nv + nlo
    z, w = (4, 2) if cplx else (1, 1)
    # HAMILT: the l-sum of two Legendre products per atom and pair; HNS: rank 4 sum(LINDEX) update of a triangle
    lsum = 25 * nat
    flops = 4.0 * nv * nv * nat * lt + z * 4.0 * n * n * lsum
    nbytes = 8.0 * w * n * n
    if kind == "matrix":
        return {"bytes": nbytes, "flops": flops}
    m = max(4, int(case["frac"] * n))
    flops += z * (2.0 * n ** 3 / 3 + 2.0 * n ** 3 + 4.0 * n ** 3 / 3 + 4.0 * n * n * m)
    nbytes += 8.0 * w * n * m
    if kind == "bands":
        return {"bytes": 8.0 * case["nk"] * (4 * n + m), "flops": case["nk"] * flops}
    flops += z * 1.0 * nv * nv * m
    if kind == "adjoint":
        flops += z * 4.0 * n * n * 25 * nat / 2
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------ plain numpy in 64 bits
def exact(case, seed):
    """SECLR4's levels and density from numpy's own Cholesky and eigensolver.  The other kinds have no such value here:
    their matrices are HAMILT's and HNS's own result."""
    if case["kind"] != "solve":
        return None
    h, s, g = _pencil(case, seed)
    low = np.linalg.cholesky(s)
    c = np.linalg.solve(low, np.linalg.solve(low, h).conj().T)
    ev, y = np.linalg.eigh(0.5 * (c + c.conj().T))
    m, w = _count(case), _box(g)
    z = np.linalg.solve(low.conj().T, y[:, :m])
    ev = ev[:m]
    gamma = (z.conj() * _occupations(ev)) @ z.T  # gamma(I, J) = sum f conj z_I z_J
    q = g[None, :, :] - g[:, None, :]
    inside = np.all(np.abs(q) <= w, axis=2)
    at = tuple((q[inside] + w).T)
    rho = np.zeros((2 * w + 1,) * 3, np.complex128)
    np.add.at(rho, at, gamma[inside])
    return {"levels": ev, "density": np.asfortranarray(rho)}
