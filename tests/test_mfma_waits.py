"""FP64 matrix-core results are not read too early: the assembly of every kernel
of the library, compiled here as the library is, is searched for
v_mfma_f64_16x16x4 instructions that accumulate onto the MFMA just before them
and whose result another instruction (copy, store, arithmetic, or an MFMA that
takes it as a factor) touches fewer than 35 wait states later: 16 passes that it
may have had to wait for the one before, its own 16, and 3.  The compiler
leaves 19, which gave wrong sums on the device (mfma.h).

Runs on the CPU: hipcc cross-compiles."""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import subprocess
import sys

import pytest

from conftest import PKG_DIR

NEED = 35
MFMA = "v_mfma_f64_16x16x4"
_REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])")
_STORE = re.compile(r"^(global_store|flat_store|buffer_store|scratch_store|ds_write|global_atomic|ds_add)")


def _regs(text):
    out = set()
    for m in _REG.finditer(text):
        lo, hi = (m.group(2), m.group(2)) if m.group(2) else (m.group(3), m.group(4))
        out.update((m.group(1), i) for i in range(int(lo), int(hi) + 1))
    return out


def _operands(ins):
    p = ins.split(None, 1)
    return re.split(r",\s*(?![^\[]*\])", p[1]) if len(p) > 1 else []


def _functions(text):
    """[(name, instructions, {label: index})] of an assembly listing"""
    out, cur = [], None
    for line in text.splitlines():
        s = line.split(";")[0].strip()
        m = re.match(r"^([\w.$]+):$", s)
        if m and m.group(1).startswith(".L"):
            if cur:
                cur[2][m.group(1)] = len(cur[1])
        elif m:
            cur = (m.group(1), [], {})
            out.append(cur)
        elif s and not s.startswith(".") and cur:
            cur[1].append(s)
    return [f for f in out if f[1]]


def _exposed(ins, labels):
    """(MFMAs, those that accumulate onto the one just before, [(MFMA, wait
    states, reader)] of those read too early)"""

    def after(k):
        i = ins[k]
        if i.startswith(("s_endpgm", "s_setpc")):
            return []
        if i.startswith("s_branch"):
            return [labels[i.split()[1]]]
        if i.startswith("s_cbranch"):
            return [k + 1, labels[i.split()[1]]]
        return [k + 1] if k + 1 < len(ins) else []

    count, chained = 0, set()
    for k, i in enumerate(ins):
        if not i.startswith(MFMA):
            continue
        count += 1
        dst, todo, seen = _regs(_operands(i)[0]), after(k), set()
        while todo:  # every way to a next MFMA
            x = todo.pop()
            if x in seen:
                continue
            seen.add(x)
            if ins[x].startswith("v_mfma"):
                if _regs(_operands(ins[x])[3]) & dst:
                    chained.add(x)
            else:
                todo += after(x)
    bad = []
    for x in sorted(chained):
        dst = _regs(_operands(ins[x])[0])
        todo, seen = [(y, 0) for y in after(x)], {}
        while todo:
            y, w = todo.pop()
            if w >= NEED or seen.get(y, NEED) <= w:
                continue
            seen[y] = w
            j, ops = ins[y], _operands(ins[y])
            if j.startswith("v_mfma"):
                # it waits for this one itself if it accumulates, and follows it in any case
                if _regs(ops[1] + " " + ops[2]) & dst:
                    bad.append((ins[x], w, j))
            elif _regs(" ".join(ops)) & dst:
                bad.append((ins[x], w, j))
            else:
                step = int(ops[0], 0) + 1 if j.startswith("s_nop") else 1
                todo += [(z, w + step) for z in after(y)]
    return count, len(chained), bad


def test_the_search_itself():
    chain = ["v_mfma_f64_16x16x4_f64 a[0:7], v[0:1], v[2:3], 0",
             "v_mfma_f64_16x16x4_f64 a[0:7], v[4:5], v[6:7], a[0:7]"]
    read = ["v_accvgpr_read_b32 v9, a1", "s_endpgm"]
    assert _exposed(chain + ["s_nop 15", "s_nop 2"] + read, {})[2] == [(chain[1], 19, read[0])]
    assert _exposed(chain + ["s_nop 15", "s_nop 15", "s_nop 2"] + read, {})[2] == []
    other = "v_mfma_f64_16x16x4_f64 a[8:15], v[4:5], v[6:7], 0"
    assert _exposed([chain[0], other, chain[1], "s_nop 15", "s_nop 2"] + read, {}) == (3, 0, [])
    # round a loop
    loop = [chain[0], chain[1], "s_cbranch_scc1 .L0", "s_endpgm", "s_nop 15", "ds_write_b64 v1, a[6:7]", "s_endpgm"]
    assert _exposed(loop, {".L0": 4})[2] == [(chain[1], 17, loop[5])]


def test_no_result_is_read_too_early(tmp_path):
    sys.path.insert(0, PKG_DIR)
    import build as hipbuild  # hack-wein2k_amd/build.py
    sys.path.pop(0)
    if not os.path.exists(hipbuild.HIPCC):
        pytest.skip("no hipcc")

    def listing(src):
        out = str(tmp_path / (os.path.basename(src) + ".s"))
        subprocess.run([hipbuild.HIPCC, *hipbuild.CXXFLAGS, "-S", "--cuda-device-only", src, "-o", out], check=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        with open(out) as f:
            return f.read()

    with cf.ThreadPoolExecutor(max_workers=8) as ex:
        texts = list(ex.map(listing, hipbuild.sources()))
    total, bad = 0, []
    for text in texts:
        for name, ins, labels in _functions(text):
            count, _, b = _exposed(ins, labels)
            total += count
            bad += [(name,) + x for x in b]
    assert total > 1000
    assert not bad, bad[:10]
