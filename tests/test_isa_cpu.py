"""CPU: properties of the compiled GPU code that no result shows reliably, looked
up in the compiler's assembly of the loop and sampler kernels.

A scalar load and a later vector store of one wave are not ordered with each
other.  Where a kernel may write what it reads, no scalar load other than of the
kernel's arguments may therefore be outstanding at a store.

A DPP operand must not have been written by the VALU in the last two wait states.
The compiler sees to it for its own instructions, not for those in inline asm
(row_newbcast): there an s_nop has to stand between, whatever else happens to.
"""
import os
import re
import shutil
import subprocess

import pytest

from cosmopp_amd import build as B

pytestmark = pytest.mark.skipif(shutil.which(B.HIPCC) is None, reason="no hipcc")


def assembly(source, tmp):
    out = os.path.join(str(tmp), source + ".s")
    subprocess.run([B.HIPCC] + B.HIP_FLAGS + ["--cuda-device-only", "-S", "-o", out, os.path.join(B.CSRC, source)],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return kernels(open(out).read())


def kernels(text):
    """{name: (instructions, successors)} of the functions of an assembly file."""
    found = {}
    for m in re.finditer(r"^(_Z\S+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.S | re.M):
        ins, labels = [], {}
        for line in m.group(2).splitlines():
            s = line.split(";")[0].strip()
            lab = re.match(r"(\.LBB\S+):", s)
            if lab:
                labels[lab.group(1)] = len(ins)
            elif s and not s.startswith("."):
                ins.append(s)
        succ = []
        for i, s in enumerate(ins):
            to = re.match(r"s_c?branch\w*\s+(\S+)", s)
            n = [labels[to.group(1)]] if to else []
            if not s.startswith(("s_branch", "s_endpgm", "s_setpc")) and i + 1 < len(ins):
                n.append(i + 1)
            succ.append(n)
        found[m.group(1)] = (ins, succ)
    return found


def registers(op):
    m = re.match(r"([sv])\[(\d+):(\d+)\]$", op)
    if m:
        return {(m.group(1), i) for i in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.match(r"([sv])(\d+)$", op)
    return {(m.group(1), int(m.group(2)))} if m else set()


def loads_at_stores(ins, succ):
    """(scalar load, store) pairs with the load outstanding at the store, loads of kernel arguments
    (through the pointer the kernel starts with, until it is overwritten) left out."""
    first = next((re.match(r"s_load_\w+\s+\S+,\s*(\S+),", s) for s in ins if s.startswith("s_load")), None)
    if first is None:
        return []
    args, until = registers(first.group(1)), len(ins)
    for i, s in enumerate(ins):
        a = s.split(None, 1)
        if len(a) == 2 and s.startswith("s_") and not s.startswith(("s_waitcnt", "s_cmp", "s_cbranch")) \
                and registers(a[1].split(",")[0].strip()) & args:
            until = i
            break
    state, work, bad = {0: frozenset()}, [0], set()
    while work:
        i = work.pop()
        s, out = ins[i], set(state[i])
        m = re.match(r"s_load_\w+\s+\S+,\s*(\S+),", s)
        if m and not (i <= until and registers(m.group(1)) == args):
            out.add(i)
        if s.startswith("s_waitcnt") and (re.search(r"lgkmcnt\(0\)", s) or "cnt(" not in s):
            out.clear()
        if re.match(r"(global|flat|buffer)_(store|atomic)", s):
            bad |= {(ins[k], s) for k in out}
        for j in succ[i]:
            new = state.get(j, frozenset()) | out
            if j not in state or new != state[j]:
                state[j] = new
                work.append(j)
    return sorted(bad)


def test_the_check_itself():
    text = ("_Zk: ; @k\n s_load_dwordx2 s[2:3], s[0:1], 0x0\n s_waitcnt lgkmcnt(0)\n s_load_dword s4, s[2:3], 0x4\n"
            "%s global_store_dword v0, v1, s[2:3] offset:4\n s_endpgm\n.Lfunc_end0:\n")
    for wait, n in (("", 1), (" s_waitcnt lgkmcnt(0)\n", 0), (" s_waitcnt lgkmcnt(1)\n", 1)):
        assert len(loads_at_stores(*kernels(text % wait)["_Zk"])) == n


@pytest.mark.parametrize("source", ["cmbl_loops.hip", "cmbl_sampler.hip"])
def test_no_scalar_load_outstanding_at_a_store(source, tmp_path):
    found = assembly(source, tmp_path)
    assert found
    bad = {k: v for k, v in ((k, loads_at_stores(*f)) for k, f in found.items()) if v}
    assert not bad, bad


def mask(regs):
    return sum(1 << i for kind, i in regs if kind == "v")


def unguarded_rows(ins, succ):
    """row_newbcast instructions whose DPP operand may come from the VALU with no s_nop of two wait states or more
    since (a bit per register written by the VALU, followed along every path)."""
    state, work, bad = {0: 0}, [0], set()
    while work:
        i = work.pop()
        s, out = ins[i], state[i]
        ops = [o.strip() for o in s.split(None, 1)[1].split(",")] if " " in s else []
        if "row_newbcast" in s and out & mask(registers(ops[1].lstrip("-").split()[0])):
            bad.add(s)
        nop = re.match(r"s_nop\s+(\d+)", s)
        if nop and int(nop.group(1)) >= 1:
            out = 0
        elif s.startswith("v_") and ops:
            out |= mask(registers(ops[0].split()[0]))
            if "swap" in s:
                out |= mask(registers(ops[1].split()[0]))
        elif s.startswith(("global_load", "ds_read", "flat_load")):
            out &= ~mask(registers(ops[0].split()[0]))
        for j in succ[i]:
            new = state.get(j, 0) | out
            if j not in state or new != state[j]:
                state[j] = new
                work.append(j)
    return sorted(bad)


def test_the_row_check_itself():
    use = " v_fmac_f64_dpp v[0:1], v[2:3], v[4:5] row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
    far = " v_mov_b64_e32 v[6:7], 0\n" * 9
    for body, n in ((" v_mov_b64_e32 v[2:3], v[8:9]\n" + far, 1), (" v_mov_b64_e32 v[2:3], v[8:9]\n s_nop 1\n", 0),
                    (" v_mov_b64_e32 v[2:3], v[8:9]\n global_load_dwordx2 v[2:3], v[8:9], off\n", 0)):
        assert len(unguarded_rows(*kernels("_Zk: ; @k\n" + body + use + " s_endpgm\n.Lfunc_end0:\n")["_Zk"])) == n


def test_row_coefficients_are_guarded(tmp_path):
    found = assembly("cmbl_kernels.hip", tmp_path)
    rows = sum("row_newbcast" in s for ins, _ in found.values() for s in ins)
    bad = {k: v for k, v in ((k, unguarded_rows(*f)) for k, f in found.items()) if v}
    assert rows > 1000 and not bad, {k: (len(v), v[:2]) for k, v in bad.items()}
