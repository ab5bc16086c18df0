"""The built gfx950 code keeps the wait states that its inline-asm loads leave to the programmer.

A VALU instruction that writes a scalar register must be five wait states ahead of a vector-memory
instruction that reads it (an instruction counts one, s_nop n counts n + 1).  The compiler pads its own
loads; it does not look into inline asm, so a load there could read a stale base.  The scan walks back
from every vector-memory instruction of the library, along every path of the control flow.
"""
import collections
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
SREG = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\b(vcc)\b")
VMEM = ("global_", "buffer_", "flat_", "scratch_")
STATES = 5


def sregs(text):
    out = set()
    for lo, hi, one, name in SREG.findall(text):
        out |= set(range(int(lo), int(hi) + 1)) if lo else {int(one)} if one else {name}
    return out


def valu_sgpr_writes(op, args):
    """Scalar registers that a vector instruction writes: its destination, or the carry / scale flag."""
    if not op.startswith("v_") or op.startswith("v_cmpx"):
        return set()
    ops = args.split(",")
    written = sregs(ops[0])
    if ("_co_" in op or op.startswith("v_div_scale")) and len(ops) > 1:
        written |= sregs(ops[1])
    return written


def violations(ins):
    """(address, load, writer) of every load that may read a scalar register too soon; ins: (op, args, address)."""
    index = {a: i for i, (_, _, a) in enumerate(ins)}
    preds = collections.defaultdict(list)
    for i, (op, args, a) in enumerate(ins):
        if i + 1 < len(ins) and not op.startswith(("s_branch", "s_endpgm", "s_setpc")):
            preds[i + 1].append(i)
        if op.startswith(("s_branch", "s_cbranch")):
            off = int(args.split()[0])
            target = a + 4 + 4 * (off - 65536 if off > 32767 else off)
            assert target in index, (op, args, hex(a))
            preds[index[target]].append(i)
    bad = []
    for i, (op, args, a) in enumerate(ins):
        read = sregs(args) if op.startswith(VMEM) else None
        if not read:
            continue
        todo, seen = [(p, 0) for p in preds[i]], set()
        while todo:
            p, states = todo.pop()
            if states >= STATES or (p, states) in seen:
                continue
            seen.add((p, states))
            o, r, _ = ins[p]
            if valu_sgpr_writes(o, r) & read:
                bad.append((hex(a), f"{op} {args}", f"{o} {r}"))
            else:
                n = int(r.split()[0], 0) + 1 if o == "s_nop" else 1
                todo += [(q, states + n) for q in preds[p]]
    return bad


def functions(lib, tmp):
    shutil.copy(lib, tmp / "l.so")
    subprocess.run([OBJDUMP, "--offloading", "l.so"], cwd=tmp, check=True, capture_output=True)
    for obj in sorted(tmp.glob("l.so.*gfx950*")):
        text = subprocess.run([OBJDUMP, "-d", str(obj)], check=True, capture_output=True, text=True).stdout
        name, ins = None, []
        for line in text.splitlines():
            if m := re.match(r"^[0-9a-f]+ <(.*)>:$", line):
                if ins:
                    yield name, ins
                name, ins = m.group(1), []
            elif m := re.match(r"^\t(\S+)\s*(.*?)\s*// ([0-9A-F]+):", line):
                ins.append((m.group(1), m.group(2), int(m.group(3), 16)))
        if ins:
            yield name, ins


def listing(*lines):
    return [(line.split(" ", 1) + [""])[:2] + [4 * i] for i, line in enumerate(lines)]


@pytest.mark.parametrize("between,ok", [
    (["s_add_u32 m0, s1, 0", "s_nop 0"], False),
    (["s_add_u32 m0, s1, 0", "s_nop 2"], False),
    (["s_add_u32 m0, s1, 0", "s_nop 3"], True),
    (["s_nop 4"], True),
])
@pytest.mark.parametrize("writer", ["v_readfirstlane_b32 s40, v1", "v_cmp_eq_u32_e64 s[40:41], v1, v2",
                                    "v_add_co_u32_e64 v1, s[40:41], v2, v3"])
def test_the_scan_sees_a_planted_hazard(writer, between, ok):
    load = "global_load_lds_dwordx4 v3, s[40:41]"
    assert (violations(listing(writer, *between, load, "s_endpgm")) == []) == ok
    # the same across a loop's back edge: the writer after the load, 5 wait states less the branch ahead of it
    tail = [load, "s_nop 7", writer, "s_cbranch_scc1 %d" % (65536 - 4 - len(between)), "s_endpgm"]
    assert (violations(listing(*between, *tail)) == []) == (ok or between[-1] == "s_nop 2")


@pytest.mark.skipif(not shutil.which(OBJDUMP), reason="needs the ROCm llvm-objdump")
def test_no_load_reads_a_scalar_register_too_soon(tmp_path):
    from estudiocanciones_amd import _ffi
    from estudiocanciones_amd.build import LIBDIR, LIBNAME
    _ffi.lib()
    n, bad = 0, []
    for name, ins in functions(LIBDIR / LIBNAME, tmp_path):
        n += sum(op.startswith("global_load_lds") for op, _, _ in ins)
        bad += [(name, *v) for v in violations(ins)]
    assert n > 0, "no LDS DMA found: the scan did not see the library's code"
    assert not bad, f"{len(bad)} loads, first {bad[:3]}"
