"""Two rules checked in the library's own machine code.

Wait states that gfx9 leaves to the program: the compiler inserts them between instructions it emits,
but does not look into inline assembly, and the LDS-DMA loads are inline assembly:

* a scalar write of M0, then an LDS-DMA load, which reads M0: 1 wait state;
* a VALU write of an SGPR (v_readlane of a spilled register, v_readfirstlane), then a vector memory
  instruction that reads it as its base address: 5 wait states.

Without them the load may use the register's previous value: a DMA into another LDS slot, or from a
stale address.

No register reloaded from scratch at the end of a divergent region before exec is restored: the
reload then misses the lanes that left the region early, which keep what the region put there. The
compiler once did that to the router of 8-token blocks (hidden sizes up to 1024): with top-k above 4 it
read its logits at an LDS address that was a left-over activation, and the run ended in a fault."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "silentotithrandousha_amd", "libmxfp4moe.so")
OBJDUMP = shutil.which("llvm-objdump", path=os.pathsep.join(["/opt/rocm/llvm/bin", os.environ.get("PATH", "")]))
SGPRS = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\bvcc(?:_lo|_hi)?\b|\bm0\b")


def sgprs(text):
    out = set()
    for m in SGPRS.finditer(text):
        if m[1]:
            out.update(range(int(m[1]), int(m[2]) + 1))
        elif m[3]:
            out.add(int(m[3]))
        else:
            out.add(m[0][:3].rstrip("_"))
    return out


def violations(lines):
    """(kernel, instruction, what) of each instruction of the disassembly that comes too early."""
    bad, kernel, pos, valu, m0 = [], "", 0, {}, -9
    for line in lines:
        if line.endswith(">:\n"):
            kernel, valu, m0 = line.split("<")[1][:-3], {}, -9
            continue
        ins = line.split("//")[0].strip()
        if not ins or not line.startswith("\t"):
            continue
        op, _, rest = ins.partition(" ")
        if op == "s_nop":
            pos += int(rest, 0) + 1
            continue
        pos += 1
        dst, _, src = rest.partition(",")
        if op.startswith(("global_", "buffer_", "flat_", "scratch_")):
            if "_lds_" in op and pos - m0 <= 1:
                bad.append((kernel, ins, "M0"))
            early = [r for r in sgprs(rest) if pos - valu.get(r, -9) <= 5]
            if early:
                bad.append((kernel, ins, early))
        elif op.startswith("v_"):
            for r in sgprs(dst) | (sgprs(src.partition(",")[0]) if "_co_" in op else set()):
                valu[r] = pos
        elif op.startswith("s_"):
            written = sgprs(dst)
            for r in written:
                valu.pop(r, None)
            if "m0" in written:
                m0 = pos
    return bad


def reloads_before_exec(lines):
    """(kernel, instruction) of each scratch reload that a restore of exec follows, with no other
    change of exec and no branch between them."""
    bad, kernel, held = [], "", []
    for line in lines:
        if line.endswith(">:\n"):
            kernel, held = line.split("<")[1][:-3], []
            continue
        ins = line.split("//")[0].strip()
        if not ins or not line.startswith("\t"):
            continue
        if ins.startswith("scratch_load"):
            held.append((kernel, ins))
        elif ins.startswith("s_or_b64 exec, exec"):
            bad += held
            held = []
        elif ins.startswith(("s_cbranch", "s_branch", "s_endpgm")) or "saveexec" in ins or " exec, " in ins:
            held = []
    return bad


def test_scan_finds_reloads():
    load, restore = "\tscratch_load_dwordx2 v[58:59], off, off // 0\n", "\ts_or_b64 exec, exec, s[20:21] // 8\n"
    assert reloads_before_exec(["0 <k>:\n", load, restore]) == [("k", load.split("//")[0].strip())]
    assert reloads_before_exec(["0 <k>:\n", restore, load]) == []
    assert reloads_before_exec(["0 <k>:\n", load, "\ts_and_saveexec_b64 s[2:3], vcc // 4\n", restore]) == []


def test_scan_finds_early_reads():
    code = ["0 <k>:\n", "\tv_readlane_b32 s9, v1, 2 // 0\n", "\ts_mov_b32 m0, s4 // 4\n"]
    load = "\tglobal_load_lds_dwordx4 v168, s[8:9] // 8\n"
    assert [v[2] for v in violations(code + [load])] == ["M0", [9]]
    assert [v[2] for v in violations(code + ["\ts_nop 2 // 6\n", load])] == [[9]]
    assert violations(code + ["\ts_nop 3 // 6\n", load]) == []
    assert violations(code + ["\ts_mov_b64 vcc, s[8:9] // 6\n", load.replace("s[8:9]", "vcc")]) == []


def test_library_keeps_the_rules(tmp_path):
    if not OBJDUMP or not os.path.exists(LIB):
        pytest.skip("needs llvm-objdump and the built library")
    lib = shutil.copy(LIB, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=tmp_path)
    objects = sorted(p for p in os.listdir(tmp_path) if p.endswith("gfx950"))
    assert objects
    loads = 0
    for o in objects:
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", o], stdout=subprocess.PIPE,
                              text=True, cwd=tmp_path) as p:
            lines = p.stdout.readlines()
        loads += sum("global_load_lds" in l for l in lines)
        bad = violations(lines)
        assert not bad, f"{o}: {len(bad)} instructions read a register too early, first {bad[0]}"
        bad = reloads_before_exec(lines)
        assert not bad, f"{o}: {len(bad)} reloads before exec is restored, first {bad[0]}"
    assert loads > 1000
