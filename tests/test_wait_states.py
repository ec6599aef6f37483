"""Wait states in the built gfx950 code: a compare's or carry's result (VCC or an SGPR pair written by
a VALU instruction) is read by no VALU instruction before two wait states have passed.  The compiler
sees to that in its own code but inserts nothing inside an asm block, so this reads the disassembly of
the whole library, which holds every block as it was laid out."""
import concurrent.futures as cf
import glob
import os
import re
import subprocess

import pytest

from sparsesnn_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT = 2
_SGPR = re.compile(r"\bvcc\b|\bs\d+\b|\bs\[\d+:\d+\]")


def _sgprs(operand):
    out = set()
    for name in _SGPR.findall(operand):
        if name[1] == "[":
            lo, hi = name[2:-1].split(":")
            out.update(range(int(lo), int(hi) + 1))
        else:
            out.add(name if name == "vcc" else int(name[1:]))
    return out


def hazards(lines):
    """(writer, reader) pairs of instructions closer than WAIT wait states, of one disassembly."""
    found, recent, pos = [], [], 0  # recent: (position, SGPRs, text) of the latest compares and carries
    for line in lines:
        if not line.startswith("\t"):
            if line.rstrip().endswith(">:"):
                recent = []  # another function
            continue
        text = line.split("//")[0].strip()
        name, _, rest = text.partition(" ")
        if name == "s_nop":
            pos += int(rest, 0) + 1
            continue
        pos += 1
        if not name.startswith("v_") or ("vcc" not in rest and " s" not in line):
            continue
        ops = re.split(r",(?![^\[]*\])", rest)
        n_dst = 2 if "_co_" in name else 1
        reads = set().union(*(_sgprs(o) for o in ops[n_dst:]))
        found += [(w, text) for at, regs, w in recent if pos - at <= WAIT and reads & regs]
        writes = set().union(*(_sgprs(o) for o in ops[:n_dst]))
        recent = [r for r in recent if pos - r[0] <= WAIT and not r[1] <= writes]
        if writes and (name.startswith("v_cmp") or "_co_" in name):
            recent.append((pos, writes, text))
    return found


def test_hazards_finds_and_spares():
    one = ["\tv_cmp_le_f32_e32 vcc, s4, v1  // 0", "\tv_cndmask_b32_e32 v1, v1, v2, vcc  // 4"]
    assert len(hazards(one)) == 1 and not hazards([one[0], "\ts_nop 1", one[1]])
    assert len(hazards([one[0], "\tv_mov_b32_e32 v5, 0", one[1]])) == 1
    pair = ["\tv_cmp_le_f32_e64 s[4:5], s2, v1", "\tv_mov_b32_e32 v5, 0",
            "\tv_addc_co_u32_e64 v3, vcc, v3, v3, s[4:5]"]
    assert len(hazards(pair)) == 1 and not hazards([*pair[:2], pair[1], pair[2]])


def test_library_waits_for_compares(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    lib = tmp_path / "lib.so"  # the code objects are extracted next to it
    os.symlink(_lib.lib_path(), lib)
    subprocess.run([OBJDUMP, "--offloading", lib.name], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    objs = sorted(glob.glob(str(tmp_path / "lib.so.*gfx950")))
    assert objs

    def scan(path):
        with subprocess.Popen([OBJDUMP, "-d", "--mcpu=gfx950", "--no-show-raw-insn", path], stdout=subprocess.PIPE,
                              text=True) as p:
            found = hazards(p.stdout)
        assert p.returncode == 0
        return found

    with cf.ThreadPoolExecutor(4) as ex:
        found = [h for hs in ex.map(scan, objs) for h in hs]
    assert not found, f"{len(found)} reads too close to a compare or carry, first {found[:3]}"
