"""Waits in the built gfx950 code.  The compiler inserts what its own instructions need, but nothing
inside an asm block, and it takes a block's outputs as written where the block stands.  So these tests
read the disassembly of the whole library, which holds every block as it was laid out:

  * a compare's or carry's result (VCC or an SGPR pair written by a VALU instruction) is read by no
    VALU instruction before two wait states have passed;
  * no instruction touches a register that an LDS read in flight will still write.
"""
import collections
import concurrent.futures as cf
import glob
import multiprocessing
import os
import re
import subprocess

import pytest

from sparsesnn_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
WAIT = 2
_SGPR = re.compile(r"\bvcc\b|\bs\d+\b|\bs\[\d+:\d+\]")
_VGPR = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")
_ADDRESS = re.compile(r"\s*([0-9A-F]{8,}):")
_TARGET = re.compile(r"<[^>+]+(?:\+0x([0-9a-f]+))?>\s*$")


def _sgprs(operand):
    out = set()
    for name in _SGPR.findall(operand):
        if name[1] == "[":
            lo, hi = name[2:-1].split(":")
            out.update(range(int(lo), int(hi) + 1))
        else:
            out.add(name if name == "vcc" else int(name[1:]))
    return out


def hazards(code):
    """(writer, reader) pairs of instructions closer than WAIT wait states, of one function."""
    found, recent, pos = [], [], 0  # recent: (position, SGPRs, text) of the latest compares and carries
    for _, text, _ in code:
        name, _, rest = text.partition(" ")
        if name == "s_nop":
            pos += int(rest, 0) + 1
            continue
        pos += 1
        if not name.startswith("v_") or ("vcc" not in rest and "s" not in rest):
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


def _vgprs(operands):
    out = set()
    for file, one, lo, hi in _VGPR.findall(operands):
        out.update((file, i) for i in (range(int(lo), int(hi) + 1) if lo else [int(one)]))
    return out


def in_flight(code):
    """Instructions that touch the destination of an LDS read not waited for, of one function, over
    all paths.  State: register -> LDS operations issued after its read (they return in order, so a
    wait for at most n outstanding ones covers those with n or more; scalar loads share the counter
    and return in any order, so they count for none)."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    ops, leaders = [], {0}
    for i, (_, text, target) in enumerate(code):
        name, _, rest = text.partition(" ")
        if name == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", rest)
            ops.append(("wait", int(m[1])) if m else None)
        elif name.startswith("ds_"):
            loads = any(k in name for k in ("read", "rtn", "permute", "swizzle"))
            dst, rest = (rest.split(", ", 1) if ", " in rest else (rest, "")) if loads else ("", rest)
            ops.append(("lds", _vgprs(dst), _vgprs(rest)))
        else:
            regs = _vgprs(rest) if not name.startswith("s_") else None
            ops.append(("use", regs) if regs else None)
        if name.startswith(("s_cbranch", "s_branch")):
            leaders |= {at[target], i + 1}
        elif name == "s_endpgm":
            leaders.add(i + 1)
    leaders = sorted(x for x in leaders if x < len(code))
    ends = dict(zip(leaders, [*leaders[1:], len(code)]))

    def run(block, state, found=None):
        state = dict(state)
        for i in range(block, ends[block]):
            op = ops[i]
            if op is None:
                continue
            if op[0] == "wait":
                state = {r: n for r, n in state.items() if n < op[1]}
                continue
            if state:
                hit = [r for r in op[-1] if r in state]
                if hit and found is not None:
                    found.append(code[i][1])
                for r in hit:
                    del state[r]
            if op[0] == "lds":
                state = {r: min(n + 1, 64) for r, n in state.items()}
                state.update((r, 0) for r in op[1])
        return state

    def successors(block):
        _, text, target = code[ends[block] - 1]
        if not text.startswith(("s_endpgm", "s_branch")) and ends[block] < len(code):
            yield ends[block]
        if target is not None:
            yield at[target]

    entry, work = {0: {}}, collections.deque([0])
    while work:
        block = work.popleft()
        out = run(block, entry[block])
        for nxt in successors(block):
            known = entry.setdefault(nxt, None)
            merged = dict(out) if known is None else {**known, **{r: n for r, n in out.items() if n < known.get(r, 99)}}
            if merged != known:
                entry[nxt] = merged
                work.append(nxt)
    found = []
    for block, state in entry.items():
        run(block, state, found)
    return found


def functions(lines):
    """(name, [(address, instruction, branch target or None)]) of a disassembly."""
    name, code = None, []
    for line in lines:
        if not line.startswith("\t"):
            m = re.match(r"(?:[0-9a-f]+ )?<(\S+)>:", line)
            if m:
                if code:
                    yield name, code
                name, code = m[1], []
            continue
        text, _, comment = line.partition("//")
        address = _ADDRESS.match(comment)
        if address is None:
            continue
        text, target = text.strip(), None
        if text.startswith(("s_cbranch", "s_branch")):
            target = (code[0][0] if code else int(address[1], 16)) + int(_TARGET.search(comment)[1] or "0", 16)
        code.append((int(address[1], 16), text, target))
    if code:
        yield name, code


def _scan(path):
    with subprocess.Popen([OBJDUMP, "-d", "--mcpu=gfx950", "--no-show-raw-insn", path], stdout=subprocess.PIPE,
                          text=True) as p:
        close, early = [], []
        for name, code in functions(p.stdout):
            close += [(name, h) for h in hazards(code)]
            if "fused_tile" in name:  # the kernels that read LDS in asm
                early += [(name, h) for h in in_flight(code)]
    return p.returncode, close, early


@pytest.fixture(scope="module")
def findings(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    tmp = tmp_path_factory.mktemp("lib")
    os.symlink(_lib.lib_path(), tmp / "lib.so")  # the code objects are extracted next to it
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp, check=True, stdout=subprocess.DEVNULL)
    objs = sorted(glob.glob(str(tmp / "lib.so.*gfx950")), key=os.path.getsize, reverse=True)
    assert objs
    with cf.ProcessPoolExecutor(4, mp_context=multiprocessing.get_context("spawn")) as ex:
        results = list(ex.map(_scan, objs))
    assert all(rc == 0 for rc, _, _ in results)
    return [[h for r in results for h in r[k]] for k in (1, 2)]


def _code(*texts):
    return [(4 * i, t, 4 * int(t.split()[1]) if t.startswith(("s_cbranch", "s_branch")) else None)
            for i, t in enumerate(texts)]


def test_hazards_finds_and_spares():
    one = ["v_cmp_le_f32_e32 vcc, s4, v1", "v_cndmask_b32_e32 v1, v1, v2, vcc"]
    assert len(hazards(_code(*one))) == 1 and not hazards(_code(one[0], "s_nop 1", one[1]))
    assert len(hazards(_code(one[0], "v_mov_b32_e32 v5, 0", one[1]))) == 1
    pair = ["v_cmp_le_f32_e64 s[4:5], s2, v1", "v_mov_b32_e32 v5, 0", "v_addc_co_u32_e64 v3, vcc, v3, v3, s[4:5]"]
    assert len(hazards(_code(*pair))) == 1 and not hazards(_code(*pair[:2], pair[1], pair[2]))


def test_in_flight_finds_and_spares():
    read, use = "ds_read_b64 v[2:3], v1", "v_mov_b32_e32 v5, v3"
    assert in_flight(_code(read, use)) == [use] and not in_flight(_code(read, "s_waitcnt lgkmcnt(0)", use))
    two = [read, "ds_read_b64 v[6:7], v1", "s_waitcnt lgkmcnt(1)"]
    assert not in_flight(_code(*two, use)) and len(in_flight(_code(*two, "v_mov_b32_e32 v6, 0"))) == 1
    # a branch around the wait: one path arrives with the read in flight
    assert in_flight(_code(read, "s_cbranch_scc0 3", "s_waitcnt lgkmcnt(0)", use, "s_endpgm")) == [use]


def test_library_waits_for_compares(findings):
    assert not findings[0], f"{len(findings[0])} reads too close to a compare or carry, first {findings[0][:3]}"


def test_library_waits_for_lds_reads(findings):
    assert not findings[1], f"{len(findings[1])} uses of registers with an LDS read in flight, first {findings[1][:3]}"
