"""Wait states that gfx950 needs from the program, checked in the listing of every kernel of the built library: around inline
asm the compiler puts none.

* an accumulator is read, copied or overwritten no sooner than 24 wait states behind the MFMA that wrote it (v_mfma
  32x32x64 on 8-bit operands needs 20; 24 is what the kernels put there, so a smaller gap has come in before them);
* an LDS-DMA load (buffer_load ... lds) comes at least one wait state behind the scalar instruction that wrote M0, its LDS
  address;
* a memory instruction reads scalar registers that a vector instruction wrote at least five wait states before;
* a lane move (DPP, permlane swap) reads a register at least two wait states behind the vector instruction that wrote it.

A wait state is one issued instruction, s_nop n counts n + 1; every path through branches and loops is followed.
"""
import os
import re
import struct
import subprocess

import pytest

from h3_tp2_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MFMA_STATES = 24
M0_STATES = 1
SGPR_STATES = 5
LANE_STATES = 2


def _code_objects(path):
    """The gfx950 code objects of a library's fat binary (one bundle per source file)."""
    data = open(path, "rb").read()
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, data):
        p = m.start()
        (n,) = struct.unpack_from("<Q", data, p + 24)
        if n > 16:                                        # the magic as a plain string of the loader
            continue
        q = p + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, q)
            if b"gfx950" in data[q + 24:q + 24 + length] and size:
                yield data[p + off:p + off + size]
            q += 24 + length


def parse(listing):
    """{kernel: [(mnemonic, operands, index of the branch target or None), ...]} of llvm-objdump's listing."""
    kernels = {}
    addr_of, insns = {}, None
    for line in listing.splitlines():
        head = re.match(r"^([0-9a-f]+) <([^>]+)>:", line)
        if head:
            base, insns, addr_of = int(head.group(1), 16), [], {}
            kernels[head.group(2)] = (insns, addr_of, base)
            continue
        m = re.match(r"^\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)$", line)
        if not m or insns is None:
            continue
        addr_of[int(m.group(3), 16)] = len(insns)
        t = re.search(r"<[^>+]+\+0x([0-9a-f]+)>", m.group(4)) if "branch" in m.group(1) else None
        insns.append((m.group(1), m.group(2), int(t.group(1), 16) if t else None))
    return {k: [(op, args, addr_of.get(base + t) if t is not None else None) for op, args, t in ins]
            for k, (ins, addr_of, base) in kernels.items()}


def _states(op, args):
    return int(args.split()[0], 0) + 1 if op == "s_nop" else 1


def _next(insns, i):
    op, _, target = insns[i]
    if op.startswith("s_endpgm"):
        return ()
    if op == "s_branch":
        return (target,)
    nxt = (i + 1,) if i + 1 < len(insns) else ()
    return nxt + ((target,) if op.startswith("s_cbranch") else ())


def _within(insns, i, states):
    """The instructions fewer than ``states`` wait states behind instruction i."""
    todo, seen = [(n, 0) for n in _next(insns, i)], {}
    while todo:
        j, gap = todo.pop()
        if gap >= states or seen.get(j, states) <= gap:
            continue
        seen[j] = gap
        yield j
        todo += [(n, gap + _states(*insns[j][:2])) for n in _next(insns, j)]


def _vregs(text):
    out = {(c, int(i)) for c, i in re.findall(r"\b([av])(\d+)\b", text)}
    for c, lo, hi in re.findall(r"\b([av])\[(\d+):(\d+)\]", text):
        out |= {(c, i) for i in range(int(lo), int(hi) + 1)}
    return out


def mfma_gaps(insns):
    """(wait states, MFMA, reader) of every access too close behind the MFMA that wrote its register."""
    regs = [None] * len(insns)
    out = []
    for i, (op, args, _) in enumerate(insns):
        if not op.startswith("v_mfma"):
            continue
        todo, seen = [(n, 0, frozenset(_vregs(args.split(", ")[0]))) for n in _next(insns, i)], {}
        while todo:
            j, gap, dest = todo.pop()
            if gap >= MFMA_STATES or not dest or seen.get((j, dest), MFMA_STATES) <= gap:
                continue
            seen[(j, dest)] = gap
            o, a, _ = insns[j]
            if o.startswith("v_mfma"):                    # its own accumulator is forwarded; the other operands are not
                d, x, y = a.split(", ")[:3]
                if dest & _vregs(x + " " + y):
                    out.append((gap, i, j))
                dest = dest - _vregs(d)
            else:
                regs[j] = _vregs(a) if regs[j] is None else regs[j]
                if dest & regs[j]:
                    out.append((gap, i, j))
                    continue
            todo += [(n, gap + _states(o, a), dest) for n in _next(insns, j)]
    return out


def m0_gaps(insns):
    """The LDS-DMA loads too close behind a write of M0."""
    return [j for i, (op, args, _) in enumerate(insns) if op.startswith("s_") and re.match(r"m0\b", args)
            for j in _within(insns, i, M0_STATES) if insns[j][0].startswith("buffer_load") and insns[j][1].endswith("lds")]


def _sgprs(text):
    out = {int(i) for i in re.findall(r"\bs(\d+)\b", text)}
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out |= set(range(int(lo), int(hi) + 1))
    return out | ({"vcc"} if re.search(r"\bvcc\b", text) else set())


def sgpr_gaps(insns):
    """The memory instructions too close behind a vector instruction that wrote one of their scalar registers."""
    out = []
    for i, (op, args, _) in enumerate(insns):
        if not op.startswith("v_"):
            continue
        dest = _sgprs(", ".join(args.split(", ")[:2 if "_co_" in op else 1]))
        out += [j for j in (_within(insns, i, SGPR_STATES) if dest else ())
                if re.match(r"(buffer|global|flat|scratch)_", insns[j][0]) and _sgprs(insns[j][1]) & dest]
    return out


def lane_gaps(insns):
    """The lane moves too close behind a vector instruction that wrote the register they move."""
    moves = {i: _vregs(args if "permlane" in op else args.split(", ")[1].split()[0])
             for i, (op, args, _) in enumerate(insns) if "permlane" in op or op.endswith("_dpp")}
    if not moves:
        return []
    return [j for i, (op, args, _) in enumerate(insns) if op.startswith("v_") and not op.startswith("v_cmp")
            for j in _within(insns, i, LANE_STATES) if j in moves and _vregs(args.split(", ")[0]) & moves[j]]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    assert os.path.exists(OBJDUMP), "the ROCm toolchain that builds the library has no llvm-objdump"
    d = tmp_path_factory.mktemp("code")
    out = {}
    for n, co in enumerate(_code_objects(_lib.LIB_PATH)):
        f = d / f"{n}.o"
        f.write_bytes(co)
        out.update(parse(subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True,
                                        text=True).stdout))
    assert sum(any(op.startswith("v_mfma") for op, _, _ in ins) for ins in out.values()) > 40
    return out


def test_accumulators_are_read_late_enough(kernels):
    bad = {k: min(g) for k, g in ((k, mfma_gaps(ins)) for k, ins in kernels.items()) if g}
    assert not bad, bad


def test_m0_is_written_early_enough(kernels):
    bad = {k: len(g) for k, g in ((k, m0_gaps(ins)) for k, ins in kernels.items()) if g}
    assert not bad, bad


def test_scalar_registers_are_written_early_enough(kernels):
    bad = {k: len(g) for k, g in ((k, sgpr_gaps(ins)) for k, ins in kernels.items()) if g}
    assert not bad, bad


def test_lanes_move_late_enough(kernels):
    bad = {k: len(g) for k, g in ((k, lane_gaps(ins)) for k, ins in kernels.items()) if g}
    assert not bad, bad


# ---- the checks themselves, on listings with a known answer ----

def _insns(*lines):
    """Instructions at 4-byte steps from 0x1000; a branch is written as ("s_cbranch_scc1 2", its target's ordinal)."""
    text = "0000000000001000 <k>:\n"
    for i, x in enumerate(lines):
        t, target = x if isinstance(x, tuple) else (x, None)
        text += f"\t{t} // {0x1000 + 4 * i:012X}: 00000000" + (f" <k+0x{4 * target:x}>" if target is not None else "") + "\n"
    (ins,) = parse(text).values()
    assert len(ins) == len(lines)
    return ins


_LOAD = "buffer_load_dwordx4 v1, s[4:7], 0 offen lds"


def test_finds_a_copy_close_behind_its_mfma():
    mfma, copy = "v_mfma_f32_32x32x64_f8f6f4 a[0:15], v[0:7], v[8:15], a[0:15]", "v_accvgpr_read_b32 v20, a15"
    assert mfma_gaps(_insns(mfma, "s_nop 15", "s_nop 6", copy)) == [(23, 0, 3)]
    assert mfma_gaps(_insns(mfma, "s_nop 15", "s_nop 7", copy)) == []
    # the next MFMA takes the block over, and what follows counts from it
    assert mfma_gaps(_insns(mfma, "s_nop 15", mfma, "s_nop 15", "s_nop 6", copy)) == [(23, 2, 5)]
    # a loop's exit is far enough, its way back to the top is not
    assert mfma_gaps(_insns(copy, mfma, ("s_cbranch_scc1 65533", 0), "s_nop 15", "s_nop 6", copy)) == [(1, 1, 0)]


def test_finds_a_load_right_behind_m0():
    assert m0_gaps(_insns("s_mov_b32 m0, s1", _LOAD, "s_mov_b32 m0, s2", "s_nop 0", _LOAD)) == [1]
    # around a loop: the load at the top right behind the write at the bottom
    assert m0_gaps(_insns("s_nop 0", _LOAD, "s_mov_b32 m0, s1", ("s_cbranch_scc1 65533", 1), "s_endpgm")) == []
    assert m0_gaps(_insns(("s_branch 1", 2), _LOAD, "s_mov_b32 m0, s1", ("s_branch 65533", 1), "s_endpgm")) == []


def test_finds_a_descriptor_right_behind_its_writer():
    write = "v_readfirstlane_b32 s6, v2"
    assert sgpr_gaps(_insns(write, "s_nop 3", _LOAD)) == [2]
    assert sgpr_gaps(_insns(write, "s_nop 4", _LOAD)) == []
    assert sgpr_gaps(_insns("s_nop 0", _LOAD, write, "s_nop 2", ("s_cbranch_scc1 65532", 1), "s_endpgm")) == [1]


def test_finds_a_lane_move_right_behind_its_writer():
    write = "v_maximum3_f32 v3, v3, |v4|, |v5|"
    dpp, swap = "v_mov_b32_dpp v6, v3 row_shl:8 row_mask:0xf bank_mask:0xf", "v_permlane32_swap_b32_e32 v7, v3"
    assert lane_gaps(_insns(write, "s_nop 0", dpp)) == [2] and lane_gaps(_insns(write, "s_nop 1", dpp)) == []
    assert lane_gaps(_insns(write, swap)) == [1] and lane_gaps(_insns(write, "s_nop 1", swap)) == []
    assert lane_gaps(_insns(write, "v_mov_b32_dpp v6, v4 row_shl:8 row_mask:0xf bank_mask:0xf")) == []
