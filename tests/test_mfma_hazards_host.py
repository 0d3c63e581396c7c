"""CPU check of the built 2 x 2-wave tiles: their MX MFMAs are written in assembly, so the compiler does not
keep the distances that the matrix cores need around them.  The code of the objects is scanned for

* a vector write of an MFMA's operand (or accumulator) less than two wait states ahead of it;
* a vector instruction that touches an MFMA's accumulator before its result is there (20 wait states after a
  sixteen-pass MFMA)."""
import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
LLVM = Path("/opt/rocm/llvm/bin")
OPERAND_STATES, RESULT_STATES = 2, 20


def _registers(operand):
    """'v[4:7]' / 'a3' -> {('v', 4), ...}; nothing for scalars, literals and modifiers."""
    m = re.match(r"([va])\[(\d+):(\d+)\]$|([va])(\d+)$", operand.strip().split(" ")[0])
    if not m:
        return set()
    if m.group(4):
        return {(m.group(4), int(m.group(5)))}
    return {(m.group(1), r) for r in range(int(m.group(2)), int(m.group(3)) + 1)}


def _instructions(lines):
    """(address, mnemonic, operands) of a disassembly's instructions."""
    for line in lines:
        m = re.match(r"\t([a-z][a-z0-9_]+)\s*(.*?)\s*// ([0-9A-F]+):", line)
        if m:
            yield int(m.group(3), 16), m.group(1), m.group(2).split(", ")


def _blocks(code):
    """{first address: (instructions, successors' addresses)} of the basic blocks."""
    target = lambda at, ops: at + 4 + 4 * ((int(ops[0]) ^ 0x8000) - 0x8000)  # noqa: E731
    branches = [i for i, (_, name, _) in enumerate(code) if name.startswith(("s_branch", "s_cbranch", "s_endpgm"))]
    starts = {code[0][0]} | {code[i + 1][0] for i in branches if i + 1 < len(code)}
    starts |= {target(code[i][0], code[i][2]) for i in branches if code[i][1] != "s_endpgm"}
    blocks, block = {}, []
    for i, ins in enumerate(code):
        block.append(ins)
        after = code[i + 1][0] if i + 1 < len(code) else None
        if after is None or after in starts:
            at, name, ops = ins
            next_ = [] if name in ("s_branch", "s_endpgm") or after is None else [after]
            if name.startswith(("s_branch", "s_cbranch")):
                next_.append(target(at, ops))
            blocks[block[0][0]] = (block, next_)
            block = []
    return blocks


def _run(block, state, fault=None):
    """The state after a block: {register: states since its vector write} and the same since the MFMA whose result it
    is, as far as they matter."""
    writes, results = ({r: -age for r, age in part.items()} for part in state)
    clock = mfmas = 0
    for at, name, operands in block:
        if name == "s_nop":
            clock += int(operands[0], 0) + 1
            continue
        clock += 1
        if not name.startswith("v_"):
            continue
        regs = [_registers(o) for o in operands]
        if name.startswith("v_mfma") and operands[0].startswith("a"):
            mfmas += 1
            for r in set().union(*regs[1:]):
                if fault and clock - writes.get(r, -100) - 1 < OPERAND_STATES:
                    fault(f"{at:x} {name}: {r} written {clock - writes[r] - 1} states before")
            for r in regs[0]:
                results[r] = clock
            continue
        for r in set().union(*regs):
            if fault and clock - results.get(r, -100) - 1 < RESULT_STATES:
                fault(f"{at:x} {name}: {r} is the result of an MFMA {clock - results[r] - 1} states before")
        for r in regs[0] | (regs[1] if "swap" in name else set()):
            writes[r] = clock
    return tuple({r: clock - c for r, c in part.items() if clock - c < RESULT_STATES} for part in (writes, results)), mfmas


def _scan(lines):
    """(assembly MFMAs, faults) of one disassembly, over every path through its branches."""
    blocks = _blocks(list(_instructions(lines)))
    into = {at: ({}, {}) for at in blocks}
    work = list(blocks)
    while work:
        at = work.pop()
        block, next_ = blocks[at]
        out, _ = _run(block, into[at])
        for to in next_:
            merged = tuple({r: min(a.get(r, 99), b.get(r, 99)) for r in a.keys() | b.keys()}
                           for a, b in zip(into[to], out))
            if merged != into[to]:
                into[to] = merged
                work.append(to)
    faults = []
    return sum(_run(block, into[at], faults.append)[1] for at, (block, _) in blocks.items()), faults


def test_scan_sees_both_faults():
    mfma = "v_mfma_scale_f32_16x16x128_f8f6f4 a[0:3], v[0:7], v[8:15], a[0:3], v16, v17 op_sel_hi:[0,0,0]"

    def scan(*code):
        return _scan([f"\t{c} // {8 * i:012X}:" for i, c in enumerate((*code, "s_endpgm"))])

    assert scan("v_mov_b32_e32 v9, v20", "s_nop 1", mfma) == (1, [])
    assert len(scan("v_mov_b32_e32 v9, v20", "s_nop 0", mfma)[1]) == 1
    assert len(scan("v_accvgpr_write_b32 a3, 0", "s_barrier", mfma)[1]) == 1
    assert len(scan(mfma, "s_nop 15", "v_accvgpr_read_b32 v1, a2")[1]) == 1
    assert scan(mfma, "s_nop 15", "s_nop 15", "v_accvgpr_read_b32 v1, a2") == (1, [])
    # by way of a branch: a loop's last write (from 32 + 4 back to 8), and past the states that would have sufficed
    assert len(scan("s_nop 0", mfma, "s_nop 15", "v_mov_b32_e32 v17, 0", "s_cbranch_scc1 65529")[1]) == 1
    assert scan("v_mov_b32_e32 v17, 0", "s_cbranch_scc0 1", "s_nop 7", mfma) == (1, [])
    assert len(scan("v_mov_b32_e32 v17, 0", "s_cbranch_scc0 3", "s_nop 7", mfma)[1]) == 1


@pytest.mark.parametrize("stem", ["gemm_tile", "gemm_tile_grouped"])
def test_built_tiles_keep_the_distances(stem, tmp_path):
    obj = ROOT / "vllm-mach_amd" / "_build" / f"{stem}.o"
    if not obj.exists() or not (LLVM / "clang-offload-bundler").exists():
        pytest.skip("no built object (run __graft_entry__.build() first) or no disassembler")
    code = tmp_path / f"{stem}.co"
    fatbin = tmp_path / f"{stem}.fatbin"
    subprocess.run([LLVM / "llvm-objcopy", f"--dump-section=.hip_fatbin={fatbin}", obj], check=True)
    subprocess.run([LLVM / "clang-offload-bundler", "--unbundle", "--type=o", f"--input={fatbin}", f"--output={code}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    text = subprocess.run([LLVM / "llvm-objdump", "-d", "--no-show-raw-insn", code], check=True, capture_output=True,
                          text=True).stdout
    mfmas, faults = _scan(text.splitlines())
    assert mfmas >= 480  # none went unread
    assert not faults, faults[:10]
