"""Wait states that the hardware asks for and that the compiler does not see to where a memory instruction is written in assembly:
five between a vector instruction that writes a scalar register and a memory instruction that reads it (a lane read into the base of
a fetch, most of all).  Read from the library as it was built, every kernel in it."""

import re
import shutil
import struct
import subprocess
from pathlib import Path

import pytest

STATES = 5
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(library: bytes):
    """The gfx950 ELF files in a library's offload bundles."""
    for found in re.finditer(MAGIC, library):
        start = found.start()
        at = start + len(MAGIC)
        (count,) = struct.unpack_from("<Q", library, at)
        at += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", library, at)
            name = library[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in name and size:
                yield library[start + offset:start + offset + size]


def scalar_registers(operand: str) -> set:
    """The scalar registers an operand names."""
    if operand in ("vcc", "vcc_lo", "vcc_hi"):
        return {"vcc"}
    one = re.fullmatch(r"s(\d+)", operand)
    if one:
        return {int(one[1])}
    several = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    return set(range(int(several[1]), int(several[2]) + 1)) if several else set()


def operands(text: str) -> list:
    return [x.strip() for x in re.split(r",\s*(?![^\[]*\])", text)] if text else []


def too_early(listing: str) -> list:
    """(kernel, instruction, the one it comes too soon after, states between) of every such pair in a disassembly, over all ways in
    which control can come to the instruction."""
    code, kernel, at_address = [], "", {}
    for line in listing.splitlines():
        symbol = re.match(r"[0-9a-f]+ <(.+)>:$", line)
        if symbol:
            kernel = symbol[1]
            continue
        # "<tab>name operands // address: words <target>"
        parts = re.match(r"\s+([a-z]\w+)\s*(.*?)\s*//\s*([0-9A-F]+):(.*)$", line)
        if not parts:
            continue
        name, text, address, rest = parts[1], parts[2], int(parts[3], 16), parts[4]
        at_address[address] = len(code)
        target = re.search(r"<(\S+?)(?:\+0x([0-9a-f]+))?>", rest) if name.startswith(("s_cbranch", "s_branch")) else None
        code.append((kernel, name, text, address, (target[1], int(target[2] or "0", 16)) if target else None))
    begins = {}
    for kernel, _, _, address, _ in code:
        begins.setdefault(kernel, address)
    jumps_to = {}
    for i, (_, _, _, _, target) in enumerate(code):
        if target and target[0] in begins:
            jumps_to.setdefault(at_address.get(begins[target[0]] + target[1]), []).append(i)
    faults = []
    for i, (kernel, name, text, _, _) in enumerate(code):
        if not name.startswith(("global_", "buffer_", "scratch_", "flat_")):
            continue
        read = set().union(*[scalar_registers(x.split()[0]) for x in operands(text) if x])
        if not read:
            continue
        ways, seen = [(i, 0)], {}
        while ways:
            to, states = ways.pop()
            # what may have run before `to`: the instruction above it, unless that always goes elsewhere, and every jump to it
            before = jumps_to.get(to, [])
            if to > 0 and code[to - 1][0] == kernel and code[to - 1][1] not in ("s_branch", "s_endpgm", "s_setpc_b64"):
                before = before + [to - 1]
            for j in before:
                _, earlier, its_text, _, _ = code[j]
                its = operands(its_text)
                if earlier.startswith("v_") and any(scalar_registers(x) & read for x in its[:2 if "_co_" in earlier or "div_scale" in earlier else 1]):
                    faults.append((kernel, f"{name} {text}", f"{earlier} {its_text}", states))
                    continue
                now = states + (int(its_text, 0) + 1 if earlier == "s_nop" else 1)
                if now < STATES and seen.get(j, STATES) > now:
                    seen[j] = now
                    ways.append((j, now))
    return faults


def listing_of(path: Path) -> str:
    tool = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
    return subprocess.run([tool, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout


def test_the_check_sees_what_it_is_for():
    """Too early, soon enough, past a jump, and a register that the memory instruction does not read."""
    def told(*lines):
        return too_early("0000000000000000 <k>:\n" + "".join(f"\t{text}   // {4 * i:012X}: 00{rest}\n" for i, (text, rest) in enumerate(lines)))

    lane, load = ("v_readfirstlane_b32 s5, v1", ""), ("global_load_lds_dwordx4 v2, s[4:5]", "")
    assert [f[3] for f in told(lane, ("s_mov_b32 m0, s7", ""), ("s_nop 0", ""), load)] == [2]
    assert not told(lane, ("s_mov_b32 m0, s7", ""), ("s_nop 3", ""), load)
    assert not told(("v_readfirstlane_b32 s6, v1", ""), load)
    assert [f[3] for f in told(("s_branch 1", " <k+0xc>"), load, ("s_endpgm", ""), lane, ("s_branch 65532", " <k+0x4>"))] == [1]
    assert [f[3] for f in told(("v_cmp_gt_f32_e64 s[4:5], v1, v2", ""), ("global_load_dword v1, v2, s[4:5] offset:16", ""))] == [0]


def test_every_memory_instruction_waits_for_its_scalar_registers(tmp_path):
    from llm_runtime_study_amd.kernels import build

    if not (shutil.which("llvm-objdump") or Path("/opt/rocm/llvm/bin/llvm-objdump").exists()):
        pytest.skip("needs llvm-objdump")
    faults, kernels = [], 0
    for n, code in enumerate(code_objects(build.ensure_built().read_bytes())):
        (tmp_path / f"{n}.elf").write_bytes(code)
        listing = listing_of(tmp_path / f"{n}.elf")
        kernels += listing.count(">:\n")
        faults += too_early(listing)
    assert kernels > 100
    assert not faults, f"{len(faults)} of them, the first: {faults[:4]}"
