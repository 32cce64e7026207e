"""Kernels whose waits count what they have asked memory for keep their values in registers: a spilled value's way back counts among
the tiles on their way, and waits for all that were asked for before it.  Read from the library as it was built."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_wait_states import code_objects


def spills(tmp_path):
    """Kernel name -> vector registers it spills."""
    from llm_runtime_study_amd.kernels import build

    tool = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
    if not Path(tool).exists():
        pytest.skip("needs llvm-readelf")
    found = {}
    for n, code in enumerate(code_objects(build.ensure_built().read_bytes())):
        (tmp_path / f"{n}.elf").write_bytes(code)
        notes = subprocess.run([tool, "--notes", str(tmp_path / f"{n}.elf")], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s+- \.", notes):
            name, count = re.search(r"\.symbol:\s+'?(\S+?)\.kd", kernel), re.search(r"\.vgpr_spill_count:\s+(\d+)", kernel)
            if name and count:
                found[name[1]] = int(count[1])
    return found


def test_prompt_kernels_of_128_dims_spill_next_to_nothing(tmp_path):
    found = {name: count for name, count in spills(tmp_path).items() if re.search("attention_prefill_d128|attention_mixed_d128", name)}
    assert len(found) >= 60
    # groups of 16 queries: none but those with a linear bias, whose three workgroups a unit leave 168 registers; others a few, before
    # and behind the walk
    short = {name: count for name, count in found.items() if re.search(r"kernelILi1E", name) and not re.search(r"Lb[01]ELi[0-3]ELi[45]E", name)}
    assert short and not any(short.values()), {name: count for name, count in short.items() if count}
    assert max(found.values()) <= 10, {name: count for name, count in found.items() if count > 10}


def test_float32_products_add_up_runs_beside_their_products(tmp_path):
    """The large tiles of float32 products: inside the walk over K no block of instructions moves or adds sums while the matrix units wait
    (what a run of K leaves is added beside the next run's first products)."""
    from llm_runtime_study_amd.kernels import build

    source, out = build.SOURCE_DIR / "gemm_f32.hip", tmp_path / "gemm_f32.s"
    subprocess.run([build._hipcc(), *build.FLAGS, *build.FILE_FLAGS[source.name], "--cuda-device-only", "-S", str(source), "-o", str(out)], capture_output=True, check=True)
    kernels = {name: text for name, text in re.findall(r"^(_Z\w*gemm_f32_mfma_kernel\w*):(.*?)\.Lfunc_end", out.read_text(), re.M | re.S)}
    large = [text for name, text in kernels.items() if re.search(r"Li2ELi[24]ELi[24]ELi2ELi3ELi16ELi16E", name)]      # 64 x 64 and 128 x 128 outputs
    assert len(large) >= 2
    for text in large:
        walk = [block for block in re.split(r"\n(?=\.LBB)", text) if re.match(r"\.LBB\w+:\s*;.*Loop", block)]
        assert sum(block.count("v_mfma_f32_16x16x4") for block in walk) >= 128
        for block in walk:
            if "v_mfma_f32_16x16x4" not in block:
                assert len(re.findall(r"^\tv_", block, re.M)) <= 8, block
