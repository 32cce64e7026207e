"""Norms of many rows have eight waves on a SIMD: the kernel that adds up no product's splits takes at most 64 registers.  Read from the library
as it was built."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_wait_states import code_objects


def test_norms_without_splits_take_few_registers(tmp_path):
    from llm_runtime_study_amd.kernels import build

    reader = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"
    if not Path(reader).exists():
        pytest.skip("needs llvm-readelf")
    taken = {}
    for n, code in enumerate(code_objects(build.ensure_built().read_bytes())):
        if b"rmsnorm_vec_kernel" not in code:
            continue
        (tmp_path / f"{n}.elf").write_bytes(code)
        notes = subprocess.run([reader, "--notes", tmp_path / f"{n}.elf"], capture_output=True, text=True, check=True).stdout
        for name, count in re.findall(r"\.name: +(\S*rmsnorm_vec_kernel\S*).*?\.vgpr_count: +(\d+)", notes, re.S):
            taken[name] = int(count)
    plain = {name: count for name, count in taken.items() if "Lb0E" in name}
    assert len(plain) == 16 and len(taken) == 32
    assert max(plain.values()) <= 64, plain
