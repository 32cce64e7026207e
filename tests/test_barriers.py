"""Barriers of the few-rows products: where the waves of a workgroup take different ways through the walk over K, none stands on one of
them.  Read from the library as it was built: each barrier of the source is there once, not once for every way."""

import re
import shutil
from pathlib import Path

import pytest

from tests.test_wait_states import code_objects, listing_of


def test_few_rows_products_have_a_barrier_once(tmp_path):
    from llm_runtime_study_amd.kernels import build

    if not (shutil.which("llvm-objdump") or Path("/opt/rocm/llvm/bin/llvm-objdump").exists()):
        pytest.skip("needs llvm-objdump")
    wrong, kernels = {}, 0
    for n, code in enumerate(code_objects(build.ensure_built().read_bytes())):
        (tmp_path / f"{n}.elf").write_bytes(code)
        for name, body in re.findall(r"<(\S*gemm_bf16_skinny_kernel\S*)>:\n((?:.+\n)*)", listing_of(tmp_path / f"{n}.elf")):
            mt, rt, norm, swiglu, whole_lines = (int(x) for x in re.search(r"ILi(\d)ELi(\d)ELi\dELi\dELb(\d)ELb(\d)ELb\dELb(\d)", name).groups())
            if whole_lines:       # its waves walk equally many steps, one way for all of them
                continue
            # around a row tile's sums; one before the sums of squares for the next norm, one before the factors of the norm it finishes
            wanted = 2 * rt - 1 + (mt == 1 and not swiglu) + (mt == 1 and not norm)
            found = len(re.findall(r"\ts_barrier\b", body))
            kernels += 1
            if found != wanted:
                wrong[name] = (found, wanted)
    assert kernels >= 40
    assert not wrong
