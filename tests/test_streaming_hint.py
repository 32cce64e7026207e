"""What several workgroups read side by side, or a cache keeps until the next step, is loaded without the hint that gives its lines up.
Read from the library as it was built."""

import re
import shutil
from pathlib import Path

import pytest

from tests.test_wait_states import code_objects, listing_of


def wide_loads(tmp_path, pattern):
    """Kernel name -> (16-byte loads with the hint, without) of the kernels whose name has the pattern."""
    from llm_runtime_study_amd.kernels import build

    if not (shutil.which("llvm-objdump") or Path("/opt/rocm/llvm/bin/llvm-objdump").exists()):
        pytest.skip("needs llvm-objdump")
    found = {}
    for n, code in enumerate(code_objects(build.ensure_built().read_bytes())):
        if re.search(pattern.encode(), code):
            (tmp_path / f"{n}.elf").write_bytes(code)
            for name, body in re.findall(rf"<(\S*{pattern}\S*)>:\n((?:.+\n)*)", listing_of(tmp_path / f"{n}.elf")):
                loads = re.findall(r"\tglobal_load_dwordx4 ([^/]*)", body)
                found[name] = (sum(" nt" in x for x in loads), sum(" nt" not in x for x in loads))
    return found


def test_experts_with_several_tiles_share_their_weights(tmp_path):
    """The kernel of tiles of 32 rows has both: weights of an expert with one tile, which are read once, and of one with more (four or two
    loads a slice, and one of the rows')."""
    found = wide_loads(tmp_path, "moe_experts_bf16_kernel")
    assert len(found) == 4
    for name, (once, shared) in found.items():
        weights = int(re.search(r"Li(\d+)E", name)[1]) // 32
        assert once >= weights and shared >= weights + 2, (name, once, shared)


def test_decode_attention_has_both(tmp_path):
    """Keys and values with the hint in the one form for it and without in the others; beside a prompt portion with and without, by the size
    of the pages (eight values and eight keys a tile, asked for at two places and more)."""
    found = wide_loads(tmp_path, "attention_decode_bf16_kernel")
    asked = {name: counts for name, counts in found.items() if re.search(r"Lb[01]ELi4ELb[01]ELb[01]ELb1E", name)}
    assert len(asked) >= 12 and all(once > 0 for once, _ in asked.values())
    assert not any(once for name, (once, _) in found.items() if name not in asked)
    mixed = wide_loads(tmp_path, "attention_mixed_d128_kernel")
    assert mixed and all(once >= 32 and plain >= 32 for once, plain in mixed.values())
