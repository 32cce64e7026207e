"""Rows of the embedding table: every form of the kernel, by the width of a row, its alignment and the bytes written."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,hidden", [(1, 8), (3, 64), (33, 1000), (7, 1001), (5, 1028), (127, 2048), (128, 2048), (129, 2056), (8191, 6144), (8192, 6144), (8193, 6152)])
def test_rows_of_the_table(tokens, hidden, dtype):
    """Rows that end inside a workgroup, rows of no whole pieces, and outputs below, at and above 1 MB and 192 MB, times a multiplier: one rounding in
    float32, so the bits are those of the table's values multiplied in float32."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(tokens + hidden)
    table, ids = torch.randn(97, hidden, generator=g).to(dtype).cuda(), torch.randint(0, 97, (tokens,), generator=g).int().cuda()
    out = torch.full((tokens, hidden), float("nan"), device="cuda")
    ops.embed(out, table, ids, 1.7)
    assert torch.equal(out, table.float()[ids.long()] * 1.7)
