"""Latent attention in parts: any number of them, ranks of whole and broken pieces of four dims, contexts that leave parts without keys."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,width", [(512, 576), (128, 192), (500, 504), (42, 48), (4, 8)])
@pytest.mark.parametrize("splits", [2, 4, 5, 15, 17, 64])
def test_parts_meet_as_if_undivided(rank, width, splits):
    """Against the same walk undivided: sums of 32 bits in another order, weights and results rounded to bfloat16 (2^-8 of values of order one,
    twice)."""
    from llm_runtime_study_amd.kernels import ops

    lengths, heads, page = [1, 33, 700, 2100], 5, 16
    g = torch.Generator().manual_seed(rank + splits)
    tokens, most = len(lengths), -(-max(lengths) // page)
    pages = torch.randn(tokens * most, 1, page, width, generator=g).bfloat16().cuda()
    values = pages[:, :, :, :rank].transpose(2, 3).contiguous()
    table = torch.randperm(tokens * most, generator=g).view(tokens, most).int().cuda()
    of, at = torch.arange(tokens, dtype=torch.int32).cuda(), torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    queries, sink = torch.randn(tokens, heads, width, generator=g).bfloat16().cuda(), torch.randn(heads, generator=g).cuda()
    gate = torch.randn(tokens, heads, generator=g).bfloat16().cuda()
    outs = []
    for parts in (1, splits):
        out = torch.full((tokens, heads * rank), float("nan"), dtype=torch.bfloat16, device="cuda")
        part_o, part_ml = (torch.full((tokens, heads * parts * n), float("nan"), device="cuda") for n in (rank, 2))
        ops.latent_attention_groups(out, queries, pages, values, table, of, at, None, None, 1, rank, width ** -0.5, sink=sink, gate=gate, splits=parts,
                                    part_o=part_o, part_ml=part_ml)
        outs.append(out.float())
    torch.testing.assert_close(outs[1], outs[0], rtol=2 ** -6, atol=2 ** -6)
