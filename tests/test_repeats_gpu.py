"""Kernels that have memory write tiles into LDS, launched many times over the same inputs: every launch gives the first one's bits.
(A wait that is missing between a wave's reads of a stage and its refilling, or before a fetch's base, shows as a rare difference.)"""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

LAUNCHES = 300


def all_alike(launch, out):
    launch()
    torch.cuda.synchronize()
    first, bad = out.clone(), torch.zeros((), dtype=torch.int64, device="cuda")
    assert torch.isfinite(first).all()
    for _ in range(LAUNCHES):
        launch()
        bad += (out != first).any()
    assert int(bad) == 0, f"{int(bad)} of {LAUNCHES} launches differ from the first"


@pytest.mark.parametrize("nq,nkv,tokens,before,window,linear", [(64, 8, 512, 0, 0, False), (16, 8, 1024, 3000, 0, False), (32, 8, 700, 0, 128, True), (40, 8, 300, 2100, 0, False)])
def test_prompt_attention(nq, nkv, tokens, before, window, linear):
    from llm_runtime_study_amd.kernels import ops

    d, page, keys = 128, 16, before + tokens
    g = torch.Generator().manual_seed(tokens)
    pages = -(-keys // page)
    k, v = torch.randn(pages, nkv, page, d, generator=g).bfloat16().cuda(), torch.randn(pages, nkv, d, page, generator=g).bfloat16().cuda()
    table = torch.randperm(pages, generator=g).int()[None].cuda()
    q, out = torch.randn(tokens, nq * d, generator=g).bfloat16().cuda(), torch.empty(tokens, nq * d, dtype=torch.bfloat16, device="cuda")
    of, at = torch.zeros(tokens, dtype=torch.int32).cuda(), torch.arange(before, keys, dtype=torch.int32).cuda()
    size = ops.attention_prefill_group(tokens, keys)
    starts = list(range(0, tokens, size))[::-1]
    first, count = (torch.tensor(x, dtype=torch.int32).cuda() for x in (starts, [min(size, tokens - s) for s in starts]))
    distance = (torch.rand(nq, generator=g) * 0.1).cuda() if linear else None
    all_alike(lambda: ops.attention_prefill(out, q, k, v, table, of, at, first, count, nq, 1 / math.sqrt(d), window, size, keys, distance=distance, one_request=True), out)


@pytest.mark.parametrize("heads,new", [(32, 1), (8, 40)])
def test_latent_attention(heads, new):
    from llm_runtime_study_amd.kernels import ops

    rank, page, requests, before = 512, 16, 8, 900
    g = torch.Generator().manual_seed(heads)
    width, blocks = rank + 64, -(-(before + new) // page)
    pages = torch.randn(requests * blocks, 1, page, width, generator=g).bfloat16().cuda()
    table = torch.randperm(requests * blocks, generator=g).int().view(requests, blocks).cuda()
    tokens = requests * new
    of = torch.arange(requests, dtype=torch.int32).repeat_interleave(new).cuda()
    at = torch.arange(before, before + new, dtype=torch.int32).repeat(requests).cuda()
    queries, out = torch.randn(tokens, heads, width, generator=g).bfloat16().cuda(), torch.empty(tokens, heads * rank, dtype=torch.bfloat16, device="cuda")
    size = min(new, 16)
    starts = [(r * new + i, min(size, new - i)) for r in range(requests) for i in range(0, new, size)]
    first, count = (torch.tensor(x, dtype=torch.int32).cuda() for x in zip(*starts)) if new > 1 else (None, None)
    values = pages[:, :, :, :rank].transpose(2, 3).contiguous()
    part_o, part_ml = (torch.empty(tokens, heads * 4 * n, device="cuda") for n in (rank, 2))
    all_alike(lambda: ops.latent_attention_groups(out, queries, pages, values, table, of, at, first, count, size, rank, 0.06, splits=4, part_o=part_o, part_ml=part_ml), out)


@pytest.mark.parametrize("rows,n,k", [((300,) * 24 + (5,), 1024, 704), ((900, 128, 1, 257), 512, 192)])
def test_routed_experts(rows, n, k):
    from llm_runtime_study_amd.kernels import ops

    g, tile = torch.Generator().manual_seed(n), 128
    tiles = [-(-m // tile) for m in rows]
    listed, experts, at = torch.full((sum(tiles), tile), -1, dtype=torch.int32), torch.empty(sum(tiles), dtype=torch.int32), 0
    order = torch.randperm(sum(rows), generator=g).int()
    for e, m in enumerate(rows):
        experts[at:at + tiles[e]] = e
        listed[at:at + tiles[e]].view(-1)[:m] = order[sum(rows[:e]):sum(rows[:e + 1])]
        at += tiles[e]
    x, w = torch.randn(sum(rows), k, generator=g).bfloat16().cuda(), torch.randn(len(rows), n, k, generator=g).bfloat16().cuda()
    out = torch.zeros(listed.numel(), n, dtype=torch.bfloat16, device="cuda")
    listed, experts = listed.flatten().cuda(), experts.cuda()
    all_alike(lambda: ops.moe_experts(out, x, w, listed, experts, tile, 1, gather=True, relu_squared=False), out)
