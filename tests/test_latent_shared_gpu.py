"""Latent attention whose tiles a workgroup shares through LDS, alone, against the kernel for any shape."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from llm_runtime_study_amd.kernels import ops

    return ops


# (cached tokens, new tokens): contexts that end at every place of a tile and a page, fewer tiles than are on their way, several requests
REQUESTS = [(0, 1), (0, 23), (31, 1), (300, 16), (77, 40), (160, 1)]


@pytest.mark.parametrize("rank,heads,page,window,splits,groups,extras", [
    (512, 32, 16, 0, 1, False, True), (512, 32, 16, 0, 4, False, False), (512, 20, 48, 40, 3, False, True), (256, 3, 16, 0, 2, False, True), (128, 70, 16, 0, 1, False, False),
    (512, 32, 16, 0, 1, True, True), (512, 5, 32, 100, 2, True, False), (256, 16, 16, -64, 1, True, True), (128, 33, 16, 0, 3, True, False)])
def test_shared_tiles(ops, rank, heads, page, window, splits, groups, extras):
    g = torch.Generator().manual_seed(rank + heads)
    width = rank + 64
    assert ops.latent_attention_groups_shares(rank, width, page)
    blocks = [-(-(a + b) // page) for a, b in REQUESTS]
    perm = torch.randperm(sum(blocks), generator=g).tolist()
    table, of, at, starts = torch.full((len(REQUESTS), max(blocks)), -1, dtype=torch.int32), [], [], []
    for r, (before, new) in enumerate(REQUESTS):
        table[r, :blocks[r]] = torch.tensor([perm.pop() for _ in range(blocks[r])])
        starts += [(len(of) + i, min(5, new - i)) for i in range(0, new, 5)]
        of += [r] * new
        at += list(range(before, before + new))
    pages = torch.randn(sum(blocks), 1, page, width, generator=g).bfloat16().cuda()
    value_pages = pages[:, :, :, :rank].transpose(2, 3).contiguous()
    tokens = len(of)
    queries = torch.randn(tokens, heads, width, generator=g).bfloat16().cuda()
    of, at, table = torch.tensor(of, dtype=torch.int32).cuda(), torch.tensor(at, dtype=torch.int32).cuda(), table.cuda()
    more = {"sink": torch.randn(heads, generator=g).cuda(), "gate": torch.randn(tokens, heads + 3, generator=g).bfloat16().cuda()[:, :heads]} if extras else {}
    want = torch.empty(tokens, heads * rank, dtype=torch.bfloat16, device="cuda")
    ops.latent_attention(want, queries, pages, table, of, at, rank, 0.06, window=window, **more)
    first, count = (torch.tensor(x, dtype=torch.int32).cuda() for x in zip(*starts)) if groups else (None, None)
    part_o, part_ml = (torch.full((tokens, heads * splits * n), float("nan"), device="cuda") for n in (rank, 2))
    got = torch.full_like(want, float("nan"))
    ops.latent_attention_groups(got, queries, pages, value_pages, table, of, at, first, count, 5 if groups else 1, rank, 0.06, window=window, splits=splits, part_o=part_o,
                                part_ml=part_ml, **more)
    # scores of a few units here: weights in bfloat16 (2^-9 each) and results rounded to it
    torch.testing.assert_close(got.float(), want.float(), rtol=2e-2, atol=2e-2)


@pytest.mark.parametrize("rank,heads,page,window,splits,size", [
    (512, 32, 16, 0, 1, 0), (512, 32, 16, 0, 4, 0), (512, 20, 48, 40, 3, 0), (256, 70, 16, 0, 2, 0), (128, 3, 16, 0, 7, 0),
    (512, 32, 16, 0, 1, 16), (512, 5, 32, 100, 2, 5), (256, 16, 16, -64, 3, 9), (128, 33, 16, 0, 5, 16)])
def test_shared_tiles_give_the_bits_of_waves_by_themselves(ops, rank, heads, page, window, splits, size):
    """A choice of experts behind such a layer may hang on the last bit, so the kernel that shares tiles makes the sums of the one that
    does not (which rows of any stride go to).  Then with slots that nothing was written to holding NaN."""
    requests = [(0, 1), (0, 45), (31, 1), (700, 1), (1000, 70), (77, 40)] if size else [(0, 1), (14, 1), (31, 1), (32, 1), (700, 1), (1500, 1)]
    g = torch.Generator().manual_seed(rank + heads + splits)
    width, blocks = rank + 64, [-(-(a + b) // page) for a, b in requests]
    perm = torch.randperm(sum(blocks), generator=g).tolist()
    table, of, at, starts, unwritten = torch.full((len(requests), max(blocks)), -1, dtype=torch.int32), [], [], [], torch.zeros(sum(blocks), page, dtype=torch.bool)
    for r, (before, new) in enumerate(requests):
        table[r, :blocks[r]] = torch.tensor([perm.pop() for _ in range(blocks[r])])
        unwritten[table[r, blocks[r] - 1], page - (blocks[r] * page - before - new):] = True
        starts += [(len(of) + i, min(size, new - i)) for i in range(0, new, size)] if size else []
        of += [r] * new
        at += list(range(before, before + new))
    pages = torch.randn(sum(blocks), 1, page, width, generator=g).bfloat16()
    tokens = len(of)
    queries = torch.randn(tokens, heads, width, generator=g).bfloat16().cuda()
    of, at, table = torch.tensor(of, dtype=torch.int32).cuda(), torch.tensor(at, dtype=torch.int32).cuda(), table.cuda()
    sink, gate = torch.randn(heads, generator=g).cuda(), torch.randn(tokens, heads, generator=g).bfloat16().cuda()
    first, count = (torch.tensor(x, dtype=torch.int32).cuda() for x in zip(*starts)) if size else (None, None)

    def run(pages, stride):
        pages = pages.cuda()
        part_o, part_ml = (torch.full((tokens, heads * splits * n), float("nan"), device="cuda") for n in (rank, 2))
        out = torch.full((tokens, stride), float("nan"), dtype=torch.bfloat16, device="cuda")[:, :heads * rank]
        ops.latent_attention_groups(out, queries, pages, pages[:, :, :, :rank].transpose(2, 3).contiguous(), table, of, at, first, count, size or 1, rank, 0.06,
                                    sink=sink, gate=gate, window=window, splits=splits, part_o=part_o, part_ml=part_ml)
        return out

    got = run(pages, heads * rank)
    assert torch.equal(got, run(pages, heads * rank + 1)) and not got.isnan().any()
    pages[:, 0][unwritten] = float("nan")
    assert torch.equal(got, run(pages, heads * rank))
