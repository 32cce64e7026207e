"""Prompt attention for heads of 128 over contexts that end about the places where a walk looks up the addresses of its next 32 tiles
of keys (two tiles into the second and every later 32), against the kernel for any shape."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from llm_runtime_study_amd.kernels import ops

    return ops


# tiles of 32 keys: one to four; the second block's end; the turn that looks up the third and the one that first uses it; the fourth
@pytest.mark.parametrize("keys", [1, 33, 65, 100, 1990, 2048, 2049, 2080, 2081, 3009, 3041, 3071, 3105, 4097, 5000])
@pytest.mark.parametrize("heads,size,page,window,splits", [(2, 32, 16, 0, 1), (4, 16, 48, 0, 1), (4, 32, 32, 0, 1), (3, 16, 16, 0, 2), (6, 32, 16, 0, 1), (9, 16, 16, 2500, 1),
                                                           (2, 32, 48, 2300, 1)])
def test_walks_of_many_tiles(ops, keys, heads, size, page, window, splits):
    nkv, d = 2, 128
    nq, tokens = heads * nkv, min(keys, 35)
    before = keys - tokens
    g = torch.Generator().manual_seed(keys + heads)
    pages = -(-keys // page)
    k_pages = torch.randn(pages, nkv, page, d, generator=g).bfloat16().cuda()
    v_pages = torch.randn(pages, nkv, d, page, generator=g).bfloat16().cuda()
    table = torch.randperm(pages, generator=g).to(torch.int32)[None].cuda()
    q = (torch.randn(tokens, nq * d, generator=g) * 2).bfloat16().cuda()
    of, at = torch.zeros(tokens, dtype=torch.int32).cuda(), torch.arange(before, keys, dtype=torch.int32).cuda()
    want, got = (torch.full((tokens, nq * d), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    ops.attention(want, q, k_pages, v_pages, table, of, at, nq, 1 / math.sqrt(d), window)
    starts = list(range(0, tokens, size))[::-1]
    first, count = (torch.tensor(x, dtype=torch.int32).cuda() for x in (starts, [min(size, tokens - s) for s in starts]))
    part_o, part_ml = (torch.full((tokens, nq * splits * n), float("nan"), device="cuda") for n in (d, 2))
    ops.attention_prefill(got, q, k_pages, v_pages, table, of, at, first, count, nq, 1 / math.sqrt(d), window, size, keys, splits, part_o, part_ml,
                          one_request=True)
    torch.testing.assert_close(got.float(), want.float(), rtol=2e-2, atol=2e-2)      # weights and results in bfloat16
