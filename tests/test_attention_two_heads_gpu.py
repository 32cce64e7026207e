"""Prompt attention with two heads of 128 a kv group, alone: the waves' two ways of sharing a group of more than 16 queries (a block
of 16 each, or two neighbouring groups that walk their keys together) against the kernel for any shape."""

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


# tokens that fill groups of 32, leave a last one ragged or a pair half empty; contexts that end inside a tile of 32 keys
@pytest.mark.parametrize("before,tokens", [(0, 17), (0, 64), (37, 33), (300, 96), (5, 131), (1000, 70)])
@pytest.mark.parametrize("page,window,splits,form", [(16, 0, 1, "plain"), (16, 0, 3, "plain"), (48, 40, 1, "plain"), (16, 0, 2, "capped"), (32, -128, 1, "linear"),
                                                     (16, 100, 1, "both"), (16, 0, 1, "sinks")])
def test_two_heads_a_group(ops, before, tokens, page, window, splits, form):
    nq, nkv, d = 4, 2, 128
    g = torch.Generator().manual_seed(before + tokens + page)
    pages = -(-(before + tokens) // page)
    k_pages = torch.randn(pages, nkv, page, d, generator=g).bfloat16().cuda()
    v_pages = torch.randn(pages, nkv, d, page, generator=g).bfloat16().cuda()
    table = torch.randperm(pages, generator=g).to(torch.int32)[None].cuda()
    q = (torch.randn(tokens, nq * d, generator=g) * 2).bfloat16().cuda()
    of, at = torch.zeros(tokens, dtype=torch.int32).cuda(), torch.arange(before, before + tokens, dtype=torch.int32).cuda()
    more = {}
    if form in ("capped", "both"):
        more["softcap"] = 20.0
    if form == "linear":
        more["distance"] = torch.rand(nq, generator=g).cuda() * 0.1
    if form == "both":
        more["distance"] = torch.rand(2, nq, generator=g).cuda()
    if form == "sinks":
        more["sinks"] = torch.randn(nq, generator=g).cuda()
    want = torch.empty(tokens, nq * d, device="cuda", dtype=torch.bfloat16)
    ops.attention(want, q, k_pages, v_pages, table, of, at, nq, 1 / math.sqrt(d), window, **more)
    starts = list(range(0, tokens, 32))[::-1]
    first, count = (torch.tensor(x, dtype=torch.int32).cuda() for x in (starts, [min(32, tokens - s) for s in starts]))
    for one_request in (False, True):
        got = torch.full_like(want, float("nan"))
        part_o, part_ml = (torch.full((tokens, nq * splits * n), float("nan"), device="cuda") for n in (d, 2))
        ops.attention_prefill(got, q, k_pages, v_pages, table, of, at, first, count, nq, 1 / math.sqrt(d), window, splits=splits, part_o=part_o, part_ml=part_ml,
                              one_request=one_request, **more)
        torch.testing.assert_close(got.float(), want.float(), rtol=2e-2, atol=2e-2)      # weights and results in bfloat16, as the other instances' tests have it
