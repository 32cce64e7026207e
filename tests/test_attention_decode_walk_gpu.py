"""The decode attention kernel's walk: every number of tiles a wave can be left with, and splits that have no tiles."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("waves,form", [(4, 1), (8, 2)])
@pytest.mark.parametrize("splits,window,page", [(1, 0, 16), (1, 300, 32), (3, 0, 48)])
def test_tiles_left_to_a_wave(waves, form, d, splits, window, page):
    """Contexts that end on either side of 1 to 6 tiles of 32 a wave, with the new key prepared and written by the kernel: against a
    tile at a time, four waves (the same sums in the same order with four waves; with eight the weights' and sums' roundings to
    8 bits differ, 2^-8 of values of order one), and the pages afterwards the same."""
    from llm_runtime_study_amd.kernels import ops

    nq, nkv = 4, 2
    lengths = [1, 33] + [32 * waves * n + extra for n in (1, 2, 3, 5) for extra in (0, 1, 31 * (n % 2) + 32)]
    g = torch.Generator().manual_seed(d + waves + splits)
    tokens, most = len(lengths), -(-max(lengths) // page)
    pages = tokens * most + 1
    k_pages = torch.randn(pages, nkv, page, d, generator=g).bfloat16().cuda()
    v_pages = torch.randn(pages, nkv, d, page, generator=g).bfloat16().cuda()
    table = torch.randperm(pages - 1, generator=g)[:tokens * most].view(tokens, most).int().cuda()
    rows = torch.randn(tokens, (nq + 2 * nkv) * d, generator=g).bfloat16().cuda()
    angle = torch.rand(tokens, d // 2, generator=g) * 6.28
    weight = (1 + 0.3 * torch.randn(d, generator=g)).bfloat16().cuda()
    prepare = ops.DecodePrepare(weight, weight.flip(0).contiguous(), 1e-5, angle.cos().cuda(), angle.sin().cuda(), nkv)
    positions, of = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda(), torch.arange(tokens, dtype=torch.int32).cuda()

    def run(form):
        k, v = k_pages.clone(), v_pages.clone()
        out = torch.full((tokens, nq * d), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.attention_decode(out, rows, k, v, table, of, positions, nq, 1 / math.sqrt(d), window, splits, torch.empty(tokens * nq * splits * d, device="cuda"),
                             torch.empty(tokens * nq * splits * 2, device="cuda"), prepare=prepare, form=form)
        torch.cuda.synchronize()
        return out, k, v

    want, got = run(0), run(form)
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2]) and not torch.equal(want[1], k_pages)
    if form == 1:
        assert torch.equal(got[0], want[0])
    else:
        assert torch.isfinite(got[0]).all()
        torch.testing.assert_close(got[0].float(), want[0].float(), rtol=2 ** -6, atol=2 ** -6)
