"""The decode attention kernel's walk: every number of tiles a wave can be left with, and splits that have no tiles."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("waves,form", [(4, 1), (8, 2), (4, 3)])
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
    if form in (1, 3):
        assert torch.equal(got[0], want[0])
    else:
        assert torch.isfinite(got[0]).all()
        torch.testing.assert_close(got[0].float(), want[0].float(), rtol=2 ** -6, atol=2 ** -6)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("waves,form", [(4, 0), (4, 1), (8, 2), (4, 3)])
@pytest.mark.parametrize("splits,window,page", [(1, 0, 16), (1, 300, 32), (3, 0, 48), (2, 70, 16)])
def test_walk_against_64_bits(waves, form, d, splits, window, page):
    """Every form of the kernel with the norm, the rotation, the new key's way into its page and the softmax worked out on the host in
    64 bits.  Weights are rounded to 8 bits for their product with the values (2^-8 of the sum of weights times magnitudes), queries and
    new keys too, whose last place may fall otherwise after sums in 32 bits (as much again in the weights), and the result once more."""
    from llm_runtime_study_amd.kernels import ops

    nq, nkv = 4, 2
    lengths = [1, 2, 32, 33] + [32 * waves * n + extra for n in (1, 2, 3) for extra in (0, 1, 31)]
    g = torch.Generator().manual_seed(d + waves + splits + window)
    tokens, most = len(lengths), -(-max(lengths) // page)
    pages = tokens * most + 1
    k_pages = torch.randn(pages, nkv, page, d, generator=g).bfloat16()
    v_pages = torch.randn(pages, nkv, d, page, generator=g).bfloat16()
    table = torch.randperm(pages - 1, generator=g)[:tokens * most].view(tokens, most).int()
    rows = torch.randn(tokens, (nq + 2 * nkv) * d, generator=g).bfloat16()
    angle = torch.rand(tokens, d // 2, generator=g) * 6.28
    cos, sin = angle.cos(), angle.sin()
    q_weight, k_weight = ((1 + 0.3 * torch.randn(d, generator=g)).bfloat16() for _ in range(2))
    k, v, out = k_pages.cuda(), v_pages.cuda(), torch.full((tokens, nq * d), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.attention_decode(out, rows.cuda(), k, v, table.cuda(), torch.arange(tokens, dtype=torch.int32).cuda(), torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda(),
                         nq, 1 / math.sqrt(d), window, splits, torch.empty(tokens * nq * splits * d, device="cuda"), torch.empty(tokens * nq * splits * 2, device="cuda"),
                         prepare=ops.DecodePrepare(q_weight.cuda(), k_weight.cuda(), 1e-5, cos.cuda(), sin.cuda(), nkv), form=form)
    torch.cuda.synchronize()

    def prepared(heads, weight, t):                              # [n, d] raw rows of token t's heads, as the pages hold them
        x = heads.double()
        x = x / (x.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * weight.double()
        a, b, c, s = x[:, :d // 2], x[:, d // 2:], cos[t].double(), sin[t].double()
        return torch.cat((a * c - b * s, b * c + a * s), -1).bfloat16()

    k_want, v_want = k_pages.clone(), v_pages.clone()
    for t, n in enumerate(lengths):
        raw = rows[t].view(-1, d)
        q, new_k, new_v = prepared(raw[:nq], q_weight, t), prepared(raw[nq:nq + nkv], k_weight, t), raw[nq + nkv:]
        at, place = int(table[t, (n - 1) // page]), (n - 1) % page
        k_want[at, :, place], v_want[at, :, :, place] = new_k, new_v
        own = table[t, :-(-n // page)].long()
        keys = k_want[own].permute(1, 0, 2, 3).reshape(nkv, -1, d)[:, :n].double()
        values = v_want[own].permute(1, 0, 3, 2).reshape(nkv, -1, d)[:, :n].double()
        first = max(0, n - window) if window else 0
        for head in range(nq):
            of = head // (nq // nkv)
            share = torch.softmax(keys[of, first:] @ q[head].double() / math.sqrt(d), 0)
            want, size = share @ values[of, first:], share @ values[of, first:].abs()
            got = out[t, head * d:(head + 1) * d].cpu().double()
            assert ((got - want).abs() <= 2.0 ** -7 * size + 2.0 ** -8 * want.abs()).all(), (t, n, head)
    # nothing but the new keys and values was written, and those as worked out (keys to the last place)
    assert torch.equal(v.cpu(), v_want)
    changed = (k.cpu() != k_pages).any(-1)
    assert not (changed & ~(k_want != k_pages).any(-1)).any()
    assert ((k.cpu().double() - k_want.double()).abs() <= 2.0 ** -7 * k_want.double().abs()).all()


@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("nq,nkv,d,page,window", [(1, 1, 64, 16, 0), (15, 1, 128, 32, 0), (16, 1, 128, 48, 0), (32, 2, 64, 16, 40), (12, 4, 128, 16, 0)])
def test_new_key_behind_any_number_of_heads(nq, nkv, d, page, window, form):
    """The new key is prepared in the column behind a kv group's heads, after them where 16 leave none: pages and results against heads
    and key prepared by qk_prep (the same norm and rotation but for the order of a sum: a last place of bfloat16)."""
    from llm_runtime_study_amd.kernels import ops

    lengths, splits = [1, 16, 17, 33, 255, 256, 300], 2
    g = torch.Generator().manual_seed(nq + d)
    tokens, most = len(lengths), -(-max(lengths) // page)
    k_pages = torch.randn(tokens * most, nkv, page, d, generator=g).bfloat16().cuda()
    v_pages = torch.randn(tokens * most, nkv, d, page, generator=g).bfloat16().cuda()
    table = torch.randperm(tokens * most, generator=g).view(tokens, most).int().cuda()
    raw = torch.randn(tokens, (nq + 2 * nkv) * d, generator=g).bfloat16().cuda()
    angle = torch.rand(tokens, d // 2, generator=g) * 6.28
    cos, sin = angle.cos().cuda(), angle.sin().cuda()
    q_weight, k_weight = ((1 + 0.3 * torch.randn(d, generator=g)).bfloat16().cuda() for _ in range(2))
    last = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    slots = (table[torch.arange(tokens).cuda(), (last // page).long()] * page + last % page).int()

    def run(fused):
        k, v, rows, out = k_pages.clone(), v_pages.clone(), raw.clone(), torch.full((tokens, nq * d), float("nan"), dtype=torch.bfloat16, device="cuda")
        if not fused:
            ops.qk_prep(rows, nq, nkv, d, q_weight, k_weight, 1e-5, cos, sin, k, v, slots, page)
        ops.attention_decode(out, rows, k, v, table, torch.arange(tokens, dtype=torch.int32).cuda(), last, nq, 1 / math.sqrt(d), window, splits,
                             torch.empty(tokens * nq * splits * d, device="cuda"), torch.empty(tokens * nq * splits * 2, device="cuda"),
                             prepare=ops.DecodePrepare(q_weight, k_weight, 1e-5, cos, sin, nkv) if fused else None, form=form)
        torch.cuda.synchronize()
        return out.float(), k.float(), v

    got, want = run(True), run(False)
    assert torch.equal(got[2], want[2]) and not torch.equal(want[1], k_pages.float())
    torch.testing.assert_close(got[1], want[1], rtol=2 ** -7, atol=1e-6)
    torch.testing.assert_close(got[0], want[0], rtol=2 ** -6, atol=2 ** -6)
