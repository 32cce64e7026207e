"""The float32 kernels on the matrix cores, alone: products against float64 and, bit for bit, against the kernel for any shape
(which a row stride that is no multiple of four sends them to); attention against float64, and the same bits however the
queries share workgroups."""

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


def dev(t):
    return t.cuda()


# few rows with few and many weight rows, K a multiple of 64 or of 32 only, tiles of 16 x 32 to 64 x 64 outputs (each of them and 128 x 128
# below), ragged in both directions; K shorter than the slices that are on their way at once
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 33, 100, 300, 1030])
@pytest.mark.parametrize("n,k", [(5, 32), (200, 64), (1027, 96), (2050, 320), (4096, 1024), (16401, 96), (16416, 128)])
def test_float32_product(ops, m, n, k):
    g = torch.Generator().manual_seed(m * 7 + n + k)
    a, w, bias = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g), torch.randn(n, generator=g)
    # a chain of k fused multiply-adds is off by at most k roundings of the sum of the products' sizes; one more for the bias
    want = a.double() @ w.double().T + bias.double()
    bound = (k + 1) * 2.0 ** -24 * (a.abs().double() @ w.abs().double().T + bias.abs().double())
    a, w, bias = dev(a), dev(w), dev(bias)
    out = torch.empty(m, n, device="cuda")
    ops.gemm(out, a, w, bias)
    assert ((out.cpu().double() - want).abs() <= bound).all()
    wide = torch.zeros(m, k + 1, device="cuda")
    wide[:, :k] = a
    plain = torch.empty(m, n, device="cuda")
    ops.gemm(plain, wide[:, :k], w, bias)
    assert torch.equal(out, plain)
    added, strided = torch.full((m, n), 0.25, device="cuda"), torch.full((m, n + 3), 0.25, device="cuda")
    ops.gemm(added, a, w, accumulate=True)
    ops.gemm(strided[:, :n], a, w, accumulate=True)
    ops.gemm(plain, wide[:, :k], w)
    assert torch.equal(added, plain + 0.25) and torch.equal(strided[:, :n], added) and (strided[:, n:] == 0.25).all()


# (cached tokens, new tokens): pieces of 64 keys cut at every place, several requests among 16 neighbouring tokens, more pieces
# than a workgroup has waves
REQUESTS = [(0, 70), (130, 1), (63, 2), (600, 17), (1030, 3), (64, 1)]


@pytest.mark.parametrize("nq,nkv,d,page,window", [(4, 2, 128, 16, 0), (8, 2, 64, 32, 0), (3, 1, 96, 16, 40), (16, 1, 32, 48, 0), (2, 2, 128, 64, 130), (6, 2, 64, 16, -128)])
def test_float32_attention(ops, nq, nkv, d, page, window):
    g = torch.Generator().manual_seed(nq * 31 + d)
    blocks = [-(-(a + b) // page) for a, b in REQUESTS]
    perm = torch.randperm(sum(blocks) + 2, generator=g).tolist()
    # slots that nothing was written to hold what they like
    k_pages, v_pages = torch.full((len(perm), nkv, page, d), float("nan")), torch.full((len(perm), nkv, d, page), float("inf"))
    table = torch.full((len(REQUESTS), max(blocks)), -1, dtype=torch.int32)
    rows, of, at, want = [], [], [], []
    for r, (before, new) in enumerate(REQUESTS):
        k, v, q = (torch.randn(before + new, nkv, d, generator=g) for _ in range(2)), None, torch.randn(new, nq, d, generator=g) * 2
        k, v = k
        for b in range(blocks[r]):
            table[r, b] = perm.pop()
            n = min(page, before + new - b * page)
            k_pages[table[r, b], :, :n] = k[b * page:b * page + n].transpose(0, 1)
            v_pages[table[r, b], :, :, :n] = v[b * page:b * page + n].permute(1, 2, 0)
        for i in range(new):
            pos = before + i
            first = 0 if window == 0 else max(0, pos - window + 1) if window > 0 else pos - pos % -window
            keys, values = (t[first:pos + 1].double().repeat_interleave(nq // nkv, 1) for t in (k, v))
            share = torch.softmax(torch.einsum("khd,hd->hk", keys, q[i].double()) / math.sqrt(d), -1)
            want.append(torch.einsum("hk,khd->hd", share, values).flatten())
        rows.append(q.reshape(new, nq * d))
        of += [r] * new
        at += list(range(before, before + new))
    q, want = torch.cat(rows), torch.stack(want)
    wide = torch.zeros(len(q), nq * d + 8)
    wide[:, :nq * d] = q
    wide, k_pages, v_pages, table, of, at = dev(wide), dev(k_pages), dev(v_pages), dev(table), dev(torch.tensor(of, dtype=torch.int32)), dev(torch.tensor(at, dtype=torch.int32))
    results = []
    for together in (16, 1, 5):
        out = torch.empty(len(q), nq * d, device="cuda")
        ops.attention(out, wide, k_pages, v_pages, table, of, at, nq, 1 / math.sqrt(d), window, together=together)
        results.append(out)
    # scores of size s are off by at most (d + 2) 2^-24 |q||k| scale (here below 2e-5), weights by as much in proportion, sums likewise
    torch.testing.assert_close(results[0].cpu().double(), want, rtol=2e-5, atol=2e-5)
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])


def test_float32_attention_keeps_odd_values_to_those_who_see_them(ops):
    """An infinite value and a NaN in a prompt: tokens before them give what they give without them, those behind see them."""
    g = torch.Generator().manual_seed(3)
    n, d = 90, 64
    q, k, v = (torch.randn(n, d, generator=g) for _ in range(3))
    pages, table, of, at = -(-n // 16), torch.arange(-(-n // 16), dtype=torch.int32)[None], torch.zeros(n, dtype=torch.int32), torch.arange(n, dtype=torch.int32)

    def run(v):
        k_pages, v_pages = torch.zeros(pages * 16, d), torch.zeros(pages * 16, d)
        k_pages[:n], v_pages[:n] = k, v
        out = torch.empty(n, d, device="cuda")
        ops.attention(out, dev(q), dev(k_pages.view(pages, 1, 16, d)), dev(v_pages.view(pages, 1, 16, d).transpose(2, 3).contiguous()), dev(table), dev(of), dev(at),
                      1, 0.125, together=16)
        return out.cpu()

    plain, odd = run(v), v.clone()
    odd[50, 7], odd[71, 9], odd[73, 8] = float("inf"), float("nan"), float("-inf")
    got = run(odd)
    expected = plain.clone()
    expected[50:, 7], expected[71:, 9], expected[73:, 8] = float("inf"), float("nan"), float("-inf")
    assert torch.equal(got.nan_to_num(nan=12345.0), expected.nan_to_num(nan=12345.0))


def test_float32_attention_gives_a_score_of_minus_infinity_no_weight(ops):
    """Keys whose scores overflow to minus infinity, alone in their piece of 64 and among others: as if they were not there."""
    g = torch.Generator().manual_seed(4)
    n, d = 200, 64
    q, k, v = (torch.randn(n, d, generator=g) for _ in range(3))
    q[:, 0], k[:, 0] = 1e20, 0.0
    k[5, 0] = k[64:130, 0] = k[199, 0] = -1e20
    pages, table, of, at = -(-n // 16), torch.arange(-(-n // 16), dtype=torch.int32)[None], torch.zeros(n, dtype=torch.int32), torch.arange(n, dtype=torch.int32)
    k_pages, v_pages = torch.zeros(pages * 16, d), torch.zeros(pages * 16, d)
    k_pages[:n], v_pages[:n] = k, v
    out = torch.empty(n, d, device="cuda")
    ops.attention(out, dev(q), dev(k_pages.view(pages, 1, 16, d)), dev(v_pages.view(pages, 1, 16, d).transpose(2, 3).contiguous()), dev(table), dev(of), dev(at), 1, 0.125, together=16)
    scores = (q[:, 1:].double() @ k[:, 1:].double().T) * 0.125
    scores[:, k[:, 0] < 0] = -math.inf
    scores[torch.ones(n, n, dtype=torch.bool).triu(1)] = -math.inf
    torch.testing.assert_close(out.cpu().double(), torch.softmax(scores, -1) @ v.double(), rtol=2e-5, atol=2e-5)


@pytest.mark.parametrize("nq,nkv,d,batch", [(32, 32, 128, 40), (8, 8, 128, 70), (32, 8, 64, 70), (6, 2, 96, 200), (16, 16, 32, 80), (4, 4, 64, 300), (16, 1, 128, 300)])
@pytest.mark.parametrize("window", [0, 20])
def test_float32_attention_over_short_contexts(ops, nq, nkv, d, batch, window):
    """Steps that workgroups of one and two waves take, and those that leave blocks out: the bits of eight waves, whatever is told."""
    g = torch.Generator().manual_seed(nq + d + batch)
    page, per = 16, 16
    lengths = [(i * 37) % 256 + 1 for i in range(batch)]
    pages = torch.randn(batch * per, nkv, page, d, generator=g).cuda(), torch.randn(batch * per, nkv, d, page, generator=g).cuda()
    table = torch.arange(batch * per, dtype=torch.int32).view(batch, per).cuda()
    q = torch.randn(batch, nq * d, generator=g).cuda()
    of = torch.arange(batch, dtype=torch.int32)
    for most in (256, 32):
        at = torch.tensor([min(n, most) - 1 for n in lengths], dtype=torch.int32).cuda()
        outs = [torch.empty(batch, nq * d, device="cuda") for _ in range(4)]
        for out, (longest, together) in zip(outs, ((0, 1), (most, 1), (most, 16), (most, 3))):
            ops.attention(out, q, *pages, table, of.cuda(), at, nq, 1 / math.sqrt(d), window, together=together, longest=longest)
        assert all(torch.equal(out, outs[0]) for out in outs[1:])


@pytest.mark.parametrize("nq,nkv,d,page", [(4, 2, 128, 16), (8, 2, 64, 48), (3, 1, 96, 16), (16, 1, 32, 32)])
@pytest.mark.parametrize("window", [0, 70])
def test_float32_attention_of_keys_straight_into_registers(ops, nq, nkv, d, page, window):
    """Keys and values through LDS and straight into registers: the same bits, infinities and NaN among the values, whichever the told length chooses."""
    g = torch.Generator().manual_seed(nq + d)
    for batch, most, together in ((5, 128, 1), (5, 190, 1), (5, 100, 3), (200, 250, 1), (240 // nkv, 900, 1)):
        if not ops.attention_f32_direct(batch * nkv, together, most):
            assert together == 1 and ops.compute_units() != 256
            continue
        per = -(-most // page)
        pages = torch.randn(batch * per, nkv, page, d, generator=g), torch.randn(batch * per, nkv, d, page, generator=g)
        for at, value in ((3, math.inf), (5, -math.inf), (7, math.nan)):
            pages[1][:, :, at, at] = torch.where(torch.rand(batch * per, nkv, generator=g) < 0.03, value, 1.0)
        pages = [p.cuda() for p in pages]
        table = torch.randperm(batch * per, generator=g).to(torch.int32).view(batch, per).cuda()
        q = torch.randn(batch, nq * d, generator=g).cuda()
        of = (torch.arange(batch, dtype=torch.int32) // together).cuda()
        at = torch.randint(0, most, (batch,), generator=g).to(torch.int32).cuda()
        outs = [torch.empty(batch, nq * d, device="cuda") for _ in range(2)]
        for out, longest in zip(outs, (0, most)):
            ops.attention(out, q, *pages, table, of, at, nq, 1 / math.sqrt(d), window, together=together, longest=longest)
        assert torch.equal(*(out.view(torch.int32) for out in outs))


def test_float32_product_of_rows_far_apart(ops):
    """Rows whose distance, times the rows of a tile, does not fit 32 bits of bytes."""
    m, n, k, stride = 16, 40, 64, 72_000_000
    g = torch.Generator().manual_seed(9)
    a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g)
    wide = torch.empty(m, stride, device="cuda")
    wide[:, :k] = a.cuda()
    far, near = torch.empty(m, n, device="cuda"), torch.empty(m, n, device="cuda")
    ops.gemm(far, wide[:, :k], w.cuda())
    ops.gemm(near, a.cuda(), w.cuda())
    assert torch.equal(far, near)


@pytest.mark.parametrize("m,n,tile", [(33, 1027, (16, 32)), (2047, 5, (16, 32)), (100, 2050, (64, 32)), (509, 4099, (64, 32)), (2047, 200, (64, 32)), (100, 4099, (64, 64)),
                                      (1500, 1027, (64, 64)), (100, 24577, (128, 128)), (509, 6145, (128, 128)), (1500, 2050, (128, 128)), (2049, 16416, (128, 128))])
@pytest.mark.parametrize("k", [32, 64, 96, 416])
def test_float32_product_of_every_tile(ops, m, n, tile, k):
    """Remainders in both directions, K shorter than, as long as and longer than the slices on their way, strided stores and sums: against
    float64, and bit for bit against the kernel for any shape."""
    assert ops.gemm_f32_tile(m, n) == tile
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, bias = (torch.randn(*shape, generator=g, device="cuda") for shape in ((m, k), (n, k), (n,)))
    # k roundings of the sum of the products' sizes, one for the bias
    want = a.double() @ w.double().T + bias.double()
    bound = (k + 1) * 2.0 ** -24 * (a.abs().double() @ w.abs().double().T + bias.abs().double())
    out, plain, strided = torch.empty(m, n, device="cuda"), torch.empty(m, n, device="cuda"), torch.full((m, n + 3), 0.25, device="cuda")
    ops.gemm(out, a, w, bias)
    assert ((out.double() - want).abs() <= bound).all()
    wide = torch.zeros(m, k + 1, device="cuda")
    wide[:, :k] = a
    ops.gemm(plain, wide[:, :k], w, bias)
    assert torch.equal(out, plain)
    ops.gemm(strided[:, :n], a, w, accumulate=True)
    ops.gemm(plain, wide[:, :k], w)
    assert torch.equal(strided[:, :n], plain + 0.25) and (strided[:, n:] == 0.25).all()
