"""Few-rows products that finish a norm: any number of parts of its sum of squares, rows and walks over K."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# (K of 896, 1,152, 1,920 and 2,880, of 416 in the widest: the last of a workgroup's waves walks less than the others and takes another way)
@pytest.mark.parametrize("n,k,swiglu", [(256, 512, False), (2048, 1536, True), (6144, 1024, False), (16416, 768, False), (272, 96, False),
                                        (256, 896, False), (2048, 1152, True), (272, 1920, False), (256, 2880, False), (6144, 896, False), (16416, 416, False)])
@pytest.mark.parametrize("m,parts", [(1, 1), (3, 31), (16, 33), (9, 320), (16, 321), (2, 700)])
def test_sums_of_squares_in_any_number_of_parts(m, parts, n, k, swiglu):
    """Against 64 bits: the factor is right to 2^-20 whatever the parts (sums of 32 bits over at most 700), a product of K bfloat16 pairs
    to 2^-20 of the sum of its terms' magnitudes, and the result is rounded to bfloat16 (2^-8; the gated activation twice)."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(n + parts + m)
    x, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16()
    sumsq = torch.rand(parts, m, generator=g) * 2 * k / parts
    out = torch.full((m, n // 2 if swiglu else n), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.gemm_norm_chain(out, x.cuda(), w.cuda(), swiglu=swiglu, in_sumsq=sumsq.cuda(), in_eps=1e-6)
    factor = 1.0 / (sumsq.double().sum(0) / k + 1e-6).sqrt()
    want = x.double() @ w.double().T * factor[:, None]
    if swiglu:
        pairs = want.view(m, n // 16, 2, 8)
        gate, up = pairs[:, :, 0].reshape(m, -1), pairs[:, :, 1].reshape(m, -1)
        want = gate * torch.sigmoid(gate) * up
    torch.testing.assert_close(out.cpu().double(), want, rtol=2 ** -8 + 2 ** -18, atol=2 ** -14)


@pytest.mark.parametrize("m,n,k,weight_dtype", [(1, 1024, 2048, torch.bfloat16), (16, 1024, 3072, torch.float32), (5, 512, 512, torch.bfloat16), (8, 40, 256, torch.float32)])
def test_product_that_begins_the_next_norm(m, n, k, weight_dtype):
    """The residual stream, the weighted row and the sums of squares that a product leaves, against 64 bits of the same values."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(n + k + m)
    x, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16()
    h, weight = torch.randn(m, n, generator=g), (1 + 0.3 * torch.randn(n, generator=g)).to(weight_dtype)
    stream, next_x = h.cuda(), torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    sums = torch.full((ops.norm_chain_parts(n), m), float("nan"), device="cuda")
    ops.gemm_norm_chain(stream, x.cuda(), w.cuda(), accumulate=True, next_x=next_x, next_sumsq=sums, next_weight=weight.cuda())
    want = h.double() + x.double() @ w.double().T
    torch.testing.assert_close(stream.cpu().double(), want, rtol=2 ** -18, atol=2 ** -16)
    torch.testing.assert_close(next_x.cpu().double(), want * weight.double(), rtol=2 ** -8, atol=2 ** -14)
    torch.testing.assert_close(sums.cpu().double().sum(0), want.pow(2).sum(1), rtol=2 ** -16, atol=0.0)


@pytest.mark.parametrize("hidden", [4, 252, 256, 260, 600, 1020, 1024, 1028, 2052, 4096, 4100, 6148, 8192])
@pytest.mark.parametrize("weight_dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
def test_norms_of_rows_of_any_length(hidden, weight_dtype, out_dtype):
    """Rows that end inside, at and behind the last chunk a thread owns: plain, gathered, and with a product's output added first (which
    the stream keeps).  Against 64 bits: a sum of `hidden` squares in 32 bits, then the output's own rounding."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(hidden)
    x, y = torch.randn(7, hidden, generator=g) * 3, torch.randn(7, hidden, generator=g).bfloat16()
    weight, rows = (1 + 0.3 * torch.randn(hidden, generator=g)).to(weight_dtype), torch.tensor([6, 0, 0, 3], dtype=torch.int32)
    near = dict(rtol=2 ** -8 if out_dtype == torch.bfloat16 else 2 ** -18, atol=2 ** -20)

    def normed(v):
        return v / (v.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * weight.double()

    stream, out = x.cuda(), torch.full((7, hidden), float("nan"), dtype=out_dtype, device="cuda")
    ops.rmsnorm(out, stream, weight.cuda(), 1e-6)
    torch.testing.assert_close(out.cpu().double(), normed(x.double()), **near)
    assert torch.equal(stream.cpu(), x)
    gathered = torch.full((4, hidden), float("nan"), dtype=out_dtype, device="cuda")
    ops.rmsnorm(gathered, stream, weight.cuda(), 1e-6, rows=rows.cuda())
    assert torch.equal(gathered, out[rows.long().cuda()])
    ops.add_rmsnorm(out, stream, y.cuda(), weight.cuda(), 1e-6)
    assert torch.equal(stream.cpu(), x + y.float())
    torch.testing.assert_close(out.cpu().double(), normed((x + y.float()).double()), **near)


@pytest.mark.parametrize("k", [256, 512, 768, 1280, 2304])
@pytest.mark.parametrize("m,splits,waves", [(17, 1, 4), (33, 2, 8), (64, 4, 4), (64, 8, 6), (100, 3, 5), (128, 16, 8)])
def test_slices_left_to_a_workgroup_of_17_to_128_rows(m, splits, waves, k):
    """K splits whose workgroups have no slice of 256, one, and a few: against 64 bits (sums of 32 bits, then the output's rounding)."""
    from llm_runtime_study_amd.kernels import ops

    n = 96
    g = torch.Generator().manual_seed(m + k)
    x, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16()
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.gemm(out, x.cuda(), w.cuda(), choice=ops.KernelChoice(mid_splits=splits, mid_waves=waves))
    torch.testing.assert_close(out.cpu().double(), x.double() @ w.double().T, rtol=2 ** -8, atol=2 ** -14)
    parts = 11
    sumsq = torch.rand(parts, m, generator=g) * 2 * k / parts
    if splits == 1:
        ops.gemm_mid_scaled(out, x.cuda(), w.cuda(), sumsq.cuda(), 1e-6, choice=ops.KernelChoice(mid_splits=splits, mid_waves=waves))
        want = x.double() @ w.double().T / (sumsq.double().sum(0) / k + 1e-6).sqrt()[:, None]
        torch.testing.assert_close(out.cpu().double(), want, rtol=2 ** -8 + 2 ** -18, atol=2 ** -14)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,hidden,offset", [(1, 8, 0), (3, 100, 0), (33, 1032, 0), (257, 16, 0), (5, 64, 4)])
def test_rows_of_the_embedding(tokens, hidden, offset, dtype):
    """Rows of whole and broken pieces of eight values, and a table that does not begin on 32 bytes: the table's rows times a factor."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(hidden)
    table = torch.randn(50 * hidden + offset, generator=g).to(dtype).cuda()[offset:].view(50, hidden)
    ids = torch.randint(0, 50, (tokens,), generator=g, dtype=torch.int32).cuda()
    out = torch.full((tokens, hidden), float("nan"), device="cuda")
    ops.embed(out, table, ids, 1.5)
    assert torch.equal(out, table[ids.long()].float() * 1.5)
