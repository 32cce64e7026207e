"""Products of many bfloat16 rows with at most 64 weight rows: remainders of rows, outputs and K, strides, and what is done
with the sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(65, 4, 32), (17, 16, 256), (128, 64, 4096), (129, 12, 96), (100, 16, 64), (300, 20, 1056), (257, 36, 2016), (511, 64, 544), (2048, 32, 4096), (9000, 60, 160),
                                   (4095, 40, 512), (4096, 36, 4096), (4097, 8, 576), (5000, 64, 512), (6001, 4, 4096)])
def test_few_outputs_of_many_rows(m, n, k):
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=g).to(torch.bfloat16).cuda()[:, :k]
    w = torch.randn(n, k, generator=g).to(torch.bfloat16).cuda()
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    bound = k * 2.0 ** -23 * size                  # float32 sums of k exact products, whatever their order
    wide = torch.full((m + 1, n + 4), -7.0, device="cuda")
    ops.gemm(wide[:m, :n], x, w)
    assert ((wide[:m, :n].double() - want).abs() <= bound).all()
    assert (wide[m] == -7.0).all() and (wide[:, n:] == -7.0).all()
    added = torch.ones(m, n, device="cuda")
    ops.gemm(added, x, w, accumulate=True)
    assert ((added.double() - 1.0 - want).abs() <= bound + 2.0 ** -23 * (1.0 + want.abs())).all()
    short = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ops.gemm(short, x, w)
    assert ((short.double() - want).abs() <= bound + 2.0 ** -8 * (want.abs() + bound)).all()


@pytest.mark.parametrize("m,n,k", [(65, 4, 32), (70, 64, 224), (129, 12, 96), (100, 16, 64), (300, 20, 1056), (257, 36, 2016), (2048, 32, 4096), (2048, 64, 2048), (1000, 8, 544),
                                   (4095, 16, 4096), (4096, 16, 2048), (4096, 64, 4096), (4097, 4, 1024), (6000, 32, 8192), (5003, 8, 4160), (5003, 8, 28672), (16400, 12, 8192)])
def test_few_outputs_have_the_bits_of_many(m, n, k):
    """A row's outputs are the same whether its weight rows stand alone or among more than one such kernel takes."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).to(torch.bfloat16).cuda(), torch.randn(128, k, generator=g).to(torch.bfloat16).cuda()
    few, many = torch.empty(m, n, device="cuda"), torch.empty(m, 128, device="cuda")
    ops.gemm(few, x, w[:n])
    ops.gemm(many, x, w)
    assert torch.equal(few, many[:, :n])
