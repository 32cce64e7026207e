"""The float32 products on the matrix cores, alone: against float64 and, bit for bit, against the kernel for any shape (which a
row stride that is no multiple of four sends them to)."""

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


# every tile of the dispatch: few rows with few and many weight rows, K a multiple of 64 or of 32 only, 16 x 32 to 128 x 128 outputs,
# ragged in both directions; K shorter than the slices that are on their way at once
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
