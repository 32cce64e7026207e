"""Float32 products whose sums over K are made in runs: every tile, with runs that end inside K, beside it and past it, gives the sums of the kernel for
any shape, and these are as close to 64 bits as chains of a run are."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 40, 130, 509])
@pytest.mark.parametrize("n,k", [(1024, 3072), (1000, 1088), (1024, 576), (2048, 192), (4100, 1024), (16400, 640), (1030, 2080)])
def test_sums_in_runs(m, n, k):
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")
    out, added = torch.empty(m, n, device="cuda"), torch.randn(m, n, generator=g, device="cuda")
    before = added.clone()
    ops.gemm(out, a, w)
    ops.gemm(added, a, w, accumulate=True)
    # a run's chain is off by at most its length in roundings of the sum of the products' sizes, adding four up by four more
    run = -(-(-(-k // 128)) // 4) * 128
    assert ((out - a.double() @ w.double().T).abs() <= (run + 4) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)).all()
    assert torch.equal(added, before + out)
    wide, plain = torch.zeros(m, k + 1, device="cuda"), torch.empty(m, n, device="cuda")
    wide[:, :k] = a
    ops.gemm(plain, wide[:, :k], w)
    assert torch.equal(out, plain)
    first = torch.empty(1, n, device="cuda")
    ops.gemm(first, a[:1], w)
    assert torch.equal(first, out[:1])


# the last five: on either side of 24 x 16,384 outputs, where workgroups of 64 weight rows share the input rows
@pytest.mark.parametrize("m,n,k", [(m, n, k) for m in (1, 9, 17, 100, 509) for n, k in ((16, 32), (48, 64), (6144, 1024), (1040, 96), (2064, 640))]
                         + [(16, 24592, 64), (16, 24560, 192), (8, 49168, 640), (15, 26224, 96), (1, 393232, 64)])
def test_gated_product(m, n, k):
    """The activation in the product's epilogue: the bits of the product and the activation's own kernel."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")
    both, want, got = torch.empty(m, n, device="cuda"), torch.empty(m, n // 2, device="cuda"), torch.full((m + 1, n // 2 + 4), 7.0, device="cuda")
    ops.gemm(both, a, w)
    ops.silu_mul(want, both, interleaved=True)
    ops.gemm_f32_gated(got[:m, :n // 2], a, w)
    assert torch.equal(got[:m, :n // 2], want) and (got[m:] == 7).all() and (got[:, n // 2:] == 7).all()
