"""Float32 attention with the pieces of a row's keys divided between workgroups: the bits of the undivided kernel, which is tested against
float64, whatever the division."""

import math

import pytest
import torch

from llm_runtime_study_amd.parts.attention import GQAAttention


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from llm_runtime_study_amd.kernels import ops

    return ops


# positions: ends of pieces of 64, of eight merged at a time, one piece and many
POSITIONS = [0, 63, 64, 511, 512, 700, 1100]


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nkv,d,page", [(4, 2, 128, 16), (8, 2, 64, 32), (3, 1, 128, 48), (2, 2, 64, 16)])
@pytest.mark.parametrize("window", [0, 130, -200])
@pytest.mark.parametrize("splits", [1, 2, 5, 64])
def test_bits(ops, nq, nkv, d, page, window, splits):
    g = torch.Generator().manual_seed(nq + d)
    n, per = len(POSITIONS), -(-(max(POSITIONS) + 1) // page)
    pages = torch.randn(n * per, nkv, page, d, generator=g), torch.randn(n * per, nkv, d, page, generator=g)
    pages[1][:, :, 3, 5] = torch.where(torch.rand(n * per, nkv, generator=g) < 0.1, math.inf, 1.0)
    pages = [p.cuda() for p in pages]
    table = torch.randperm(n * per, generator=g).to(torch.int32).view(n, per).cuda()
    q = torch.randn(n, (nq + 2 * nkv) * d, generator=g).cuda()
    of, at = torch.arange(n, dtype=torch.int32).flip(0).contiguous().cuda(), torch.tensor(POSITIONS, dtype=torch.int32).cuda()
    want = torch.empty(n, nq * d, device="cuda")
    ops.attention(want, q, *pages, table, of, at, nq, 1 / math.sqrt(d), window)
    for slots in (18, 40):
        out, part_o, part_ml = torch.empty_like(want), torch.full((n * nq * slots, d), math.nan, device="cuda"), torch.full((n * nq * slots, 2), math.nan, device="cuda")
        ops.attention_f32_divided(out, q, *pages, table, of, at, nq, 1 / math.sqrt(d), window, splits, slots, part_o, part_ml)
        assert torch.equal(out.view(torch.int32), want.view(torch.int32))
    with pytest.raises(Exception, match="too small"):
        ops.attention_f32_divided(out, q, *pages, table, of, at, nq, 1 / math.sqrt(d), window, splits, 41, part_o, part_ml)


def test_rule(monkeypatch):
    """No division of short contexts or of steps that fill the chip; never more parts than pieces."""
    from llm_runtime_study_amd.kernels import ops

    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    for workgroups in (1, 8, 64, 96, 128, 129, 512):
        for longest in (1, 255, 256, 511, 512, 2000, 40000):
            splits = GQAAttention._piece_splits(workgroups, longest)
            assert splits >= 1 and (splits == 1 or (longest >= 256 and workgroups <= 128 and splits * 32 <= longest))
