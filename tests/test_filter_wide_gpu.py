"""Top-k and top-p over the whole chip: bit for bit what the one-kernel form keeps, and a workspace left with zeros where the next call counts."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,stride,offset", [(151936, 151936, 0), (16384, 16384, 0), (16387, 16388, 0), (50257, 50257, 0), (20479, 20480, 1), (20000, 20000, 0),
                                                 (20480, 20480, 0), (20483, 20484, 0)])
def test_keeps_what_the_one_kernel_form_keeps(vocab, stride, offset):
    """Rows whose values spread, crowd into a bin (more than a list holds), tie at the threshold, or are not finite; greedy rows; k and p
    alone, together and off; rows that do not begin on 16 bytes.  Called twice: the second call finds the workspace zero."""
    from llm_runtime_study_amd.kernels import ops

    cases = [(0.8, 50, 1.0), (1.0, 0, 0.9), (0.7, 50, 0.9), (1.0, 1000, 0.95), (1.5, 7, 0.3), (0.0, 50, 0.9), (1.0, 20, 0.9), (1.0, 0, 0.5),
             (0.9, 6000, 1.0), (1.0, vocab, 0.2), (1.0, 1, 1.0), (2.0, 40, 0.8), (1.0, 5, 0.9), (1.0, 0, 1.0), (1.0, 300, 0.99)]
    g = torch.Generator().manual_seed(vocab)
    logits = torch.randn(len(cases), vocab, generator=g) * 3
    logits[6] = 16 + 4 * torch.rand(vocab, generator=g)          # one bin of the first digit holds them all
    logits[7] = -1e-3 * torch.rand(vocab, generator=g) - 1e-4
    logits[9, 17] = 40.0
    logits[11] = torch.randint(-4, 5, (vocab,), generator=g).float()                 # ties by the thousand
    logits[12, 5], logits[13, vocab - 1] = float("nan"), float("inf")
    logits[14, vocab - 3:] = 30.0
    temps, ks = torch.tensor([c[0] for c in cases]).cuda(), torch.tensor([c[1] for c in cases], dtype=torch.int32).cuda()
    ps = torch.tensor([c[2] for c in cases]).cuda()
    space = torch.zeros(len(cases), ops.filter_words(), dtype=torch.int32, device="cuda")
    for top_k, top_p in ((ks, ps), (ks, None), (None, ps), (ks, ps)):
        both = [torch.zeros(len(cases) * stride + 4, device="cuda")[offset:].as_strided((len(cases), vocab), (stride, 1)) for _ in range(2)]
        for work, workspace in zip(both, (None, space)):
            work.copy_(logits)
            ops.filter_logits(work, temps, top_k, top_p, workspace)
        want, got = (w.contiguous().view(torch.int32) for w in both)
        assert torch.equal(torch.isnan(both[0]), torch.isnan(both[1]))
        assert torch.equal(got.masked_fill(torch.isnan(both[1]), 0), want.masked_fill(torch.isnan(both[0]), 0))
        # the words before the list, but the threshold (whose place is the head's fourth): what the next call counts in
        counted = ops.filter_words() - 4096
        assert counted == 16 + 2048
        assert not space[:, :counted].masked_fill(torch.arange(counted, device="cuda") == 3, 0).any()
    assert torch.isinf(both[1]).any()


def test_refuses_a_short_workspace():
    from llm_runtime_study_amd.kernels import ops

    logits, temps = torch.zeros(2, 16384, device="cuda"), torch.ones(2, device="cuda")
    with pytest.raises(Exception, match="workspace"):
        ops.filter_logits(logits, temps, None, torch.full((2,), 0.5, device="cuda"), torch.zeros(1, ops.filter_words(), dtype=torch.int32, device="cuda"))
