"""The delta rule's preparation in runs of tokens and its gate in groups of heads: the values that steps of a few tokens make one by one, bit for bit."""

import itertools

import pytest
import torch


def test_short_steps_are_prepared_token_by_token():
    """Runs save launching, which short steps have little of, and lengthen a wave's chain, which they wait for."""
    from llm_runtime_study_amd.kernels import ops

    for tokens, requests, runs in ((8, 1, False), (128, 8, False), (144, 16, False), (320, 64, False), (341, 1, False), (342, 1, True), (500, 100, True),
                                   (2048, 1, True), (2048, 1024, True), (2048, 1025, False)):
        assert ops.delta_in_runs(tokens, requests, 4, 8, 32, 128, 128) == runs, (tokens, requests)
    assert not ops.delta_in_runs(512, 1, 4, 4, 8, 64, 64) and ops.delta_in_runs(1024, 1, 4, 4, 8, 64, 64)
    assert not ops.delta_in_runs(2048, 1, 3, 8, 32, 128, 128) and not ops.delta_in_runs(2048, 1, 4, 8, 32, 130, 128) and not ops.delta_in_runs(2048, 1, 4, 8, 32, 128, 130)


@pytest.mark.gpu
# portions that begin and end inside runs, runs that span two and three requests, a last run that is short, heads below, at and above a wave's lanes;
# enough (token, head) pairs for the gate's groups, not a multiple of them
@pytest.mark.parametrize("heads,groups,d,e,lengths", [(2, 1, 24, 40, (9, 1, 2, 30, 8)), (3, 3, 128, 65, (16,)), (4, 2, 100, 128, (3, 70, 1, 1, 21)), (6, 2, 64, 64, (8, 8, 1)),
                                                      (32, 4, 32, 36, (257, 6)), (31, 1, 128, 17, (300,)), (2, 2, 128, 128, (4097,)),
                                                      (32, 16, 24, 40, (9, 1, 2, 30, 8, 250)), (40, 4, 128, 65, (403,)), (64, 2, 100, 128, (3, 70, 1, 1, 21, 170)),
                                                      (60, 2, 64, 64, (8, 8, 1, 250)), (32, 16, 32, 36, (257, 6)), (62, 1, 128, 17, (300,))])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16)])
def test_runs_and_groups(heads, groups, d, e, lengths, dtype, out_dtype):
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(sum(lengths) + d)
    tokens, requests, taps = sum(lengths), len(lengths), 4
    assert ops.delta_in_runs(tokens, requests, taps, groups, heads, d, e) == (tokens * (2 * groups + heads) >= 16384) and not ops.delta_in_runs(7, 1, taps, groups, heads, d, e)
    channels = 2 * groups * d + heads * e
    proj = torch.randn(tokens, channels + heads * e + 2 * heads + 3, generator=g).to(dtype).cuda()
    conv = torch.randn(channels, taps, generator=g).cuda()
    a_log, dt_bias, norm = torch.randn(heads, generator=g).cuda() - 3, torch.randn(heads, generator=g).cuda(), torch.rand(e, generator=g).cuda()
    begun = (0.3 * torch.randn(requests, ops.delta_state_floats(heads, groups, d, e, taps), generator=g)).cuda()

    def step(rows, state, slots, counts):
        n = len(rows)
        cu = torch.tensor([0] + list(itertools.accumulate(counts)), dtype=torch.int32, device="cuda")
        of = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)).int().cuda()
        made = [torch.empty(n, heads * e, device="cuda", dtype=out_dtype)] + [torch.empty(n, size, device="cuda") for size in (channels, 2 * heads, heads * e)]
        ops.delta_rule(made[0], rows, state, of, cu, torch.tensor(slots, dtype=torch.int32, device="cuda"), len(counts), conv, groups, heads, d, e,
                       a_log, dt_bias, norm, 1e-6, *made[1:])
        return made

    whole_state, state = begun.clone(), begun.clone()
    whole = step(proj, whole_state, list(range(requests)), list(lengths))
    at = 0
    for r, n in enumerate(lengths):
        for first in range(0, n, 7):                             # seven tokens at most: one by one
            count = min(7, n - first)
            for a, b in zip(whole, step(proj[at + first:at + first + count], state, [r], [count])):
                assert torch.equal(a[at + first:at + first + count], b)
        at += n
    assert torch.equal(whole_state, state)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,hidden", [(3, 4), (5, 1023), (2, 1024), (3, 2047), (2, 2048), (4, 4096), (2, 4100), (3, 8192), (2, 8196)])
def test_norm_and_add_of_held_rows(rows, hidden):
    """residual += weight * y / rms(y), and the sum in bfloat16; the mean of squares in float32, hidden / 256 terms a thread and then a tree."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(hidden)
    residual, y, weight = torch.randn(rows, hidden, generator=g), torch.randn(rows, hidden, generator=g), torch.randn(hidden, generator=g)
    want = residual.double() + weight.double() * y.double() * torch.rsqrt(y.double().square().mean(-1, keepdim=True) + 1e-6)
    got, rounded = residual.clone().cuda(), torch.empty(rows, hidden, dtype=torch.bfloat16, device="cuda")
    ops.norm_add(got, y.cuda(), weight.cuda(), 1e-6, rounded=rounded)
    assert ((got.cpu().double() - want).abs() <= (residual.abs() + (want - residual).abs()) * 48 * 2.0 ** -24).all()
    assert torch.equal(rounded, got.bfloat16())
