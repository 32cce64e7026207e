"""The vendor library's handle and workspace: every runner's products use one of its own, since the library's kernels leave sums and
flags in the workspace and products of two engines may run at the same time."""

from types import SimpleNamespace

import pytest
import torch

from llm_runtime_study_amd.engine import step
from llm_runtime_study_amd.kernels import ops
from llm_runtime_study_amd.parts import linear as linear_part


def test_products_of_two_runners_use_states_of_their_own(monkeypatch):
    used = []
    monkeypatch.setattr(ops, "LibraryState", lambda: SimpleNamespace(address=object()))
    monkeypatch.setattr(ops, "library_gemm", lambda out, a, w, state=None: used.append(state))
    monkeypatch.setattr(ops, "silu_mul", lambda *a, **k: None)
    monkeypatch.setattr(ops, "add_into", lambda *a, **k: None)
    monkeypatch.setattr(linear_part, "plan", lambda *a, **k: ("library", ""))
    x, w = torch.zeros(300, 64, dtype=torch.bfloat16), torch.zeros(128, 64, dtype=torch.bfloat16)
    for arena in (step.ScratchArena("cpu"), step.ScratchArena("cpu")):
        ctx = step.StepContext.__new__(step.StepContext)
        ctx._runner, ctx.memo, ctx.dtype, ctx.kernels = SimpleNamespace(arena=arena), {}, torch.bfloat16, ops.DEFAULT_CHOICE
        linear_part.linear(ctx, torch.zeros(300, 128, dtype=torch.bfloat16), x, w)
        linear_part.linear(ctx, torch.zeros(300, 64, dtype=torch.bfloat16), x, w, swiglu=True)
        linear_part.linear(ctx, torch.zeros(300, 128), x, w, accumulate=True)
    assert None not in used and len(used) == 6
    assert used[0] is used[1] is used[2] and used[3] is used[4] is used[5] and used[0] is not used[3]


@pytest.mark.gpu
def test_states_are_given_back_and_taken_again():
    first, second = ops.LibraryState(), ops.LibraryState()
    addresses = {first.address, second.address}
    assert len(addresses) == 2
    del first, second
    again = ops.LibraryState()
    assert again.address in addresses and ops.LibraryState().address != again.address


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(509, 1024, 3072), (512, 2560, 9728), (300, 4096, 4096)])
def test_products_on_two_streams_at_once(m, n, k):
    g = torch.Generator().manual_seed(m)
    a = [torch.randn(m, k, generator=g).bfloat16().cuda() for _ in range(2)]
    w = torch.randn(n, k, generator=g).bfloat16().cuda()
    states, streams = [ops.LibraryState() for _ in range(2)], [torch.cuda.Stream() for _ in range(2)]
    alone = [torch.empty(m, n, device="cuda") for _ in range(2)]
    for i in range(2):
        ops.library_gemm(alone[i], a[i], w, state=states[i])
    outs = [[torch.empty(m, n, device="cuda") for _ in range(20)] for _ in range(2)]
    torch.cuda.synchronize()
    for turn in range(20):
        for i in range(2):
            with torch.cuda.stream(streams[i]):
                ops.library_gemm(outs[i][turn], a[i], w, state=states[i])
    torch.cuda.synchronize()
    # the same kernel over the same operands: where it divides K, it adds the parts' sums in a fixed order
    assert all(torch.equal(out, alone[i]) for i in range(2) for out in outs[i])
