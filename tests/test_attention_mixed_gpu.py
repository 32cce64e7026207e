"""A mixed step's attention in one launch: the single tokens at its head and the prompt portions behind them give, bit for bit, what the
two kernels give in launches of their own."""

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


# (tokens before, tokens in the step): single tokens first, then one or two portions; contexts that end at every place of a tile
STEPS = {"one": [(0, 1), (31, 1), (500, 1), (97, 70)], "two": [(1300, 1), (0, 40), (64, 33)], "many": [(40 + 13 * i, 1) for i in range(40)] + [(512, 200)]}


@pytest.mark.parametrize("step", sorted(STEPS))
@pytest.mark.parametrize("nq,nkv,page,window,size,prepared", [(8, 2, 16, 0, 16, True), (8, 2, 16, 0, 32, False), (4, 2, 16, 0, 32, True), (4, 2, 48, 60, 16, True), (10, 2, 16, -128, 32, True),
                                                             (16, 1, 32, 0, 16, False)])
def test_one_launch(ops, step, nq, nkv, page, window, size, prepared):
    d, requests = 128, STEPS[step]
    g = torch.Generator().manual_seed(nq + page + len(requests))
    blocks = [-(-(a + b) // page) for a, b in requests]
    perm = torch.randperm(sum(blocks), generator=g).tolist()
    table, of, at, groups = torch.full((len(requests), max(blocks)), -1, dtype=torch.int32), [], [], []
    singles = sum(b == 1 for _, b in requests)
    for r, (before, new) in enumerate(requests):
        table[r, :blocks[r]] = torch.tensor([perm.pop() for _ in range(blocks[r])])
        if new > 1:
            groups += [(before + i, len(of) + i - singles, min(size, new - i)) for i in range(0, new, size)]
        of += [r] * new
        at += list(range(before, before + new))
    groups.sort(key=lambda x: -x[0])
    tokens = len(of)
    k_pages, v_pages = (torch.randn(sum(blocks), nkv, *shape, generator=g).bfloat16().cuda() for shape in ((page, d), (d, page)))
    q = torch.randn(tokens, (nq + 2 * nkv) * d, generator=g).bfloat16().cuda()
    of, at, first, count, table = (torch.tensor(x, dtype=torch.int32).cuda() for x in (of, at, [x[1] for x in groups], [x[2] for x in groups], table.tolist()))
    weight, cos, sin = (1 + 0.1 * torch.randn(d, generator=g)).bfloat16().cuda(), *(torch.randn(tokens, d // 2, generator=g).cuda() for _ in range(2))
    one = singles + 1 == len(requests)

    def prepare(first, end):
        return ops.DecodePrepare(weight, weight, 1e-6, cos[first:end], sin[first:end], 0) if prepared else None

    want, got = (torch.full((tokens, nq * d), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    scale = 1 / math.sqrt(d)
    ops.attention_decode(want[:singles], q[:singles], k_pages, v_pages, table, of, at, nq, scale, window, prepare=prepare(0, singles), form=1)
    whole = ops.DecodePrepare(weight, None, 1e-6, cos, sin, 0) if prepared else None
    behind = ops.DecodePrepare(weight, None, 1e-6, cos[singles:], sin[singles:], 0) if prepared else None
    ops.attention_prefill(want[singles:], q[singles:], k_pages, v_pages, table, of[singles:], at[singles:], first, count, nq, scale, window, size, prepare=behind, one_request=one)
    ops.attention_mixed(got, q, k_pages, v_pages, table, of, at, singles, first, count, nq, scale, window, size, prepare=whole, one_request=one)
    assert torch.equal(got, want) and not got.isnan().any()


def test_mixed_steps_from_plans_and_graphs(ops, tmp_path, monkeypatch):
    """Nine decoding requests beside a portion long enough for groups of 32, whose neighbours walk together (two heads a kv group): the
    shape comes back with other tokens, contexts and pages, through the parts, from the recorded plan and from its graph.  Every row of
    logits equals, bit for bit, that of a runner without plans, and agrees with the plain implementation."""
    import numpy as np

    from llm_runtime_study_amd.config import config_from_dict
    from llm_runtime_study_amd.engine.step import StepEntry
    from llm_runtime_study_amd.weights import write_model_dir
    from tests.helpers import TINY_C
    from tests.plain import model as plain
    from tests.test_step_gpu import make_runner

    write_model_dir(config_from_dict(dict(TINY_C, head_dim=128, num_attention_heads=32, num_key_value_heads=16, max_position_embeddings=4096)), seed=5, model_dir=tmp_path, init="scaled")
    cfg, weights = plain.load_model_dir(tmp_path, torch.float64)
    launched, mixed = [], ops.attention_mixed
    monkeypatch.setattr(ops, "attention_mixed", lambda *a, **k: (launched.append((a[7], a[13], k["one_request"])), mixed(*a, **k)))
    rng = np.random.default_rng(23)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        runners = [make_runner(tmp_path, torch.bfloat16, pages=400, requests=10, seq=2560, step_tokens=2100) for _ in range(2)]
        runners[1].use_plans = False
        history = {r: rng.integers(0, cfg["vocab_size"], n).tolist() for r, n in enumerate((30, 100, 301, 15, 16, 17, 31, 64, 5))}
        caches = [[r.cache.admit(i) for i in range(9)] for r in runners]
        for runner, mine in zip(runners, caches):
            runner.step([StepEntry(mine[i], history[i]) for i in range(9)])
        got, prompts = [], []
        rounds = runners[0].PLAN_GRAPH_AFTER + 4
        for turn in range(rounds):
            tokens = rng.integers(0, cfg["vocab_size"], 9).tolist()
            prompts.append(rng.integers(0, cfg["vocab_size"], 2061).tolist())
            outs = []
            for runner, mine in zip(runners, caches):
                fresh = runner.cache.admit(9 + turn)
                outs.append(runner.step([StepEntry(mine[i], tokens[i:i + 1], [0]) for i in range(9)] + [StepEntry(fresh, prompts[-1], [700, 2060])]).clone())
                runner.cache.release(fresh)
            assert torch.equal(outs[0], outs[1]), f"turn {turn}"
            for i in range(9):
                history[i].append(tokens[i])
            got.append(outs[0].cpu())
        side.synchronize()
        assert launched and set(launched) == {(9, 32, True)}
        assert runners[0].plan_graph_replays >= 2 and runners[0].plan_replays > runners[0].plan_graph_replays and runners[1].plan_replays == 0
    whole = [plain.qwen3_forward(weights, cfg, history[i]) for i in range(9)]
    for turn in (0, rounds - 1):
        prompt = plain.qwen3_forward(weights, cfg, prompts[turn])
        want = [whole[i][len(history[i]) - rounds + turn] for i in range(9)] + [prompt[700], prompt[2060]]
        for row, ref in zip(got[turn], want):
            assert (row.double() - ref).norm() / ref.norm() < 3e-2
