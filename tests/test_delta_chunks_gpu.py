"""The gated delta rule in chunks on the matrix cores against the recurrence in 64 bits, beside the scan on the same numbers."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def recurrence(qkv, gates, begun, lengths, groups, heads, d, e):
    """Read-outs [T, heads, e] and last states [R, heads, d, e] in 64 bits."""
    q, k, v = qkv.double().split((groups * d, groups * d, heads * e), 1)
    of = torch.arange(heads) // (heads // groups)
    q, k, v = q.view(-1, groups, d)[:, of], k.view(-1, groups, d)[:, of], v.view(-1, heads, e)
    beta, decay = gates.double().view(-1, 2, heads).unbind(1)
    outs, states, t = [], [], 0
    for r, n in enumerate(lengths):
        S = begun[r].clone()
        for t in range(t, t + n):
            S = decay[t, :, None, None] * S
            u = beta[t, :, None] * (v[t] - torch.einsum("hde,hd->he", S, k[t]))
            S = S + k[t, :, :, None] * u[:, None, :]
            outs.append(torch.einsum("hde,hd->he", S, q[t]))
        t, states = t + 1, states + [S]
    return torch.stack(outs), torch.stack(states)


def matrices(rows, heads, d, e):
    """The heads' matrices [R, heads, d, e] of state rows: element (i, j) at ((i % rows) * e + j) * 16 + i / rows."""
    per = 4 if d <= 64 else 8
    S = rows[:, :heads * per * e * 16].view(-1, heads, per, e, 16).permute(0, 1, 4, 2, 3)
    return S.reshape(len(rows), heads, 16 * per, e)


@pytest.mark.parametrize("heads,groups,d,e,lengths,singles,kind", [
    (4, 2, 24, 40, (130, 1, 64, 65), 0, "slow"), (2, 1, 128, 128, (200, 3), 0, "slow"), (6, 2, 128, 96, (64, 128, 5, 1, 63), 0, "fast"),
    (1, 1, 100, 17, (1,) * 70 + (300,), 0, "slow"), (1, 1, 101, 17, (1,) * 70 + (300, 1, 2), 70, "fast"), (4, 4, 64, 50, (1, 1, 1, 90), 2, "zero"),
    (3, 3, 65, 1, (256,), 0, "zero"), (2, 2, 10, 7, (17, 66), 0, "alike"), (8, 1, 128, 128, (511,), 0, "alike")])
def test_chunks_against_the_recurrence_in_64_bits(heads, groups, d, e, lengths, singles, kind):
    """Portions that end inside, at and behind a chunk, twice in a row over one state; keys' sizes at the edges of blocks; single
    tokens before the portions; decays near one, far from one and of exactly zero, keys that are nearly all alike with step sizes
    near one (every token then rewrites what the one before wrote)."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(len(lengths) + d)
    tokens, requests, taps = sum(lengths), len(lengths), 4
    channels = 2 * groups * d + heads * e
    proj = torch.randn(tokens, channels + heads * e + 2 * heads + 3, generator=g)
    if kind == "alike":
        proj[:, groups * d:2 * groups * d] = 3 + 0.05 * proj[:, groups * d:2 * groups * d]
        proj[:, channels + heads * e:channels + heads * e + heads] += 4
    proj = proj.cuda()
    conv = (torch.randn(channels, taps, generator=g).abs() * 0.5).cuda()
    a_log = {"slow": -5.0, "fast": 0.5, "zero": 6.0, "alike": -4.0}[kind] + torch.randn(heads, generator=g)
    if kind == "zero":
        proj[::3, channels + heads * e + heads:channels + heads * e + 2 * heads] -= 12.0        # zeros among decays near one
    a_log, dt_bias, norm = a_log.cuda(), torch.randn(heads, generator=g).cuda(), (torch.rand(e, generator=g) + 0.5).cuda()
    floats = ops.delta_state_floats(heads, groups, d, e, taps)
    begun = 0.3 * torch.randn(requests + 1, floats, generator=g)
    per = 4 if d <= 64 else 8
    padding = torch.ones(heads * per * e * 16).view(1, heads, per, e, 16)
    padding = (torch.arange(16)[:, None] * per + torch.arange(per) < d).float().t().reshape(1, 1, per, 1, 16) * padding       # rows past d are zero
    begun[:, :padding.numel()] *= padding.reshape(1, -1)
    cu = torch.tensor([0] + list(np.cumsum(lengths)), dtype=torch.int32, device="cuda")
    of = torch.repeat_interleave(torch.arange(requests), torch.tensor(lengths)).int().cuda()
    slots = torch.randperm(requests, generator=g)
    qkv, gates = torch.empty(tokens, channels, device="cuda"), torch.empty(tokens, 2 * heads, device="cuda")
    raw = torch.empty(tokens, heads * e, device="cuda")
    errors = []
    for chunked in (False, True):
        out, state = torch.zeros(tokens, heads * e, dtype=torch.bfloat16, device="cuda"), begun.cuda()
        worst = [0.0, 0.0]
        for _ in range(2):
            before = state.cpu()
            packs = torch.full((ops.delta_pack_floats(tokens, requests, heads, d, e),), float("nan"), device="cuda") if chunked else None
            ops.delta_rule(out, proj, state, of, cu, slots.int().cuda(), requests, conv, groups, heads, d, e, a_log, dt_bias, norm, 1e-5, qkv, gates, raw,
                           packs, singles if chunked else 0)
            torch.cuda.synchronize()
            want, S = recurrence(qkv.cpu(), gates.cpu(), matrices(before.double(), heads, d, e)[slots][:, :, :d], lengths, groups, heads, d, e)
            got = matrices(state.cpu().double(), heads, d, e)[slots]
            assert torch.isfinite(raw).all() and not got[:, :, d:].any()
            worst[0] = max(worst[0], float((raw.cpu().double().view(want.shape) - want).norm() / want.norm()))
            worst[1] = max(worst[1], float((got[:, :, :d] - S).norm() / S.norm()))
        assert torch.equal(state[requests].cpu(), begun[requests])
        errors.append(worst)
    print(kind, d, e, "scan %.2e %.2e, chunks %.2e %.2e" % (*errors[0], *errors[1]))
    # 24 bits: a unit in the last place is 6e-8; a sum of up to 128 products, the one of 64 tokens behind it and the product with the
    # chunk's inverse add independent roundings, some ten units at the most
    assert max(errors[1]) < 2e-6, errors


def test_packs_are_as_large_as_the_walked_requests_need():
    """Single tokens before a portion take no room in the packs: the part's buffer is the portion's, and a buffer of just that size,
    with a guard behind it, gives the read-outs that a larger one gives.  Where there is no memory for it the scan runs."""
    from types import SimpleNamespace

    from llm_runtime_study_amd.kernels import ops
    from llm_runtime_study_amd.parts import PartSpec, create

    heads, d, e, taps, portion = 4, 64, 32, 4, 700
    part = create("mixer", PartSpec("gated_delta_rule", {"hidden_size": 64, "num_heads": heads, "num_kv_heads": heads, "head_dim": d, "value_dim": e, "conv_taps": taps, "norm_eps": 1e-5}))
    g = torch.Generator().manual_seed(5)
    part.bind({name: (torch.randn(spec.shape, generator=g) * 0.1).to(torch.bfloat16).cuda() for name, spec in part.tensors().items()}, torch.bfloat16)
    sizes = []
    for singles, room in ((0, True), (64, True), (0, False)):
        tokens, requests, sized = singles + portion, singles + 1, {}

        def scratch(name, shape, dtype):
            if name == "delta_packs" and not room:
                raise torch.OutOfMemoryError("no room")
            sized[name] = torch.zeros(shape, dtype=dtype, device="cuda")
            return sized[name]

        lengths = torch.tensor([1] * singles + [portion])
        cu = torch.cat((torch.zeros(1), lengths.cumsum(0))).int().cuda()
        ctx = SimpleNamespace(dtype=torch.bfloat16, R=requests, single_rows=singles, scratch=scratch, kernels=ops.KernelChoice(library=False), cu_seqlens_q=cu,
                              token_request=torch.repeat_interleave(torch.arange(requests), lengths).int().cuda(), slot_ids=torch.arange(requests).int().cuda())
        cache = SimpleNamespace(state=torch.zeros(requests, part.state_floats(), device="cuda"))
        assert part.in_chunks(tokens, requests, singles)
        out = torch.zeros(tokens, 64, device="cuda")
        part.forward(ctx, torch.randn(tokens, 64, generator=g).bfloat16().cuda(), out, cache)
        torch.cuda.synchronize()
        assert torch.isfinite(out).all() and out.any()
        if room:
            sizes.append(sized["delta_packs"].numel())
    assert sizes[1] - sizes[0] <= -(-64 // 64) * ops.delta_pack_floats(0, 0, heads, d, e)      # 64 tokens more are a chunk more at most

    singles = 64
    tokens, requests = singles + portion, singles + 1
    lengths = torch.tensor([1] * singles + [portion])
    cu = torch.cat((torch.zeros(1), lengths.cumsum(0))).int().cuda()
    of = torch.repeat_interleave(torch.arange(requests), lengths).int().cuda()
    channels, raws = 2 * heads * d + heads * e, []
    args = (cu, torch.arange(requests).int().cuda(), requests, torch.rand(channels, taps, generator=g).cuda(), heads, heads, d, e, torch.zeros(heads).cuda() - 2,
            torch.zeros(heads).cuda(), torch.ones(e).cuda(), 1e-5)
    proj = torch.randn(tokens, channels + heads * e + 2 * heads, generator=g).cuda()
    for floats, guard in ((ops.delta_pack_floats(tokens, 1, heads, d, e), 4096), (ops.delta_pack_floats(tokens, requests, heads, d, e), 0)):
        room, raw = torch.full((floats + guard,), -7.0, device="cuda"), torch.empty(tokens, heads * e, device="cuda")
        state = torch.zeros(requests, ops.delta_state_floats(heads, heads, d, e, taps), device="cuda")
        ops.delta_rule(torch.empty(tokens, heads * e, dtype=torch.bfloat16, device="cuda"), proj, state, of, *args,
                       torch.empty(tokens, channels, device="cuda"), torch.empty(tokens, 2 * heads, device="cuda"), raw, room[:floats], singles)
        torch.cuda.synchronize()
        assert (room[floats:] == -7.0).all()
        raws.append(raw.cpu())
    assert torch.equal(raws[0], raws[1])


@pytest.mark.parametrize("lengths,chunked", [((1, 1, 400), True), ((1, 300, 40), False), ((255, 256), True), ((700,), True), ((64, 64, 64), False)])
def test_the_part_chooses_and_both_forms_agree(lengths, chunked):
    """Steps on either side of the rule, the second on the state that the first left: the part's bfloat16 rows against its own scan.
    Differences of the last places of 24 bits turn few roundings to 8 bits: an 8-bit unit is 2^-8 at most, in one value of some hundred."""
    from llm_runtime_study_amd.parts import PartSpec, create

    from tests.test_nobodra_gpu import bf16_values
    from tests.test_parts_gpu import PartHarness

    part = create("mixer", PartSpec("gated_delta_rule", {"hidden_size": 64, "num_heads": 4, "num_kv_heads": 2, "head_dim": 96, "value_dim": 48,
                                                        "conv_taps": 4, "norm_eps": 1e-5}))
    w = {name: bf16_values(*spec.shape, scale=spec.shape[-1] ** -0.5 if len(spec.shape) == 2 else 0.5, seed=i) for i, (name, spec) in enumerate(part.tensors().items())}
    w["A_log"] = w["A_log"] - 2.0
    part.bind({name: t.to(torch.bfloat16).cuda() for name, t in w.items()}, torch.bfloat16)
    assert part.in_chunks(sum(lengths), len(lengths), next(i for i, n in enumerate(lengths) if n > 1)) is chunked
    rule, rows = part.in_chunks, []
    for choose in (rule, lambda *a: False):
        part.in_chunks = choose
        harness = PartHarness([part.cache_need()], torch.bfloat16, max_step_tokens=1408)
        live = [harness.cache.admit(str(i)) for i in range(len(lengths))]
        for turn in range(2):
            x = bf16_values(sum(lengths), 64, seed=7 + turn).to(torch.bfloat16).cuda()
            out = torch.zeros(sum(lengths), 64, device="cuda")
            ctx = harness.context([(seq, [0] * n) for seq, n in zip(live, lengths)])
            part.forward(ctx, x, out, ctx.layer_cache(0))
        torch.cuda.synchronize()
        rows.append(out.double().cpu())
    part.in_chunks = rule
    assert (rows[0] - rows[1]).norm() < 2.0 ** -8 * 0.1 * rows[1].norm()


def test_chunks_are_as_near_to_64_bits_as_the_scan():
    """Inputs as a delta layer of random weights has them (rows of order one behind a convolution, decays about 0.5), portions from a
    zero state: over a few of them the chunks' read-outs and states are no further from those of 64 bits than the scan's.  (Means of
    some 100,000 roundings a portion; a single portion's last chunk may add a few per cent to its state, which is what the twentieth is for.)"""
    from llm_runtime_study_amd.kernels import ops

    heads, groups, d, e, taps = 4, 2, 128, 128, 4
    channels, errors = 2 * groups * d + heads * e, []
    for seed, n in enumerate((512, 448, 211, 640, 320)):
        g = torch.Generator().manual_seed(seed)
        proj = torch.randn(n, channels + heads * e + 2 * heads, generator=g).cuda()
        conv, a_log, dt_bias = (torch.randn(channels, taps, generator=g) * 0.5).cuda(), (torch.randn(heads, generator=g) * 0.1).cuda(), (torch.randn(heads, generator=g) * 0.1).cuda()
        cu, of, slots = torch.tensor([0, n], dtype=torch.int32).cuda(), torch.zeros(n, dtype=torch.int32).cuda(), torch.zeros(1, dtype=torch.int32).cuda()
        qkv, gates, raw = torch.empty(n, channels, device="cuda"), torch.empty(n, 2 * heads, device="cuda"), torch.empty(n, heads * e, device="cuda")
        row = []
        for chunked in (False, True):
            state = torch.zeros(1, ops.delta_state_floats(heads, groups, d, e, taps), device="cuda")
            packs = torch.empty(ops.delta_pack_floats(n, 1, heads, d, e), device="cuda") if chunked else None
            ops.delta_rule(torch.empty(n, heads * e, dtype=torch.bfloat16, device="cuda"), proj, state, of, cu, slots, 1, conv, groups, heads, d, e, a_log, dt_bias,
                           torch.ones(e, device="cuda"), 1e-5, qkv, gates, raw, packs)
            torch.cuda.synchronize()
            want, S = recurrence(qkv.cpu(), gates.cpu(), torch.zeros(1, heads, d, e, dtype=torch.float64), (n,), groups, heads, d, e)
            got = matrices(state.cpu().double(), heads, d, e)
            row += [float((raw.cpu().double().view(want.shape) - want).norm() / want.norm()), float((got - S).norm() / S.norm())]
        errors.append(row)
    scan_read, scan_state, read, kept = np.mean(errors, 0)
    print("scan %.2e %.2e, chunks %.2e %.2e" % (scan_read, scan_state, read, kept))
    assert read <= scan_read and kept <= 1.05 * scan_state, errors


@pytest.mark.parametrize("what,value", [("q", "nan"), ("k", "inf"), ("k", "nan"), ("v", "inf"), ("v", "nan"), ("beta", "nan"), ("decay", "nan")])
@pytest.mark.parametrize("token", [0, 5, 37, 63, 79])
@pytest.mark.parametrize("d", [64, 128])
def test_a_token_that_is_not_finite_spoils_no_token_before_it(what, value, token, d):
    """An infinity or NaN in one column of one token: the same read-outs are finite as in the scan (those of every token before it, of
    the other request, of the other columns if it is a value's, of later tokens if it is a query's) and agree with it."""
    from llm_runtime_study_amd.kernels import ops

    heads, groups, e, taps, lengths = 2, 2, 24, 4, (100, 70)
    g = torch.Generator().manual_seed(token + d)
    tokens, requests, channels = sum(lengths), len(lengths), 2 * groups * d + heads * e
    proj = torch.randn(tokens, channels + heads * e + 2 * heads, generator=g)
    proj[token, {"q": 3, "k": groups * d + 3, "v": 2 * groups * d + 3, "beta": channels + heads * e, "decay": channels + heads * e + heads}[what]] = float(value)
    conv = torch.randn(channels, taps, generator=g).abs() * 0.5 + 0.01
    a_log, dt_bias, norm = torch.randn(heads, generator=g) - 3, torch.randn(heads, generator=g), torch.rand(e, generator=g) + 0.5
    proj, conv, a_log, dt_bias, norm = (t.cuda() for t in (proj, conv, a_log, dt_bias, norm))
    cu = torch.tensor([0] + list(np.cumsum(lengths)), dtype=torch.int32, device="cuda")
    of = torch.repeat_interleave(torch.arange(requests), torch.tensor(lengths)).int().cuda()
    raws, states = [], []
    for chunked in (False, True):
        state = torch.zeros(requests, ops.delta_state_floats(heads, groups, d, e, taps), device="cuda")
        raw, out = torch.empty(tokens, heads * e, device="cuda"), torch.empty(tokens, heads * e, dtype=torch.bfloat16, device="cuda")
        packs = torch.empty(ops.delta_pack_floats(tokens, requests, heads, d, e), device="cuda") if chunked else None
        ops.delta_rule(out, proj, state, of, cu, torch.arange(requests, dtype=torch.int32, device="cuda"), requests, conv, groups, heads, d, e, a_log, dt_bias,
                       norm, 1e-5, torch.empty(tokens, channels, device="cuda"), torch.empty(tokens, 2 * heads, device="cuda"), raw, packs)
        torch.cuda.synchronize()
        raws.append(raw.cpu().double())
        states.append(matrices(state.cpu().double(), heads, d, e))
    scan, chunks = raws
    assert torch.isfinite(scan[:token]).all() and torch.isfinite(scan[lengths[0]:]).all() and not torch.isfinite(scan[token]).all()
    assert torch.equal(torch.isfinite(chunks), torch.isfinite(scan)) and torch.equal(torch.isfinite(states[1]), torch.isfinite(states[0]))
    for got, want in ((chunks, scan), (states[1], states[0])):
        kept = torch.isfinite(want)
        assert (got[kept] - want[kept]).norm() <= 4e-6 * want[kept].norm()       # twice what either may be from 64 bits, above


def test_chunks_refuse_what_they_do_not_serve():
    from llm_runtime_study_amd.kernels import ops

    def call(d, tokens, requests, singles, floats):
        heads, e, taps = 1, 16, 2
        channels = 2 * d + e
        t = lambda *shape: torch.zeros(*shape, device="cuda")
        ops.delta_rule(t(tokens, e).bfloat16(), t(tokens, channels + e + 2), t(requests, ops.delta_state_floats(heads, 1, d, e, taps)), t(tokens).int(),
                       t(requests + 1).int(), t(requests).int(), requests, t(channels, taps), 1, heads, d, e, t(heads), t(heads), t(e), 1e-5,
                       t(tokens, channels), t(tokens, 2), t(tokens, e), t(floats), singles)

    plenty = 1 << 20
    for case in ((129, 20, 1, 0, plenty), (64, 20, 2, 2, plenty), (64, 2, 2, 0, plenty), (64, 20, 1, 0, 64)):
        with pytest.raises(Exception, match="delta_rule"):
            call(*case)
