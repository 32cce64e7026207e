"""The choice of experts by one wave a token: numbers of experts around a wave's lanes and beyond, ties, several choices a lane."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,groups,keep,scale", [("softmax_chosen", 0, 0, 1.0), ("sigmoid", 0, 0, 2.5), ("sigmoid", 4, 2, 1.0), ("sigmoid_scores", 0, 0, 0.5), ("softmax_scores", 0, 0, 1.5)])
@pytest.mark.parametrize("experts,top", [(4, 1), (60, 8), (64, 32), (68, 3), (64, 7), (132, 66), (512, 8)])
def test_choices_and_weights(experts, top, kind, groups, keep, scale):
    """Against 64 bits on the host: logits a step of 1/64 apart or equal (the lowest index goes first then), sums of at most 66 shares."""
    from llm_runtime_study_amd.kernels import ops

    if groups and keep * (experts // groups) < top:
        pytest.skip("fewer experts in the kept groups than choices")
    tokens = 19
    g = torch.Generator().manual_seed(experts + top)
    logits = torch.randint(-128, 129, (tokens, experts), generator=g).float() / 64
    ids = torch.full((tokens, top), -1, dtype=torch.int32, device="cuda")
    weights = torch.full((tokens, top), float("nan"), device="cuda")
    ops.moe_route(logits.cuda(), None, ids, weights, ops.RouteRule(kind, groups, keep, scale))
    z = logits.double()
    score = z if kind == "softmax_chosen" else torch.softmax(z, 1) if kind == "softmax_scores" else torch.sigmoid(z)
    order = score if groups else z
    if groups:
        kept = score.view(tokens, groups, -1).topk(min(2, experts // groups), -1).values.sum(-1).sort(dim=-1, descending=True, stable=True).indices[:, :keep]
        allowed = torch.zeros(tokens, groups, dtype=torch.bool).scatter_(1, kept, True)
        order = order.view(tokens, groups, -1).masked_fill(~allowed[:, :, None], -torch.inf).flatten(1)
    chosen = order.sort(dim=-1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(ids.cpu().long(), chosen)
    share = score.gather(1, chosen)
    if kind == "softmax_chosen":
        share = torch.softmax(share, 1)
    elif kind == "sigmoid":
        share = share / (share.sum(1, keepdim=True) + 1e-20)
    torch.testing.assert_close(weights.cpu().double(), share * (1.0 if kind == "softmax_chosen" else scale), rtol=2 ** -17, atol=0.0)


@pytest.mark.parametrize("experts", [1, 63, 64, 65, 200])
def test_runs_of_pairs(experts):
    """Every expert's pairs lie in one run of whole tiles, in the order of the experts."""
    from llm_runtime_study_amd.kernels import ops

    tokens, top = 23, 3
    g = torch.Generator().manual_seed(experts)
    ids = torch.randint(0, experts, (tokens, top), generator=g).int()
    tile, tiles = ops.moe_tile_rows(tokens * top, experts), ops.moe_max_tiles(tokens * top, experts)
    rows, place, owner = (torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (tiles * tile, tokens * top, tiles))
    ops.moe_align(ids.cuda(), experts, rows, place, owner)
    rows, place, owner, flat = rows.cpu().tolist(), place.cpu().tolist(), owner.cpu().tolist(), ids.flatten().tolist()
    want = [e for e in range(experts) for _ in range(-(-flat.count(e) // tile))]
    assert owner == want + [-1] * (tiles - len(want))
    assert [rows[at] for at in place] == list(range(tokens * top)) and sorted(r for r in rows if r >= 0) == list(range(tokens * top))
    assert all(owner[at // tile] == flat[pair] for pair, at in enumerate(place))
