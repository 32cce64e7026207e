"""The grouped products of large steps deal the tiles in use to the dies, whose number only the device knows: lists whose
used part ends anywhere, among them lists longer than one look of a wave."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# experts, choices, tokens, how many experts are chosen at all: one tile, few of many, all, more than 64 in the list
@pytest.mark.parametrize("count,top,tokens,chosen", [(2, 1, 96, 1), (6, 2, 145, 6), (16, 2, 400, 2), (40, 4, 640, 40), (70, 1, 3500, 3), (70, 1, 3500, 70), (3, 1, 9000, 3)])
def test_every_tile_in_use_is_made_once(count, top, tokens, chosen):
    from llm_runtime_study_amd.kernels import ops

    n, k = 260, 64
    g = torch.Generator().manual_seed(count + tokens)
    x = torch.randn(tokens, k, generator=g).to(torch.bfloat16)
    w = torch.randn(count, n, k, generator=g).to(torch.bfloat16)
    ids = torch.stack([torch.randperm(chosen, generator=g)[:top] for _ in range(tokens)]).to(torch.int32)
    tile, tiles = ops.moe_tile_rows(tokens * top, count), ops.moe_max_tiles(tokens * top, count)
    assert tile == 128
    sorted_pairs, place = torch.empty(tiles * tile, dtype=torch.int32, device="cuda"), torch.empty(tokens * top, dtype=torch.int32, device="cuda")
    tile_expert = torch.empty(tiles, dtype=torch.int32, device="cuda")
    ops.moe_align(ids.cuda(), count, sorted_pairs, place, tile_expert)
    out = torch.full((tiles * tile, n), -7.0, device="cuda")
    ops.moe_experts(out, x.cuda(), w.cuda(), sorted_pairs, tile_expert, tile, top, gather=True, relu_squared=False)
    got, listed = out.cpu(), sorted_pairs.cpu()
    assert (got[listed < 0] == -7.0).all()                      # rows that only pad are not written
    rows = got[place.cpu().long()].double().view(tokens, top, n)
    for e in range(chosen):
        t, c = (ids == e).nonzero(as_tuple=True)
        want = x[t].double() @ w[e].double().T
        size = x[t].double().abs() @ w[e].double().abs().T
        assert ((rows[t, c] - want).abs() <= k * 2.0 ** -23 * size).all()        # float32 sums of k exact products, whatever their order


@pytest.mark.parametrize("count,top,tokens", [(6, 2, 145), (40, 4, 640), (70, 1, 3500)])
def test_lists_with_tiles_not_in_use_between_those_in_use(count, top, tokens):
    from llm_runtime_study_amd.kernels import ops

    n, k, tile = 260, 64, 128
    g = torch.Generator().manual_seed(count)
    x, w = torch.randn(tokens, k, generator=g).to(torch.bfloat16).cuda(), torch.randn(count, n, k, generator=g).to(torch.bfloat16).cuda()
    ids = torch.stack([torch.randperm(count, generator=g)[:top] for _ in range(tokens)]).to(torch.int32).cuda()
    tiles = ops.moe_max_tiles(tokens * top, count)
    assert ops.moe_tile_rows(tokens * top, count) == tile
    sorted_pairs, place = torch.empty(tiles * tile, dtype=torch.int32, device="cuda"), torch.empty(tokens * top, dtype=torch.int32, device="cuda")
    tile_expert = torch.empty(tiles, dtype=torch.int32, device="cuda")
    ops.moe_align(ids, count, sorted_pairs, place, tile_expert)
    # every tile two or three places further on than the one before it
    to = torch.cumsum(torch.randint(1, 4, (tiles,), generator=g), 0)
    spread = int(to[-1]) + 2
    wide_expert, wide_pairs = torch.full((spread,), -1, dtype=torch.int32), torch.full((spread, tile), -1, dtype=torch.int32)
    wide_expert[to], wide_pairs[to] = tile_expert.cpu(), sorted_pairs.view(tiles, tile).cpu()
    want, got = torch.full((tiles * tile, n), -7.0, device="cuda"), torch.full((spread * tile, n), -7.0, device="cuda")
    ops.moe_experts(want, x, w, sorted_pairs, tile_expert, tile, top, gather=True, relu_squared=False)
    ops.moe_experts(got, x, w, wide_pairs.flatten().cuda(), wide_expert.cuda(), tile, top, gather=True, relu_squared=False)
    got = got.view(spread, tile, n)
    assert torch.equal(got[to.cuda()].view(tiles * tile, n), want)
    between = torch.ones(spread, dtype=torch.bool)
    between[to] = False
    assert (got[between.cuda()] == -7.0).all()


# runs of one tile, two, an odd and an even number of them, one of more than 64 tiles, and few or many columns; K of one slice of 64, two
# and more (and of half a slice more, which another kernel takes); rows gathered and rows as they are
@pytest.mark.parametrize("rows,n,k", [((1,), 256, 64), ((128, 129, 256, 257, 1), 260, 128), ((384, 0, 500, 128), 516, 192), ((9000, 130, 640), 68, 448), ((300,) * 70, 256, 320),
                                      ((200, 700), 260, 96)])
@pytest.mark.parametrize("gather,kind", [(True, "bf16"), (True, "pairs"), (False, "f32")])
def test_two_tiles_and_one(rows, n, k, gather, kind):
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator().manual_seed(n + k)
    count, tile = len(rows), 128
    tiles = [-(-m // tile) for m in rows]
    total = sum(tiles)
    spare = 3                                                    # tiles not in use at the end
    listed = torch.full((total + spare, tile), -1, dtype=torch.int32)
    experts, pair, at = torch.full((total + spare,), -1, dtype=torch.int32), 0, 0
    order = torch.randperm(sum(rows), generator=g).to(torch.int32)
    for e, m in enumerate(rows):
        experts[at:at + tiles[e]] = e
        listed[at:at + tiles[e]].view(-1)[:m] = order[pair:pair + m]
        at, pair = at + tiles[e], pair + m
    x = torch.randn(sum(rows) if gather else listed.numel(), k, generator=g).to(torch.bfloat16)
    w = torch.randn(count, n, k, generator=g).to(torch.bfloat16)
    out = torch.full((listed.numel(), n // 2 if kind == "pairs" else n), -7.0, device="cuda", dtype=torch.float32 if kind == "f32" else torch.bfloat16)
    ops.moe_experts(out, x.cuda(), w.cuda(), listed.flatten().cuda(), experts.cuda(), tile, 1, gather=gather, relu_squared=False, silu_pairs=kind == "pairs")
    got, flat = out.cpu().double(), listed.flatten()
    assert (got[flat < 0] == -7.0).all()
    for e in range(count):
        rows_of = ((experts == e).repeat_interleave(tile) & (flat >= 0)).nonzero().flatten()
        a = x[flat[rows_of].long()] if gather else x[rows_of]
        want, size = a.double() @ w[e].double().T, a.double().abs() @ w[e].double().abs().T
        bound = k * 2.0 ** -23 * size                            # float32 sums of k exact products, whatever their order
        if kind == "pairs":
            # silu' is at most 1.1; a rounding to bfloat16 of at most 2^-8 at the end, exp and division in float32 below it
            gate, up = want[:, 0::2], want[:, 1::2]
            bound = 1.1 * bound[:, 0::2] * up.abs() + gate.abs() * bound[:, 1::2] + 1e-6 * (gate * up).abs()
            want = torch.nn.functional.silu(gate) * up
        if kind != "f32":
            bound = bound + (want.abs() + bound) * 2.0 ** -8
        assert ((got[rows_of] - want).abs() <= bound + 1e-30).all()


# more items than 256 compute units work on at once: all pairs kept, the last ones of some rounds parted (in the middle of a run, at the
# end of 64 places of the list, all of a small expert's), and whole rounds of nothing but pairs; and a K too short for pairs of so many items
@pytest.mark.parametrize("rows,n,k", [((9000, 130, 640), 1028, 640), ((9000, 130, 640), 2052, 640), ((300, 8000, 1, 257, 256), 2308, 704), ((256,) * 96, 772, 640),
                                      ((512,) * 32 + (3,), 1024, 640), ((9000, 130, 640), 1028, 576)])
@pytest.mark.parametrize("gather,kind", [(True, "pairs"), (False, "f32")])
def test_pairs_kept_and_parted(rows, n, k, gather, kind):
    test_two_tiles_and_one(rows, n, k, gather, kind)


# tiles of 32 rows: an expert's tiles side by side or alone, at both ends of the list, beside tiles not in use (whose rows must stay as they are)
@pytest.mark.parametrize("experts", [(0,), (1, 1), (0, 1, 1), (2, 2, 2, 0), (-1, 1, -1, 1, 1, -1), (0, 1, 2, -1, -1), (1, 0, 0, -1, 2, 2)])
@pytest.mark.parametrize("n,k", [(64, 64), (132, 192), (4160, 128)])
def test_experts_with_one_tile_of_32_rows_and_with_more(experts, n, k):
    from llm_runtime_study_amd.kernels import ops

    g, tile = torch.Generator().manual_seed(n + len(experts)), 32
    x, w = torch.randn(len(experts) * tile, k, generator=g).to(torch.bfloat16), torch.randn(3, n, k, generator=g).to(torch.bfloat16)
    listed = torch.randperm(len(experts) * tile, generator=g).to(torch.int32).view(len(experts), tile)
    listed[:, 20:] = torch.where(torch.arange(len(experts))[:, None] % 2 == 0, listed[:, 20:], -1)
    listed[torch.tensor(experts) < 0] = -1
    out = torch.full((len(experts) * tile, n), -7.0, device="cuda")
    ops.moe_experts(out, x.cuda(), w.cuda(), listed.flatten().cuda(), torch.tensor(experts, dtype=torch.int32).cuda(), tile, 1, gather=True, relu_squared=False)
    got = out.cpu().view(len(experts), tile, n)
    assert (got[listed < 0] == -7.0).all()
    for i, e in enumerate(experts):
        rows = x[listed[i][listed[i] >= 0].long()].double()
        want, size = rows @ w[max(e, 0)].double().T, rows.abs() @ w[max(e, 0)].double().abs().T
        assert ((got[i][listed[i] >= 0].double() - want).abs() <= k * 2.0 ** -23 * size).all()      # float32 sums of k exact products
