"""bfloat16 products of many rows in tiles: the choice of tile and parts, registers, and every tile at its edges."""

import itertools

import pytest
import torch

from tests.test_registers import spills


def test_the_choice_of_tile_and_parts():
    from llm_runtime_study_amd.kernels import ops

    room = ops.gemm_workspace_bytes()
    for m in (1, 65, 129, 256, 500, 1024, 2047, 8192):
        for n in (4, 68, 128, 132, 1024, 4096, 10304, 151936):
            for k in (64, 128, 192, 1088, 4096, 12288):
                bm, bn, parts = ops.gemm_tiles_choice(m, n, k)
                panels = 2 if (bm, bn) in ((128, 128), (64, 128), (64, 64)) else 1
                steps = k // (64 * panels)
                assert k % (64 * panels) == 0 and 1 <= parts <= 8
                if parts > 1:
                    each = -(-steps // parts)
                    assert (parts - 1) * each < steps and each * panels >= 8 and parts * m * n * 4 <= room
                    assert n > 128 or m > 4096 or (m == 4096 and k >= 4096)
                assert ops.gemm_tiles_choice(m, n, k, 0)[2] == 1
    if ops.compute_units() in (0, 256):
        assert ops.gemm_tiles_choice(2048, 24576, 4096) == (256, 256, 1) and ops.gemm_tiles_choice(512, 19456, 2560) == (256, 160, 1)
        # few outputs: divided from 4,096 rows on, where a router's own kernel has more than a round of the chip, all up to 128 alike
        assert ops.gemm_tiles_choice(4096, 64, 8192)[2] > 1 and ops.gemm_tiles_choice(8192, 8, 8192)[2] > 1 and ops.gemm_tiles_choice(4095, 64, 8192)[2] == 1
        for m, n, k in itertools.product((4096, 5000, 16384, 20000), (8, 64, 100), (512, 2048, 8192, 28672)):
            mine, all_of_them = ops.gemm_tiles_choice(m, n, k), ops.gemm_tiles_choice(m, 128, k)
            assert mine == all_of_them or mine[2] == all_of_them[2] == 1           # divided: the same tile too, whose slices the parts begin at
        # rows that stream from memory: no parts a multiple of 4 KB apart, no parts for less than a tenth, others as ever
        assert ops.gemm_tiles_choice(16384, 256, 8192) == (128, 128, 1) and ops.gemm_tiles_choice(32768, 192, 8192) == (128, 192, 1)
        assert ops.gemm_tiles_choice(28000, 128, 5120)[2] == 1 and ops.gemm_tiles_choice(16384, 8, 8192) == (64, 64, 1)
        assert [ops.gemm_tiles_choice(m, n, k)[2] for m, n, k in ((17000, 192, 8192), (5000, 192, 28672), (5000, 8, 28672), (8192, 256, 8192))] == [3, 6, 6, 4]
        # weights that the cache does not hold are divided like any
        assert ops.gemm_tiles_choice(129, 8192, 28672) == (256, 256, 8) and ops.gemm_tiles_choice(256, 5120, 27648) == (256, 160, 8)
        assert ops.gemm_tiles_choice(256, 1024, 1024) == (64, 64, 1) and ops.gemm_tiles_choice(512, 4096, 12288)[2] > 1


def test_what_goes_to_the_tiles_rather_than_to_the_library():
    from llm_runtime_study_amd.kernels import ops

    pay = ops.gemm_tiles_pay
    assert [pay(m, 6144, 2560, "nothing") for m in (129, 160, 161, 191, 192, 200, 224, 255, 256)] == [True, True, False, False, True, False, True, False, True]
    assert pay(200, 4096, 2560, "nothing") and pay(200, 6144, 1536, "nothing") and pay(200, 6144, 4096, "nothing")
    assert pay(256, 6144, 4096, "nothing") and not pay(257, 6144, 4096, "nothing") and not pay(128, 6144, 4096, "nothing")
    assert pay(2048, 24576, 4096, "gate") and pay(129, 6144, 1024, "gate") and not pay(512, 6144, 1056, "gate") and not pay(512, 6152, 1024, "gate")
    assert pay(2048, 4096, 12288, "norm") and not pay(2048, 4096, 4096, "norm") and not pay(300, 64, 4096, "norm") and not pay(300, 8196, 65536, "norm")
    assert not pay(512, 24576, 448, "gate")
    if ops.compute_units() in (0, 256):
        # tiles that rows or columns leave half empty: by the library
        assert [pay(m, 32000, 4096, "nothing, float32") for m in (256, 300, 420, 512, 560, 768, 2048)] == [True, False, True, True, False, True, True]
        assert [pay(m, 4096, 12288, "norm") for m in (2049, 3000, 3500, 6000, 7000)] == [True, False, True, False, True]
        assert [pay(m, 28672, 4096, "gate") for m in (129, 256, 300, 512, 2048)] == [True, True, False, True, True] and pay(300, 12288, 2048, "gate")
        assert not pay(160, 1536, 4096, "gate") and pay(160, 1536, 4096, "nothing")              # divided: the gate behind it is a kernel of single values
    assert pay(300, 10304, 4096, "nothing, float32") and not pay(2048, 8192, 4096, "nothing, float32")


def test_tiles_keep_their_values_in_registers(tmp_path):
    """Its waits count the fetches on their way: a spilled value's way back would count among them."""
    found = {name: count for name, count in spills(tmp_path).items() if "gemm_bf16_tiles" in name}
    assert len(found) == 9 and not any(found.values()), found


# every tile, whole and with K in parts, the last of them shorter than the others, with rows and columns that end inside a tile
EDGES = {(256, 256, 1): (263, 24792, 512), (256, 256, 7): (142, 8400, 9344), (256, 192, 1): (258, 22072, 512), (256, 192, 5): (140, 8664, 5696),
         (256, 160, 1): (388, 16444, 512), (256, 160, 3): (138, 12348, 2240), (256, 128, 1): (130, 24800, 512), (256, 128, 4): (143, 8080, 1856),
         (128, 256, 1): (265, 17672, 512), (128, 256, 4): (65, 16376, 2112), (128, 192, 1): (67, 532, 576), (128, 192, 2): (92, 240, 960),
         (128, 128, 1): (65, 17400, 512), (128, 128, 5): (71, 5636, 3072), (64, 128, 1): (70, 8268, 512), (64, 128, 5): (72, 3036, 2432),
         (64, 64, 1): (122, 144, 640), (64, 64, 4): (86, 136, 1664)}


def test_the_edges_are_of_every_tile():
    """What the cases below reach follows from the table of costs: one that is fitted anew has to bring cases that reach every tile again."""
    from llm_runtime_study_amd.kernels import ops

    if ops.compute_units() not in (0, 256):
        pytest.skip("another number of compute units makes other choices")
    for (bm, bn, parts), (m, n, k) in EDGES.items():
        assert ops.gemm_tiles_choice(m, n, k) == (bm, bn, parts) and m % bm and n % bn and n > 128
        if parts > 1:
            steps = k // (128 if (bm, bn) in ((128, 128), (64, 128), (64, 64)) else 64)
            assert steps % -(-steps // parts)
    assert {tile[:2] for tile in EDGES} == {tile[:2] for tile in EDGES if tile[2] == 1} == {tile[:2] for tile in EDGES if tile[2] > 1} and len(EDGES) == 18


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [*EDGES.values(),
    (2047, 24560, 128), (2048, 24576, 64), (1500, 12276, 192), (512, 19452, 320), (257, 19456, 640), (1030, 6148, 1024), (2048, 4096, 128), (1537, 4092, 576),
    (385, 12288, 192), (300, 9000, 1088), (129, 12300, 448), (1020, 4100, 256), (700, 2052, 384), (129, 68, 64), (65, 4096, 128), (191, 1028, 512), (129, 132, 1024),
    (1020, 12272, 320), (512, 4096, 4096), (300, 1024, 3072), (145, 2560, 9728), (1024, 2560, 2816)])
def test_products_in_tiles(m, n, k):
    """Every output form against 64 bits.  A float32 sum of k exact products in any order is off by at most k 2^-24 times the sum of their sizes;
    bfloat16 (8 bits) rounds once more, by up to 2^-8 of the value.  Rows and columns past the matrix are not written."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device="cuda").bfloat16()
    w = (torch.randn(n, k, generator=g, device="cuda") / k ** 0.5).bfloat16()
    want, bound = a.double() @ w.double().T, (a.double().abs() @ w.double().abs().T) * k * 2.0 ** -24
    wide = torch.full((m + 1, n + 4), 7.0, device="cuda")
    ops.gemm(wide[:m, :n], a, w)
    assert ((wide[:m, :n] - want).abs() <= bound).all() and (wide[m:] == 7).all() and (wide[:, n:] == 7).all()
    added = torch.randn(m, n, generator=g, device="cuda")
    before = added.clone()
    ops.gemm(added, a, w, accumulate=True)
    assert torch.equal(added, before + wide[:m, :n])
    stored = torch.full((m + 1, n + 4), 7.0, device="cuda", dtype=torch.bfloat16)
    ops.gemm(stored[:m, :n], a, w)
    assert torch.equal(stored[:m, :n], wide[:m, :n].bfloat16()) and (stored[m:] == 7).all() and (stored[:, n:] == 7).all()
    if n % 16 == 0:
        gated = torch.empty(m, n // 2, device="cuda", dtype=torch.bfloat16)
        ops.gemm(gated, a, w, swiglu=True)
        pairs = wide[:m, :n].double().reshape(m, n // 16, 2, 8)
        gate, up = (pairs[:, :, i].reshape(m, n // 2) for i in range(2))
        exact = gate * torch.sigmoid(gate) * up
        # the exponential and the quotient in float32: a few 2^-24 of the value for every unit of the exponent, at most 40 of them here
        assert ((gated.double() - exact).abs() <= exact.abs() * (2.0 ** -8 + 2.0 ** -18) + 1e-30).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(256, 1024, 2048), (2048, 4096, 12288), (300, 8192, 1024), (129, 2052, 4096)])
def test_residual_add_and_norm(m, n, k):
    """The product, the add and the norm in two kernels: the stream's bits are those of the product added by itself, the norm is the norm
    kernel's of that stream to the rounding of its output."""
    from llm_runtime_study_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w = torch.randn(m, k, generator=g, device="cuda").bfloat16(), (torch.randn(n, k, generator=g, device="cuda") / k ** 0.5).bfloat16()
    weight = 1 + 0.1 * torch.randn(n, generator=g, device="cuda")
    stream = torch.randn(m, n, generator=g, device="cuda")
    alone = stream.clone()
    normed = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    ops.gemm_tiles_add_rmsnorm(stream, a, w, weight, 1e-6, normed)
    ops.gemm(alone, a, w, accumulate=True)
    assert torch.equal(stream, alone)
    exact = stream.double() * torch.rsqrt(stream.double().square().mean(-1, keepdim=True) + 1e-6) * weight.double()
    assert ((normed.double() - exact).abs() <= exact.abs() * (2.0 ** -8 + 2.0 ** -18)).all()
