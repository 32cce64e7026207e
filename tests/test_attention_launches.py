"""How many launches the attention of a mixed step takes where the kernels for any shape serve it: two only where the tokens of the
portion can share workgroups."""

from types import SimpleNamespace

import pytest
import torch

from llm_runtime_study_amd.kernels import ops
from llm_runtime_study_amd.parts.attention import GQAAttention


@pytest.mark.parametrize("form,launches", [("plain", 2), ("bfloat16", 1), ("heads of 160", 1), ("gates", 1), ("kept", 1), ("sinks", 1), ("capped", 1), ("distance", 1), ("narrow values", 1),
                                           ("all decode", 1), ("no singles", 1)])
def test_launches(monkeypatch, form, launches):
    calls = []
    monkeypatch.setattr(ops, "attention", lambda out, q, k, v, table, of, at, *a, together=1, **more: calls.append((out.shape[0], of.tolist()[:out.shape[0]], together, more)))
    part = GQAAttention.__new__(GQAAttention)
    torch.nn.Module.__init__(part) if isinstance(part, torch.nn.Module) else None
    d = 160 if form == "heads of 160" else 64
    part.num_heads, part.head_dim, part.value_dim, part.scale, part.reach, part.keep_first = 4, d, 32 if form == "narrow values" else d, 0.125, 0, 4 if form == "kept" else 0
    dtype = torch.bfloat16 if form == "bfloat16" else torch.float32
    of = torch.tensor([3, 1, 2, 0, 0, 0, 0], dtype=torch.int32)
    ctx = SimpleNamespace(all_decode=form == "all decode", single_rows=0 if form == "no singles" else 3, dtype=dtype, memo={}, max_k=20, token_slot=of, positions=of + 9)
    cache = SimpleNamespace(k_pages=torch.zeros(1, 2, 16, d), v_pages=torch.zeros(1, 2, part.value_dim, 16))
    more = {"sinks": None, "softcap": 0.0, "distance": None}
    if form in ("sinks", "distance"):
        more[form] = torch.ones(4)
    if form == "capped":
        more["softcap"] = 30.0
    gates = torch.zeros(7, 4) if form == "gates" else None
    part._attend(ctx, torch.zeros(7, 4 * part.value_dim), torch.zeros(7, 8 * d), cache, SimpleNamespace(block_table=None, page_size=16), gates=gates, **more)
    assert [c[0] for c in calls] == ([3, 4] if launches == 2 else [7])
    assert sum((c[1] for c in calls), []) == of.tolist()
    if launches == 2:
        assert [c[2] for c in calls] == [1, 16]


def test_short_contexts_are_told_and_go_straight_into_registers(monkeypatch):
    """A launch is told a bound of its contexts that all steps of a shape share; a piece or two of keys, and rows that nearly fill the chip over some
    hundreds, come straight into registers, as every other launch did better through LDS."""
    direct = ops.attention_f32_direct
    for workgroups in (1, 8, 64, 200, 256, 2000):
        assert direct(workgroups, 1, 100) and direct(workgroups, 16, 128) and direct(workgroups, 1, 192)
        assert not direct(workgroups, 1, 0) and not direct(workgroups, 16, 129) and not direct(workgroups, 1, 2047)
    if ops.compute_units() in (0, 256):
        assert not direct(127, 1, 255) and direct(128, 1, 255) and direct(2000, 1, 256)
        assert [direct(n, 1, 511) for n in (64, 192, 193, 256, 257, 512)] == [False, False, True, True, False, False] and direct(256, 1, 1023)
    told = []
    monkeypatch.setattr(ops, "attention", lambda *a, longest=0, **more: told.append(longest))
    part = GQAAttention.__new__(GQAAttention)
    part.num_heads, part.head_dim, part.value_dim, part.scale, part.reach, part.keep_first = 16, 96, 96, 0.125, 0, 0
    of = torch.zeros(7, dtype=torch.int32)
    cache = SimpleNamespace(k_pages=torch.zeros(1, 8, 16, 96), v_pages=torch.zeros(1, 8, 96, 16))
    for max_k in (20, 255, 256, 300, 511, 512, 5000):
        ctx = SimpleNamespace(all_decode=True, single_rows=0, dtype=torch.float32, memo={}, max_k=max_k, token_slot=of, positions=of)
        part._attend(ctx, torch.zeros(7, 16 * 96), torch.zeros(7, 32 * 96), cache, SimpleNamespace(block_table=None, page_size=16))
    assert told == [20, 255, 511, 511, 511, 1023, 8191]


@pytest.mark.parametrize("decode", [True, False])
@pytest.mark.parametrize("span,reach", [(None, 0), (300, 300), (450, -450), (1000, 1000)])
@pytest.mark.parametrize("max_k", [256, 300, 2000, 9000])
def test_rows_of_their_own_are_divided(monkeypatch, decode, span, reach, max_k):
    """Long float32 rows of a request each go to the divided form, a mixed step's other tokens to attention(), every row once, with places for
    every piece that a row can see; where the places would take too much, everything goes to attention()."""
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    divided, whole = [], []
    monkeypatch.setattr(ops, "attention_f32_divided", lambda out, q, k, v, table, of, at, nq, scale, window, splits, slots, o, ml: divided.append((of.tolist()[:out.shape[0]], window, splits, slots, o.numel(), ml.numel())))
    monkeypatch.setattr(ops, "attention", lambda out, q, k, v, table, of, at, nq, scale, window, *a, together=1, **more: whole.append((of.tolist()[:out.shape[0]], window, together)))
    part = GQAAttention.__new__(GQAAttention)
    part.num_heads, part.head_dim, part.value_dim, part.scale, part.reach, part.keep_first, part.span = 4, 64, 64, 0.125, reach, 0, span
    of = torch.tensor([3, 1, 2, 0, 0, 0, 0], dtype=torch.int32)
    bound = -(-max_k // 256) * 256
    ctx = SimpleNamespace(all_decode=decode, single_rows=0 if decode else 3, dtype=torch.float32, memo={}, max_k=max_k, max_k_bound=bound, token_slot=of, positions=of,
                          scratch=lambda name, shape, dtype: torch.empty(shape, dtype=dtype))
    cache = SimpleNamespace(k_pages=torch.zeros(1, 2, 16, 64), v_pages=torch.zeros(1, 2, 64, 16))
    out, qkv, alone = torch.zeros(7, 4 * 64), torch.zeros(7, 8 * 64), 7 if decode else 3

    def step():
        divided.clear(), whole.clear()
        part._attend(ctx, out, qkv, cache, SimpleNamespace(block_table=None, page_size=16))

    step()
    (rows, window, splits, slots, sums, maxima), = divided
    assert rows == of.tolist()[:alone] and window == reach and splits > 1 and (sums, maxima) == (alone * 4 * slots * 64, alone * 4 * slots * 2)
    assert whole == ([] if decode else [(of.tolist()[3:], reach, 16)])
    for pos in range(bound):
        first = 0 if not reach else max(pos - reach + 1, 0) if reach > 0 else pos - pos % -reach
        assert pos // 64 - first // 64 + 1 <= slots
    part.PIECE_RESULTS = alone * 4 * slots * (64 + 2) - 1
    step()
    assert not divided and whole == ([(of.tolist(), reach, 1)] if decode else [(of.tolist()[:3], reach, 1), (of.tolist()[3:], reach, 16)])
    part.PIECE_RESULTS += 1
    for heads, d in ((10, 64), (4, 96)):                   # more than four heads a kv head; heads of another size
        part.num_heads, part.head_dim, part.value_dim = heads, d, d
        cache = SimpleNamespace(k_pages=torch.zeros(1, 2, 16, d), v_pages=torch.zeros(1, 2, d, 16))
        out, qkv = torch.zeros(7, heads * d), torch.zeros(7, (heads + 4) * d)
        step()
        assert not divided and sum((rows for rows, *_ in whole), []) == of.tolist()
