"""Into how many workgroups a decode token's keys are divided: what the rule may not do, over batches, contexts and head sizes."""

import pytest

from llm_runtime_study_amd.kernels import ops
from llm_runtime_study_amd.parts.attention import GQAAttention


@pytest.mark.parametrize("head_dim", [32, 64, 96, 128, 192])
def test_parts_of_a_decode_step(monkeypatch, head_dim):
    monkeypatch.setattr(ops, "compute_units", lambda: 256)
    for workgroups in list(range(1, 300)) + [512, 2048]:
        for longest in (1, 255, 256, 511, 512, 600, 1023, 1024, 2047, 2048, 5000, 8192, 40000, 140000):
            splits, form = GQAAttention._decode_shape(workgroups, longest, longest, 16, head_dim)
            fits = -(-longest // (4096 * 16))                  # what one workgroup's block table entries ask for
            assert splits >= fits
            if workgroups > 256 or head_dim > 128:
                assert (splits, form) == (GQAAttention._decode_splits(workgroups, longest, longest, 16), 1)
                continue
            if form == 1:      # one round is full and contexts are long: as for workgroups of four waves in every respect
                assert longest >= 4096 and 256 % workgroups == 0 and splits == GQAAttention._decode_splits(workgroups, longest, longest, 16)
                continue
            assert splits <= max(1, longest // 256, fits)
            # one round of workgroups; over longer contexts two or three, as full as they can be
            rounds = -(-splits * workgroups // 256)
            assert splits == fits or rounds == 1 or (longest >= 1024 and rounds == 2) or (longest >= 8192 and rounds == 3)
            assert splits == fits or rounds == 1 or (splits + 1) * workgroups > 256 * rounds
            # a context that is far longer than the others is not left to few workgroups
            assert longest < 4096 or splits >= 0.45 * GQAAttention._decode_splits(workgroups, longest, longest, 16)


@pytest.mark.parametrize("head_dim,page,longest,window,splits,form,wanted", [
    (128, 16, 255, None, 1, 1, 1), (128, 16, 256, None, 1, 1, 3), (64, 32, 2048, None, 1, 1, 3), (128, 16, 2048, None, 4, 2, 2),      # short ones; eight waves
    (128, 48, 2048, None, 1, 1, 1), (64, 64, 2048, None, 1, 1, 1), (192, 16, 8192, None, 2, 1, 1),                                  # pages and heads
    (128, 16, 4096, None, 16, 1, 3), (128, 16, 4096, None, 64, 1, 1), (128, 16, 4096, 128, 1, 1, 3), (128, 16, 4096, 64, 1, 1, 1)])   # a workgroup's share
def test_which_keys_are_loaded_as_read_once(head_dim, page, longest, window, splits, form, wanted):
    """Form 3 where a workgroup walks 128 keys and more, of pages and heads whose lines it reads alone."""
    part = GQAAttention.__new__(GQAAttention)
    part.head_dim, part.span = head_dim, window
    assert part._keys_read_once(splits, form, longest, page) == wanted


def test_which_mixed_steps_go_in_one_launch(monkeypatch):
    monkeypatch.setattr(ops, "compute_units", lambda: 256)

    def one(singles, nq, nkv, bound, portion, size):
        splits, _ = GQAAttention._decode_shape(singles * nkv, bound, bound, 16, 128)
        return GQAAttention._one_launch(singles * nkv, splits, -(-portion // size) * nkv, size, nq // nkv, bound)

    assert one(24, 32, 8, 1536, 488, 16) and one(24, 40, 8, 1536, 488, 16) and one(24, 32, 8, 8192, 2028, 32) and not one(24, 32, 8, 60160, 2028, 32)
    assert not one(8, 32, 8, 1536, 488, 16)
    # a decoding request far on among short ones: its keys are divided in a launch of their own
    assert one(17, 32, 8, 8192, 2028, 32) and not one(17, 32, 8, 16128, 2028, 32) and not one(19, 32, 8, 60160, 2028, 32)
    # many heads a group beside a long portion, whose own launch walks its keys once
    assert not one(33, 32, 4, 2048, 2028, 32) and not one(100, 12, 2, 2048, 2028, 32) and one(40, 32, 4, 8192, 2028, 32) and one(66, 12, 2, 1536, 1100, 16)
