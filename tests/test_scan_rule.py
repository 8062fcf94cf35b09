"""Which sequences of a step the recurrences take in chunks: a rule on the host."""

from types import SimpleNamespace

import numpy as np
import pytest

from socrates_amd.kernels.attention import Attention
from socrates_amd.kernels.scan import Scan


class Rule(Scan):
    _portion_lengths = staticmethod(Attention._portion_lengths)


def step(lengths):
    return SimpleNamespace(n_seqs=len(lengths), max_q_len=max(lengths), host={"seq_qstart": np.cumsum([0] + lengths)})


@pytest.mark.parametrize("lengths,least", [
    ([200], 200), ([100], 0), ([1] * 50 + [160], 0), ([1] * 7 + [160], 1), ([200] + [1] * 60, 200), ([2000] + [1] * 60, 2000), ([200] * 5, 200),
    ([1100, 698, 330], 330), ([1, 500, 300, 1, 7], 1), ([1] * 20 + [500, 300, 7], 300), ([260] + [64] * 30, 64), ([1] * 64, 0)])
def test_decoding_rows_are_not_in_chunks(lengths, least):
    """20 heads of 128 x 128: 160 blocks of 16 columns."""
    rule, ctx = Rule(), step(lengths)
    assert rule._chunks_from(ctx, 128, 160) == least
    assert rule._split(ctx, least or 1 << 20) == (sum(n >= (least or 1 << 20) for n in lengths), min(lengths) < (least or 1 << 20))
    assert not rule._chunks_from(ctx, 129, 160)


def test_heads_that_fill_the_chip_side_by_side_are_not_walked_in_turns():
    """80 heads of 128 x 64: five walks of 1,000 tokens have twice the blocks that run at once."""
    assert Rule()._chunks_from(step([1000] * 5), 128, 320) == 1000


@pytest.mark.parametrize("lengths,least", [
    ([300], 300), ([200], 0), ([300] + [1] * 60, 0), ([2000] + [1] * 60, 2000), ([500] * 2, 500), ([500] * 3, 0), ([1000] * 5, 0), ([1000] * 8, 0)])
def test_the_delta_rule_weighs_its_chunks(lengths, least):
    assert Rule()._delta_in_chunks(step(lengths), sum(lengths), 128, 20, 128) == least


@pytest.mark.parametrize("work,lengths,least", [
    (9 / 5, [287], 0), (9 / 5, [288], 288), (9 / 5, [162] * 2, 0), (9 / 5, [200] * 2, 200), (9 / 5, [260, 215, 169, 124, 78], 78),
    (9 / 5, [150] * 8, 0), (9 / 5, [300] + [1] * 30, 0), (9 / 5, [400] + [1] * 30, 400), (9 / 5, [300] + [1] * 7, 1),
    (23 / 20, [183], 0), (23 / 20, [184], 184), (23 / 20, [162] * 2, 162), (23 / 20, [200] + [1] * 60, 0), (23 / 20, [250] + [1] * 60, 250)])
def test_steps_that_wait_for_the_host_walk(work, lengths, least):
    """Where a step of few tokens is no faster for its kernels, the launches decide: by the longest sequence and all tokens."""
    rule = Rule()
    assert rule._chunks_from(step(lengths), 64, 160, work) == least
    rule.scan_from = 0
    assert not rule._chunks_from(step(lengths), 64, 160, work)


def test_a_step_that_does_not_say_its_lengths_is_in_chunks_whole():
    rule, ctx = Rule(), SimpleNamespace(n_seqs=61, max_q_len=2000)
    assert rule._chunks_from(ctx, 128, 160) == 1 and rule._split(ctx, 1) == (61, False)


def test_slots_hold_every_chunk():
    """Numbers as the kernels give them: qstart / 64 + l for the l-th sequence in chunks."""
    rng = np.random.default_rng(0)
    for _ in range(200):
        n = rng.integers(1, 150)
        lens = np.where(rng.random(n) < 0.7, 1, rng.integers(1, 400, n))
        lens[rng.integers(len(lens))] = rng.integers(1, 3000)
        least = min(int(rng.choice([1, 2, 64, 3000])), int(lens.max()))
        start = np.cumsum(lens) - lens
        long = lens >= least
        first = start[long] // 64 + np.arange(long.sum())
        end = first + -(-lens[long] // 64)
        assert (end[:-1] <= first[1:]).all() and end[-1] <= lens.sum() // 64 + long.sum()
