"""The penalties' host side: the summaries (csrc/hostops.c) against numpy's distinct values and
counts, and their upload."""

import math
import time
from collections import deque

import numpy as np
import pytest
import torch

from mvsd import _hostops
from mvsd.sample.rejection_sampler import _penalty_entries, _upload


def check(prompts, outputs, specs):
    off, tok, info = _penalty_entries(prompts, outputs, specs)
    assert off.dtype == tok.dtype == info.dtype == np.int32
    assert off.shape == (len(specs) + 1,) and off[0] == 0 and tok.size == info.size == off[-1]
    for r, spec in enumerate(specs):
        prompt = list(prompts[r]) if r < len(prompts) else []
        output = list(outputs[r]) if r < len(outputs) else []
        got = {int(t): int(i) for t, i in zip(tok[off[r]:off[r + 1]], info[off[r]:off[r + 1]])}
        assert len(got) == off[r + 1] - off[r]  # distinct
        want = {t: output.count(t) | (-2 ** 31 if t in prompt else 0)
                for t in {*prompt, *output, *spec}}
        assert got == want


@pytest.mark.parametrize("n", [0, 1, 7, 8, 9, 300])
@pytest.mark.parametrize("vocab", [1, 5, 150000])
def test_counts(n, vocab):
    rng = np.random.default_rng(n + vocab)
    lists = lambda scale: [rng.integers(0, vocab, rng.integers(0, scale * n + 1)).tolist()
                           for _ in range(9)]
    check(lists(3), lists(1), [s[:6] for s in lists(1)])


def test_forms_of_input():
    check([], [], [])
    check([], [[5]], [[1, 2], [], [-1]])                       # missing tail requests
    check([(1, 2, 1)], [np.array([2, 2, 9])], [range(3)])      # any sequence of integers
    check([[np.int64(7), 7, True]], [[0]], [[7]])
    check([[2 ** 31 - 1, -1, -2 ** 31]], [[2 ** 31 - 1]], [[]])
    off, tok, info = _penalty_entries([[1.0, 2.0]], [[2.0]], [[3]])  # as np.asarray reads them
    assert sorted(zip(tok.tolist(), info.tolist())) == [(1, -2 ** 31), (2, 1 - 2 ** 31), (3, 0)]


def test_sequences_without_slices():
    check(deque([[1, 2, 1], (3,)]), deque([[2]]), deque([[4], []]))


@pytest.mark.parametrize("order", [1, -1])
def test_long_and_short_histories(order):
    """Each request's table has its own size, whatever came before it."""
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, 1500, n).tolist() for n in (5000, 900, 40, 3, 0)][::order]
    check(prompts, [p[:50] for p in prompts], [[7, 8]] * 5)


def test_a_long_history_costs_no_more_first_than_last():
    rng = np.random.default_rng(4)
    short = [rng.integers(0, 150000, 20).tolist() for _ in range(2000)]
    long = [rng.integers(0, 150000, 200000).tolist()]

    def seconds(prompts):
        best = math.inf
        for _ in range(3):
            start = time.perf_counter()
            _penalty_entries(prompts, [[]] * 2001, [[]] * 2001)
            best = min(best, time.perf_counter() - start)
        return best

    assert seconds(long + short) < 10 * seconds(short + long)  # about 40 with one table for all


def test_errors():
    room = np.empty(64, dtype=np.int32)
    with pytest.raises(TypeError):
        _hostops.penalty_entries([["a"]], [[]], [[]], room)
    with pytest.raises(TypeError):
        _hostops.penalty_entries([3], [[]], [[]], room)
    with pytest.raises(OverflowError):
        _hostops.penalty_entries([[2 ** 70]], [[]], [[]], room)
    with pytest.raises(ValueError):
        _hostops.penalty_entries([[1, 2, 3]], [[4]], [[5]], room[:8])
    with pytest.raises(ValueError):
        _hostops.penalty_entries([], [], [[]] * 9, room[:4])


def test_uploads_are_refused_in_a_capture(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="capture"):
        _upload([np.zeros(3, np.int32)], torch.device("cpu"))
