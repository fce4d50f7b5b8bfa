"""Prompt lookup with histories split over workgroups, at the edges of its tiles, against the
oracle's brute force and, with tokens appended by the call, against one workgroup per history."""

import numpy as np
import pytest
import torch

from mvsd import _native as nat
from mvsd.spec_decode import ngram_proposer_gpu as ngram
from mvsd.spec_decode.ngram_proposer_gpu import ngram_propose_device
from oracle import ngram as oracle_ngram

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 3, 4095, 4096, 4097, 4098, 4099, 8192, 8193, 8194, 12290, 20000]


def histories(rng, lens, width, vocab):
    tokens = rng.integers(0, vocab, size=(len(lens), width)).astype(np.int32)
    for i, n in enumerate(lens):
        if i % 3 and n > 40:  # end on a copy of an earlier span, at a tile's edge or anywhere
            w = 8
            src = min(4096 - w // 2, n - 2 * w) if i % 3 == 1 else int(rng.integers(0, n - 2 * w))
            tokens[i, n - w:n] = tokens[i, src:src + w]
    return tokens


@pytest.mark.parametrize("B", [1, 5, 60, 500])
@pytest.mark.parametrize("vocab", [3, 50000])
def test_lengths_match_oracle(device, B, vocab):
    rng = np.random.default_rng(B + vocab)
    lens = np.array([LENGTHS[(i + B) % len(LENGTHS)] for i in range(B)], dtype=np.int32)
    tokens = histories(rng, lens, 20000, vocab)
    t, n = torch.from_numpy(tokens).to(device), torch.from_numpy(lens).to(device)
    for min_n, max_n, k in ((2, 5, 5), (1, 1, 3), (1, 32, 8)):
        want, counts = oracle_ngram.brute_device_batch(tokens, lens, min_n, max_n, k)
        for _ in range(2):  # the workspace is left as the next call needs it
            drafts, valid = ngram_propose_device(t, n, min_n=min_n, max_n=max_n, k=k)
            assert np.array_equal(drafts.cpu().numpy(), want)
            assert np.array_equal(valid.cpu().numpy(), counts)


def test_appended_tokens_equal_one_workgroup(device):
    """Tokens appended by the call (some -1, some past the buffer) around tile edges."""
    rng = np.random.default_rng(3)
    width, k = 12300, 6
    lens = np.array([4090, 4095, 4096, 4097, 8189, 8192, 12297, 12300, 5000, 3], dtype=np.int32)
    B = len(lens)
    tokens = torch.from_numpy(histories(rng, lens, width, 4)).to(device)
    new = torch.from_numpy(rng.integers(-1, 4, size=(B, 7)).astype(np.int32)).to(device)
    counts = torch.from_numpy(rng.integers(0, 8, size=B).astype(np.int32)).to(device)
    n = torch.from_numpy(lens).to(device)
    a, b = tokens.clone(), tokens.clone()
    drafts, valid = ngram_propose_device(a, n, min_n=2, max_n=6, k=k, new_tokens=new,
                                         new_counts=counts, gate_on_new_counts=True)
    want = torch.empty((B, k), dtype=torch.int32, device=device)
    want_valid = torch.empty(B, dtype=torch.int32, device=device)
    nat.check(nat.lib().mvsd_ngram_propose(
        want.data_ptr(), want_valid.data_ptr(), b.data_ptr(), width, width, n.data_ptr(),
        new.data_ptr(), new.stride(0), 7, counts.data_ptr(), None, 1, B, 2, 6, k, 0, 0,
        nat.stream_of(device)), "mvsd_ngram_propose")
    assert torch.equal(a, b)
    assert torch.equal(drafts, want) and torch.equal(valid, want_valid)


def test_kept_workspaces_are_bounded(device, monkeypatch):
    """One workspace per stream, the oldest given back; each stream's results as before."""
    monkeypatch.setattr(ngram, "_WORKSPACES", {})
    monkeypatch.setattr(ngram, "_MAX_WORKSPACES", 2)
    rng = np.random.default_rng(5)
    lens = np.array([20000, 12290, 4097], dtype=np.int32)
    tokens = histories(rng, lens, 20000, 50000)
    want, counts = oracle_ngram.brute_device_batch(tokens, lens, 2, 5, 5)
    t, n = torch.from_numpy(tokens).to(device), torch.from_numpy(lens).to(device)
    torch.cuda.synchronize()
    for _ in range(2):
        for stream in [torch.cuda.Stream(device) for _ in range(4)]:
            with torch.cuda.stream(stream):
                drafts, valid = ngram_propose_device(t, n, min_n=2, max_n=5, k=5)
            stream.synchronize()
            assert len(ngram._WORKSPACES) <= 2
            assert np.array_equal(drafts.cpu().numpy(), want)
            assert np.array_equal(valid.cpu().numpy(), counts)
