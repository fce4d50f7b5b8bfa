"""The split logprobs path (mvsd_topk_scores_split, mvsd_spec_logprobs_split) at the edges of its
chunks, groups and candidate buffers, against sorting the rows in plain torch.

ids and ranks are exact (raw values decide them); values are a log-softmax whose log-sum is an
fp32 sum in another order: 2e-6 absolute + 1e-6 relative, the bar of test_logprobs_gpu.py."""

import math

import pytest
import torch

from mvsd import _native as nat
from mvsd.sample import rejection_sampler as rs
from mvsd.sample.sampler import Sampler
from mvsd.testing.spec_metadata import make_metadata
from mvsd.worker.gpu.sample.logprob import compute_topk_scores

pytestmark = pytest.mark.gpu


def reference(x, k, tokens, logits_mode=False):
    x = x.float()
    ids = torch.sort(x, dim=-1, descending=True, stable=True).indices[:, :k]
    ids = torch.cat([tokens.view(-1, 1), ids], dim=-1)
    lp = x.double() if logits_mode else torch.log_softmax(x.double(), dim=-1)
    ranks = (x >= x.gather(1, tokens.view(-1, 1))).sum(-1)
    return ids, lp.gather(1, ids), ranks


def check(x, k, tokens, logits_mode=False):
    got = compute_topk_scores(x, k, tokens, logits_mode=logits_mode)
    ids, lps, ranks = reference(x, k, tokens, logits_mode)
    assert torch.equal(got.logprob_token_ids, ids)
    assert torch.equal(got.selected_token_ranks, ranks)
    assert torch.allclose(got.logprobs.double(), lps, atol=2e-6, rtol=1e-6, equal_nan=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1, 7, 2047, 2048, 2049, 8191, 8193, 50257, 151936])
@pytest.mark.parametrize("n,k", [(1, 0), (3, 1), (5, 20), (2, 128)])
def test_chunk_edges(device, dtype, V, n, k):
    g = torch.Generator(device=device).manual_seed(V * 31 + n)
    x = (torch.randn(n, V, device=device, generator=g) * 2.5).to(dtype)
    tokens = torch.randint(0, V, (n,), device=device, generator=g)
    check(x, min(k, V), tokens)
    # a view whose rows start at an odd element and are not adjacent
    if V > 2:
        check(x[:, 1:], min(k, V - 1), tokens.clamp(max=V - 2))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [40961, 151936])
def test_long_chunks(device, dtype, V):
    """Enough rows for the 8192-column chunks."""
    g = torch.Generator(device=device).manual_seed(V)
    x = (torch.randn(210, V, device=device, generator=g) * 2.5).to(dtype)
    check(x, 20, torch.randint(0, V, (210,), device=device, generator=g))


@pytest.mark.parametrize("n", [1, 200])
@pytest.mark.parametrize("k", [1, 20, 128])
@pytest.mark.parametrize("logits_mode", [False, True])
def test_special_rows(device, n, k, logits_mode):
    V = 50257
    g = torch.Generator(device=device).manual_seed(k)
    rows = [torch.zeros(V, device=device), torch.full((V,), -3.0, device=device)]
    few = torch.full((V,), -math.inf, device=device)  # fewer finite entries than k
    few[[5, 4000, V - 1]] = torch.tensor([1.0, 2.0, 1.0], device=device)
    rows.append(few)
    cluster = torch.randn(V, device=device, generator=g)  # one chunk holds all large values
    cluster[8192:16384] += 50.0
    rows.append(cluster)
    rows.append((torch.randn(V, device=device, generator=g) * 2).round())  # long runs of ties
    x = torch.stack(rows).repeat(n, 1)
    check(x, k, torch.arange(x.shape[0], device=device) * 97 % V, logits_mode)


def test_nan_and_infinite_rows(device):
    """Raw order: NaN first; a NaN or +inf anywhere makes every log-softmax value NaN."""
    V = 9000
    x = torch.randn(3, V, device=device)
    x[0, 8500] = math.nan
    x[1, 3] = math.inf
    x[2] = -math.inf
    tokens = torch.tensor([7, 8, 9], device=device)
    check(x, 5, tokens)
    check(x, 5, tokens, logits_mode=True)


@pytest.mark.parametrize("scale,rank", [(1e-12, 3000), (1.0, None)])
def test_merged_logprobs(device, scale, rank):
    """The V1 order compares the fp32 log-softmax: values it merges tie and rank by index."""
    V, k = 3000, 9
    row = torch.arange(V, device=device, dtype=torch.float32) * (scale / V)
    logits = row.repeat(3, 1)
    meta = make_metadata([[1, 2]], device=device)
    sampled = torch.tensor([[10, 20, 30]], dtype=torch.int32, device=device)
    t = rs.RejectionSampler(Sampler())._get_logprobs_tensors(k, meta, logits, None, None, sampled)
    lp = (row - row.max()) - torch.logsumexp((row - row.max()).double(), 0).float()
    order = torch.sort(lp, descending=True, stable=True).indices[:k].to(torch.int32)
    if rank is not None:
        assert torch.equal(order, torch.arange(k, device=device, dtype=torch.int32))
        assert t.selected_token_ranks.tolist() == [rank] * 3
    assert torch.equal(t.logprob_token_ids[:, 1:], order.expand(3, -1))
    assert torch.equal(t.logprob_token_ids[:, 0], sampled.view(-1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_in_place_equal_gathered_rows(device, dtype):
    """Verify and bonus rows read from the compact logits in their own dtype (with padding
    positions reading the rows the clamp gives) equal the gathered fp32 rows."""
    V = 8200
    drafts = [[1, 2, 3], [], [4], [5, 6, 7, 8, 9], []]
    meta = make_metadata(drafts, device=device)
    rows = sum(len(d) + 1 for d in drafts)
    logits = (torch.randn(rows, V, device=device) * 2.5).to(dtype)
    sampled = torch.full((5, 6), -1, dtype=torch.int32, device=device)
    sampled[:, 0] = torch.tensor([11, 12, 13, 14, 15], device=device)
    sampler = rs.RejectionSampler(Sampler())
    here = sampler._get_logprobs_tensors(6, meta, logits, None, None, sampled)
    there = sampler._get_logprobs_tensors(
        6, meta, logits, logits[meta.target_logits_indices].float(),
        logits[meta.bonus_logits_indices].float(), sampled)
    assert torch.equal(here.logprob_token_ids, there.logprob_token_ids)
    assert torch.equal(here.selected_token_ranks, there.selected_token_ranks)
    # a 16-bit row's chunks sum in another order than the fp32 row's, which can move the log-sum
    # and each value (magnitude below 32) by one rounding: 2 * 2^-20
    assert (here.logprobs - there.logprobs).abs().max() <= 2 * 2.0 ** -20


@pytest.mark.parametrize("V", [33, 2049, 50257, 151936])
@pytest.mark.parametrize("k", [31, 32, 33])
def test_bound_of_64_or_256_unions(device, V, k):
    """The bound on the k-th largest comes from 64 unions of groups up to k = 32, from 256 above."""
    g = torch.Generator(device=device).manual_seed(V + k)
    x = torch.randn(5, V, device=device, generator=g) * 2.5
    x[1] = x[1].sort(descending=True).values  # the largest side by side in one chunk
    x[2, V // 2:] = -math.inf
    x[3] = x[3].round()
    check(x, k, torch.arange(5, device=device) * 5 % V)
    check(x, k, torch.arange(5, device=device) * 5 % V, logits_mode=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_row_indices_outside_the_logits_read_the_nearest_row(device, dtype):
    V = 4100
    meta = make_metadata([[1, 2], [], [3]], device=device)
    logits = (torch.randn(6, V, device=device) * 2.5).to(dtype)
    sampled = torch.tensor([[5, 6, 7], [8, -1, -1], [9, 10, -1]], dtype=torch.int32, device=device)
    sampler = rs.RejectionSampler(Sampler())
    tables = []
    for target, bonus in (([0, 1, 4], [0, 3, 5]), ([-1, 1, 4], [-2 ** 31, 3, 2 ** 31 - 1])):
        meta.target_logits_indices = torch.tensor(target, dtype=torch.int32, device=device)
        meta.bonus_logits_indices = torch.tensor(bonus, dtype=torch.int32, device=device)
        tables.append(sampler._get_logprobs_tensors(4, meta, logits, None, None, sampled))
    for want, got in zip(*(t[:3] for t in tables)):
        assert torch.equal(want, got)


@pytest.mark.parametrize("n,V,k,split", [
    (3, 1024, 128, True), (3, 1025, 20, False), (257, 1025, 20, True),   # fewer groups than k
    (5, 2048 * 6, 96, True), (5, 2048 * 6 - 1100, 96, False),             # as many, and one less
    (15, 16384, 128, True), (16, 16384, 128, False), (16, 17000, 128, True),                        # a sixteenth more
    (150, 50257, 128, True), (150, 50257, 20, True),                      # short, long chunks
    (1, 33, 33, True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_of_few_groups(device, dtype, n, V, k, split):
    """Where the groups of a row are few beside k: the lists kernel, shorter chunks, or the split
    path's own lists, all the same answers."""
    assert (nat.lib().mvsd_logprobs_workspace_bytes(n, V, k) > 0) == split
    g = torch.Generator(device=device).manual_seed(V + k)
    x = (torch.randn(n, V, device=device, generator=g) * 2.5).to(dtype)
    check(x, k, torch.arange(n, device=device) * 7 % V)
    check(x, k, torch.arange(n, device=device) * 7 % V, logits_mode=True)
