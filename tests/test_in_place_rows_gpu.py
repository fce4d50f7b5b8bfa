"""The sampler and RejectionSampler.forward on rows read in place (row masks, the masked race, raw
rows' logprobs) against the general path, which writes the rows' fp32 copy, its quotient by the
temperature and its masked entries: the same RNG state gives the same tokens, ids and ranks."""

import numpy as np
import pytest
import torch

from mvsd.sample import rejection_sampler as rs
from mvsd.sample import sampler as smp
from mvsd.sample.sampler import Sampler
from mvsd.testing.spec_metadata import make_metadata, sampling_metadata
from mvsd.worker.gpu.sample.logprob import compute_topk_scores

pytestmark = pytest.mark.gpu


class General(Sampler):
    """The sampler under another type, which takes the general path."""


def params(n, V, limits, greedy, g):
    temps = [0.0 if i % 4 < greedy else 0.5 + 0.1 * (i % 8) for i in range(n)]
    top_k = top_p = None
    if "k" in limits:
        top_k = [V if i % 3 == 0 else 1 + 17 * i % 200 for i in range(n)]
        top_k = [min(k, V) for k in top_k]
    if "p" in limits:
        top_p = [1.0 if i % 5 == 0 else 0.2 + 0.1 * (i % 8) for i in range(n)]
    return temps, top_k, top_p


def same(a, b, lp_atol):
    assert torch.equal(a.sampled_token_ids, b.sampled_token_ids)
    if b.logprobs_tensors is None:
        assert a.logprobs_tensors is None
        return
    ids, lps, ranks = a.logprobs_tensors[:3]
    want_ids, want_lps, want_ranks = b.logprobs_tensors[:3]
    assert torch.equal(ids, want_ids) and torch.equal(ranks, want_ranks)
    assert (lps - want_lps).abs().max() <= lp_atol


# logprob values: one fp32 sum in two orders moves the log-sum and then each value (magnitude
# below 32) by one rounding
LP_ATOL = 2 * 2.0 ** -20


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("limits", ["", "k", "p", "kp"])
@pytest.mark.parametrize("n,V,greedy", [(1, 9, 0), (6, 8193, 1), (5, 65537, 2), (129, 1000, 1),
                                        (4, 2049, 4)])
def test_sampler(device, dtype, limits, n, V, greedy):
    g = torch.Generator(device=device).manual_seed(V)
    logits = (torch.randn(n, V, device=device, generator=g) * 2.5).to(dtype)
    temps, top_k, top_p = params(n, V, limits, greedy, g)
    sm = sampling_metadata(temps, [[]] * n, device=device, top_k=top_k, top_p=top_p,
                           max_num_logprobs=min(5, V))
    for mode in ("raw_logprobs", "raw_logits"):
        outs = []
        for cls in (Sampler, General):
            torch.manual_seed(7)
            outs.append(cls(mode).forward(logits.clone(), sm))
        same(*outs, LP_ATOL)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("limits", ["k", "p", "kp"])
@pytest.mark.parametrize("V,B", [(4097, 6), (65600, 6), (66001, 40)])
@pytest.mark.parametrize("greedy", [0, 2])
def test_forward(device, dtype, limits, V, B, greedy):
    """40 requests pass the split path's 128 rows; fewer share one call for verify and bonus rows."""
    g = torch.Generator(device=device).manual_seed(V + B)
    host = torch.Generator().manual_seed(V)
    drafts = [torch.randint(0, V, (i % 5,), generator=host).tolist() for i in range(B)]
    meta = make_metadata(drafts, device=device)
    P = sum(len(d) for d in drafts)
    logits = (torch.randn(P + B, V, device=device, generator=g) * 2.5).to(dtype)
    probs = torch.softmax(torch.randn(P, V, device=device, generator=g) * 2.5, -1)
    temps, top_k, top_p = params(B, V, limits, greedy, g)
    sm = sampling_metadata(temps, drafts, device=device, top_k=top_k, top_p=top_p,
                           max_num_logprobs=3)
    outs = []
    for cls in (Sampler, General):
        torch.manual_seed(11)
        outs.append(rs.RejectionSampler(cls()).forward(meta, probs, logits.clone(), sm))
    same(*outs, LP_ATOL)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("limits", ["", "kp"])
@pytest.mark.parametrize("V,B,greedy", [(500, 7, 0), (65600, 6, 2), (3001, 5, 4), (700, 1, 0)])
def test_forward_with_penalties(device, dtype, limits, V, B, greedy):
    """Verify and bonus rows penalised in one launch against the general path's two."""
    g = torch.Generator(device=device).manual_seed(V + B)
    host = torch.Generator().manual_seed(V)
    tokens = lambda n: torch.randint(0, min(V, 60), (n,), generator=host).tolist()
    drafts = [tokens((i + 1) % 5) for i in range(B)]
    meta = make_metadata(drafts, device=device)
    P = sum(len(d) for d in drafts)
    logits = (torch.randn(P + B, V, device=device, generator=g) * 2.5).to(dtype)
    probs = torch.softmax(torch.randn(P, V, device=device, generator=g) * 2.5, -1)
    temps, top_k, top_p = params(B, V, limits, greedy, g)
    sm = sampling_metadata(
        temps, drafts, device=device, top_k=top_k, top_p=top_p, max_num_logprobs=3,
        no_penalties=False, prompt_token_ids=[tokens(20 * i) for i in range(B)],
        output_token_ids=[tokens(9 * (B - i)) for i in range(B)],
        presence_penalties=[0.3 * (i % 3) for i in range(B)],
        frequency_penalties=[0.2 * (i % 2) for i in range(B)],
        repetition_penalties=[1.0 + 0.3 * (i % 4) for i in range(B)])
    before = logits.clone()
    outs = []
    for cls in (Sampler, General):
        torch.manual_seed(11)
        outs.append(rs.RejectionSampler(cls()).forward(meta, probs, logits, sm))
    same(*outs, LP_ATOL)
    assert torch.equal(logits, before)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("limits", ["", "kp"])
@pytest.mark.parametrize("overlap", ["one row", "shifted"])
def test_overlapping_rows(device, dtype, limits, overlap):
    """Rows nearer than a row's length (an expanded row, a sliding view) are copied, not refused."""
    n, V = 5, 1000
    base = (torch.randn(2 * V, device=device) * 2.5).to(dtype)
    logits = (base[:V].expand(n, V) if overlap == "one row" else base.as_strided((n, V), (3, 1)))
    temps, top_k, top_p = params(n, V, limits, 1, None)
    sm = sampling_metadata(temps, [[]] * n, device=device, top_k=top_k, top_p=top_p,
                           max_num_logprobs=4)
    outs = []
    for rows in (logits, logits.clone(memory_format=torch.contiguous_format)):
        torch.manual_seed(3)
        outs.append(Sampler().forward(rows, sm))
    same(*outs, LP_ATOL)
    if dtype != torch.float32:
        tokens = torch.arange(n, device=device)
        got, want = (compute_topk_scores(rows, 4, tokens) for rows in (logits, logits.float()))
        assert torch.equal(got.logprob_token_ids, want.logprob_token_ids)
        assert torch.equal(got.selected_token_ranks, want.selected_token_ranks)
        assert (got.logprobs - want.logprobs).abs().max() <= LP_ATOL


def test_noise_of_any_layout(device, monkeypatch):
    """A replaced noise function may return any strides, as random_sample takes them."""
    n, V = 4, 1000
    logits = (torch.randn(n, V, device=device) * 2.5).to(torch.bfloat16)
    sm = sampling_metadata([1.0] * n, [[]] * n, device=device, top_k=[7] * n)
    noise = torch.empty(V, n, device=device).exponential_()
    outs = []
    for given in (noise.t(), noise.t().contiguous()):
        monkeypatch.setattr(smp, "generate_sampler_noise", lambda *args: given)
        outs.append(Sampler().forward(logits, sm))
    same(*outs, 0.0)


@pytest.mark.parametrize("form", ["no draft lists", "array of counts"])
def test_forward_with_penalties_in_other_forms(device, form):
    V, drafts = 500, [[3, 4], [], [5]]
    meta = make_metadata(drafts, device=device)
    logits = torch.randn(6, V, device=device) * 2.5
    sm = sampling_metadata([1.0, 0.0, 0.7], drafts, device=device, no_penalties=False,
                           prompt_token_ids=[[1, 2]] * 3, output_token_ids=[[3], [4, 4], []],
                           presence_penalties=[0.5] * 3)
    if form == "no draft lists":
        sm.spec_token_ids = None
    else:
        meta.num_draft_tokens = np.array(meta.num_draft_tokens)
    outs = []
    for cls in (Sampler, General):
        torch.manual_seed(11)
        outs.append(rs.RejectionSampler(cls()).forward(meta, None, logits, sm))
    same(*outs, 0.0)


def test_forward_calls_a_replaced_rejection_sample(device, monkeypatch):
    """A batch without limits races its bonus rows, then calls rejection_sample by its name, with
    the arguments it had before there were limits on that route."""
    V, drafts = 300, [[3], []]
    meta = make_metadata(drafts, device=device)
    logits = torch.randn(3, V, device=device)
    real, seen = rs.rejection_sample, []

    def replacement(*args, synthetic_mode, synthetic_conditional_rates, uniform_probs, exp_noise,
                    target_rows, apply_temperature):
        seen.append(args)
        return real(*args, uniform_probs=uniform_probs, exp_noise=exp_noise,
                    target_rows=target_rows, apply_temperature=apply_temperature)

    outs = []
    for function in (real, replacement):
        monkeypatch.setattr(rs, "rejection_sample", function)
        torch.manual_seed(2)
        outs.append(rs.RejectionSampler(Sampler()).forward(
            meta, None, logits, sampling_metadata([1.0, 0.6], drafts, device=device)))
    same(*outs, 0.0)
    assert len(seen) == 1
