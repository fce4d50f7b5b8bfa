"""Rows at any element alignment take the vector loads: verification (V1, V2) and the bonus race on
rows of an odd vocabulary, or starting at an odd element of a wider tensor, equal the same rows in
an aligned tensor.  The values are the same and the work is split by columns only, so the outputs
are equal."""

import pytest
import torch

from mvsd.sample.metadata import SamplingMetadata
from mvsd.sample.rejection_sampler import rejection_sample
from mvsd.sample.sampler import race_rows
from mvsd.worker.gpu.spec_decode import rejection_sample as v2_rejection_sample

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def moved(x, V, offset, pad):
    """The same values as rows x[..., :V] of a tensor with an odd start and row length."""
    out = torch.zeros((*x.shape[:-1], offset + V + pad), dtype=x.dtype, device=x.device)
    out[..., offset:offset + V] = x[..., :V]
    return out[..., offset:offset + V]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V", [5, 2049, 16384 + 3, 50257])
@pytest.mark.parametrize("greedy", [0, 1, 2])
def test_verify(device, dtype, V, greedy):
    g = torch.Generator(device=device).manual_seed(V)
    B, k = 6, 3
    P = B * k
    wide = (V + 7) // 8 * 8
    logits = (torch.randn(P, wide, device=device, generator=g) * 2).to(dtype)
    probs = torch.softmax(torch.randn(P, V, device=device, generator=g) * 2, -1)
    noise = torch.empty(B, wide, device=device).exponential_(generator=g)
    drafts = torch.randint(0, V, (P,), device=device, generator=g, dtype=torch.int32)
    drafts[::2] = logits[::2, :V].float().argmax(-1).to(torch.int32)
    temps = torch.full((B,), 0.8, device=device)
    if greedy == 1:
        temps[::2] = 0
    sm = SamplingMetadata(temperature=temps, all_greedy=greedy == 2, all_random=greedy == 0,
                          top_k=None, top_p=None)
    u = torch.rand(P, dtype=torch.float64, device=device, generator=g).clamp_min(1e-9)
    cu = torch.arange(k, P + 1, k, dtype=torch.int32, device=device)
    bonus = torch.arange(B, dtype=torch.int32, device=device).view(B, 1) % V
    outs = []
    for x, e in ((logits[:, :V], noise[:, :V]), (moved(logits, V, 1, 2), moved(noise, V, 3, 0))):
        outs.append(rejection_sample(drafts, [k] * B, k, cu, probs, x, bonus, sm, uniform_probs=u,
                                     exp_noise=e, apply_temperature=True))
    assert torch.equal(*outs)
    index = torch.tensor([0, P - 1, 3], dtype=torch.int32, device=device)
    picks = [race_rows(x, index, e[:3], temps[:3]) for x, e in
             ((logits[:, :V], noise[:, :V]), (moved(logits, V, 1, 2), moved(noise, V, 3, 0)))]
    assert torch.equal(*picks)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("V", [5, 4097, 50257])
@pytest.mark.parametrize("block", [False, True])
def test_v2(device, dtype, V, block):
    g = torch.Generator(device=device).manual_seed(V)
    B, K = 5, 3
    rows = B * (K + 1)
    wide = (V + 7) // 8 * 8
    target = (torch.randn(rows, wide, device=device, generator=g) * 2).to(dtype)
    draft = (torch.randn(B, K, wide, device=device, generator=g) * 2).to(dtype)
    temps = torch.full((B,), 0.8, device=device)
    temps[1] = 0
    ar = torch.arange(B, dtype=torch.int32, device=device)
    args = dict(draft_sampled=torch.randint(0, V, (rows,), device=device, generator=g,
                                            dtype=torch.int32),
                cu_num_logits=torch.arange(0, rows + 1, K + 1, dtype=torch.int32, device=device),
                pos=torch.arange(rows, device=device) + 100, idx_mapping=ar,
                expanded_idx_mapping=ar.repeat_interleave(K + 1),
                expanded_local_pos=torch.arange(K + 1, dtype=torch.int32, device=device).repeat(B),
                temperature=temps, seed=torch.arange(B, device=device) + 5,
                num_speculative_steps=K, use_block_verification=block)
    outs = []
    for t, d in ((target[:, :V], draft[..., :V]), (moved(target, V, 1, 2), moved(draft, V, 3, 0))):
        sampled, count = v2_rejection_sample(target_logits=t, draft_logits=d, **args)
        valid = torch.arange(K + 1, device=device) < count.view(-1, 1)
        outs.append((torch.where(valid, sampled, -1), count))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
