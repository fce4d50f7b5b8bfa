"""Which batches RejectionSampler.forward takes its bonus tokens for without the caller's sampler."""

from types import SimpleNamespace

import pytest
import torch

from mvsd.sample.metadata import SamplingMetadata
from mvsd.sample.rejection_sampler import RejectionSampler
from mvsd.sample.sampler import Sampler, TopKTopPSampler


def race_only(sampler, **kw):
    sm = SamplingMetadata(temperature=torch.ones(2), all_greedy=False, all_random=True,
                          top_k=torch.tensor([5, 9]), top_p=None, **kw)
    meta = SimpleNamespace(num_draft_tokens=[1, 2])
    return RejectionSampler(sampler)._bonus_rows_race_only(meta, sm, torch.zeros(5, 16))


def test_a_replaced_top_k_top_p_sampler_is_used():
    class Own(TopKTopPSampler):
        pass

    class OwnSampler(Sampler):
        pass

    plain, own = Sampler(), Sampler()
    own.topk_topp_sampler = Own()
    assert race_only(plain)
    assert not race_only(own)
    assert not race_only(OwnSampler())
    assert not race_only(plain, min_p=torch.tensor([0.1, 0.0]))


@pytest.mark.parametrize("shape", [(1,), (3,), (1, 1), (0,)])
def test_gather_logprobs_takes_one_token_per_row(shape):
    with pytest.raises(RuntimeError, match="shape"):
        Sampler.gather_logprobs(torch.zeros(2, 16), 1, torch.zeros(shape, dtype=torch.int64))
