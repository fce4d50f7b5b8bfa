"""Which batches RejectionSampler.forward and Sampler.forward take a shorter route for, past the
steps of the general one."""

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from mvsd.sample import rejection_sampler as rs
from mvsd.sample import sampler as smp
from mvsd.sample.metadata import SamplingMetadata
from mvsd.sample.rejection_sampler import RejectionSampler
from mvsd.sample.sampler import Sampler, TopKTopPSampler, runs_own_steps

LIMITS = {"top_k": torch.tensor([5, 9])}
PENALTIES = {"no_penalties": False, "prompt_token_ids": [[1], [2]],
             "output_token_ids": [[], []], "spec_token_ids": [[3], [4, 5]]}
LOGPROBS = {"max_num_logprobs": 2}


def race_only(sampler, batch=LIMITS, *, rejection_sampler=RejectionSampler, counts=None):
    sm = SamplingMetadata(**{"temperature": torch.ones(2), "all_greedy": False,
                             "all_random": True, "top_k": None, "top_p": None, **batch})
    meta = SimpleNamespace(num_draft_tokens=[1, 2] if counts is None else counts)
    if not isinstance(rejection_sampler, RejectionSampler):
        rejection_sampler = rejection_sampler(sampler)
    return rejection_sampler._bonus_rows_race_only(meta, sm, torch.zeros(5, 16))


class OwnLimits(TopKTopPSampler):
    pass


class OwnSampler(Sampler):
    pass


class OwnProcessors(RejectionSampler):
    def apply_logits_processors(self, logits, sampling_metadata, metadata):
        return logits


def with_own_limits():
    sampler = Sampler()
    sampler.topk_topp_sampler = OwnLimits()
    return sampler


@pytest.mark.parametrize("batch", [LIMITS, PENALTIES, LOGPROBS, {**PENALTIES, **LIMITS}])
def test_a_replaced_sampler_is_used(batch):
    assert race_only(Sampler(), batch)
    assert not race_only(with_own_limits(), batch)
    assert not race_only(OwnSampler(), batch)
    assert not race_only(Sampler(), {**batch, "min_p": torch.tensor([0.1, 0.0])})


@pytest.mark.parametrize("batch", [LIMITS, PENALTIES, LOGPROBS])
@pytest.mark.parametrize("step", sorted(smp._STEPS))
def test_a_replaced_step_is_used(batch, step, monkeypatch):
    sampler = Sampler()
    setattr(sampler, step, lambda *args, **kw: None)
    assert not race_only(sampler, batch) and not runs_own_steps(sampler)
    monkeypatch.setattr(Sampler, step, lambda *args, **kw: None)
    assert not race_only(Sampler(), batch) and not runs_own_steps(Sampler())


@pytest.mark.parametrize("owner,name", [(smp, "apply_top_k_top_p"), (smp, "random_sample"),
                                        (TopKTopPSampler, "__call__")])
def test_a_replaced_function_of_the_sampler_is_used(owner, name, monkeypatch):
    assert race_only(Sampler()) and runs_own_steps(Sampler())
    monkeypatch.setattr(owner, name, lambda *args, **kw: None)
    assert not race_only(Sampler()) and not runs_own_steps(Sampler())


@pytest.mark.parametrize("batch", [LIMITS, PENALTIES, LOGPROBS])
def test_a_replaced_rejection_sample_is_used(batch, monkeypatch):
    monkeypatch.setattr(rs, "rejection_sample", lambda *args, **kw: None)
    assert not race_only(Sampler(), batch)
    assert race_only(Sampler(), {})  # the race-only batch calls it by its name


def test_replaced_processors_are_used(monkeypatch):
    assert not race_only(Sampler(), PENALTIES, rejection_sampler=OwnProcessors)
    assert race_only(Sampler(), LIMITS, rejection_sampler=OwnProcessors)  # not called there
    own = RejectionSampler(Sampler())
    own.apply_logits_processors = lambda *args: None
    assert not race_only(None, PENALTIES, rejection_sampler=own)
    for name in ("apply_sampling_constraints", "apply_top_k_top_p"):
        with monkeypatch.context() as m:
            m.setattr(rs, name, lambda *args: None)
            assert not race_only(Sampler(), PENALTIES)
    assert race_only(Sampler(), PENALTIES)


def test_batches_without_limits_race_whatever_the_logprobs_mode():
    assert race_only(with_own_limits(), {})
    assert race_only(Sampler("processed_logprobs"), {})
    assert not race_only(Sampler("processed_logprobs"), LIMITS)


@pytest.mark.parametrize("specs", [None, []])
def test_penalties_without_draft_lists(specs):
    assert not race_only(Sampler(), {**PENALTIES, "spec_token_ids": specs})


@pytest.mark.parametrize("counts", [np.array([1, 2]), [np.int64(1), 2], (1, 2)])
def test_draft_counts_of_any_integer_type(counts):
    assert race_only(Sampler(), PENALTIES, counts=counts)
    assert not race_only(Sampler(), {**PENALTIES, "spec_token_ids": [[3], [4]]}, counts=counts)
    assert not race_only(Sampler(), {**PENALTIES, "spec_token_ids": [[3]]}, counts=counts)


@pytest.mark.parametrize("shape", [(1,), (3,), (1, 1), (0,)])
def test_gather_logprobs_takes_one_token_per_row(shape):
    with pytest.raises(RuntimeError, match="shape"):
        Sampler.gather_logprobs(torch.zeros(2, 16), 1, torch.zeros(shape, dtype=torch.int64))


@pytest.mark.parametrize("rows", [None, torch.zeros(0, dtype=torch.int32)])
def test_no_rows_have_no_masks(rows):
    """A batch without requests is taken, with limits as without."""
    sm = SamplingMetadata(temperature=torch.ones(0), all_greedy=False, all_random=True,
                          top_k=torch.ones(0), top_p=torch.ones(0))
    logits = torch.zeros(0 if rows is None else 3, 16)
    assert smp.constraint_masks(logits, rows, sm) is None
