"""Sampling constraints with rows split over workgroups (mvsd_sampling_masks_split,
mvsd_apply_top_k_top_p_split) against the one-workgroup-per-row path (mvsd_sampling_masks,
mvsd_apply_top_k_top_p): both find the same first kept entry with the same exact integer sums, so
the masks are equal bit for bit."""

import math

import pytest
import torch

from mvsd import _native as nat
from mvsd.sample.metadata import SamplingMetadata
from mvsd.sample.ops.topk_topp_sampler import apply_top_k_top_p
from mvsd.sample.rejection_sampler import sampling_masks

pytestmark = pytest.mark.gpu


def general_masks(x, cu, rows, sm):
    masks = torch.full((rows.shape[0], 4), 7.0, device=x.device)
    args = nat.RejectionArgs(
        target_logits=x.data_ptr(), target_dtype=nat.dtype_code(x.dtype),
        target_stride=x.stride(0), target_rows=rows.data_ptr(), target_num_rows=x.shape[0],
        cu_num_draft_tokens=cu.data_ptr(), temperature=nat.ptr(sm.temperature), all_greedy=0,
        apply_temperature=1, batch_size=cu.shape[0], num_tokens=rows.shape[0],
        vocab_size=x.shape[1], top_k=nat.ptr(sm.top_k), top_p=nat.ptr(sm.top_p))
    nat.check(nat.lib().mvsd_sampling_masks(args, masks.data_ptr(), nat.stream_of(x.device)),
              "mvsd_sampling_masks")
    return masks


def make_rows(V, dtype, device, g):
    """One row of each kind a pass can go wrong on."""
    n = torch.randn(8, V, device=device, generator=g)
    rows = [n[0] * 2, n[1] * 6, n[2] * 0.05, torch.zeros(V, device=device),
            (n[3] * 3).round(), -n[4].abs() * 100, n[5] * 2 + 80]
    inf = n[6].clone()
    inf[V // 2] = math.inf
    nan = n[7].clone()
    nan[V - 1] = math.nan
    some = torch.full((V,), -math.inf, device=device)
    some[::max(1, V // 7)] = n[0][::max(1, V // 7)]
    peak = n[1] - 30
    peak[V // 3] = 20.0
    return torch.stack([*rows, inf, nan, some, torch.full((V,), -math.inf, device=device),
                        peak]).to(dtype)


def kinds_of(V):
    """(top-k or 0, top-p, temperature) of every class of row."""
    return [(0, 0.9, 0.8), (0, 0.3, 1.5), (0, 0.999, 1.0), (0, 1e-6, 0.7), (0, 0.0, 1.0),
            (1, 1.0, 0.8), (20, 1.0, 1.3), (50, 0.9, 0.8), (300, 0.5, 1.0), (600, 0.9, 1.0),
            (V - 1, 0.8, 0.9), (0, 0.9, 0.0), (0, 0.2, 0.0), (5, 0.5, 0.0), (5, 1.0, 0.0),
            (0, 1.0, 0.9), (0, 0.9, 1e-30), (3, 0.9, 1e25)]


def long_chunks(rows, V):
    """Whether a call takes 8192-column chunks (csrc/constraints.hip, split_chunk)."""
    return rows * -(-V // 8192) >= 300 or -(-V // 2048) > 256


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [65536, 65537, 73727, 151936, 524288])
def test_masks_equal_general_path(device, dtype, V):
    g = torch.Generator(device=device).manual_seed(V)
    x = make_rows(V, dtype, device, g)
    kinds = kinds_of(V)
    n = x.shape[0]
    # every kind on every row, the rows in another order for each request
    for part in (kinds[:9], kinds[9:]):  # at most 128 rows a call
        assert long_chunks(n * len(part), V)
        _compare(x, part, g)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [65536, 65537, 73727, 151936, 524288])
def test_masks_of_few_rows_equal_general_path(device, dtype, V):
    """The same kinds and rows in calls small enough for the 2048-column chunks; 524288 columns
    have the most chunks and groups of a row."""
    g = torch.Generator(device=device).manual_seed(V + 1)
    x = make_rows(V, dtype, device, g)
    kinds, n = kinds_of(V), x.shape[0]
    per_call = min(n, 299 // -(-V // 8192))  # rows
    for i in range(0, n, per_call):
        for kind in kinds:
            assert not long_chunks(per_call, V)
            _compare(x[i:i + per_call], [kind], g)


def _compare(x, kinds, g):
    device, n, V = x.device, x.shape[0], x.shape[1]
    rows = torch.cat([torch.randperm(n, device=device, generator=g) for _ in kinds]).to(torch.int32)
    assert rows.shape[0] <= 128
    cu = torch.arange(n, n * len(kinds) + 1, n, dtype=torch.int32, device=device)
    sm = SamplingMetadata(
        temperature=torch.tensor([t for _, _, t in kinds], device=device), all_greedy=False,
        all_random=False,
        top_k=torch.tensor([k or V for k, _, _ in kinds], dtype=torch.int64, device=device),
        top_p=torch.tensor([p for _, p, _ in kinds], device=device))
    for top_k, top_p in ((True, True), (False, True)):
        part = SamplingMetadata(temperature=sm.temperature, all_greedy=False, all_random=False,
                                top_k=sm.top_k if top_k else None,
                                top_p=sm.top_p if top_p else None)
        got = sampling_masks(x, cu, part, target_rows=rows)
        want = general_masks(x, cu, rows, part)
        same = (got.view(torch.int32) == want.view(torch.int32)).all(dim=1)
        bad = [(kinds[j // n], int(rows[j]), got[j].tolist(), want[j].tolist())
               for j in (~same).nonzero().view(-1).tolist()]
        assert not bad, bad[:5]


@pytest.mark.parametrize("n,V", [(3, 65536), (5, 65539), (100, 151936)])
def test_apply_in_place_equals_general_path(device, n, V):
    """Rows of a wider tensor (an odd stride), in place; the long chunks from 16 rows on."""
    g = torch.Generator(device=device).manual_seed(n)
    wide = torch.randn(n, V + 3, device=device, generator=g) * 2.5
    k = torch.randint(1, 200, (n,), device=device, generator=g)
    k[::3] = V
    p = torch.rand(n, device=device, generator=g)
    p[::4] = 1.0
    want = wide.clone()
    nat.check(nat.lib().mvsd_apply_top_k_top_p(
        want[:, 1:V + 1].data_ptr(), want.stride(0), k.data_ptr(), p.data_ptr(), n, V,
        nat.stream_of(device)), "mvsd_apply_top_k_top_p")
    apply_top_k_top_p(wide[:, 1:V + 1], k, p)
    assert torch.equal(wide, want)


@pytest.mark.parametrize("ties", [2, 300, 100000, 150000])
def test_greedy_ties_at_the_limit(device, ties):
    """Greedy rows of tied maxima whose mass below is within 3e-4 of what 1 - p takes: the first
    maximum is kept or masked as the exact sums say, also where a float sum of the ties (a multiple
    of 1/64 at 150000) is off by more."""
    V, n = 151936, 128
    # t (ties + below) = below + 1 + e, t = 1 - p a multiple of 2^-24
    t = (torch.linspace(1.2, 1.9 if ties == 2 else 4.0, n, dtype=torch.float64) / ties * 2 ** 24
         ).round() / 2 ** 24
    e = 3e-4 * (1 - 2 * (torch.arange(n) % 2))
    below = (t * ties - 1 - e) / (1 - t)
    x = torch.full((n, V), -math.inf, device=device)
    x[:, 500:500 + ties] = 0.0
    x[:, :20] = (below / 20).log().float().to(device)[:, None]
    cu = torch.arange(1, n + 1, dtype=torch.int32, device=device)
    rows = torch.arange(n, dtype=torch.int32, device=device)
    sm = SamplingMetadata(temperature=torch.zeros(n, device=device), all_greedy=False,
                          all_random=False, top_k=None, top_p=(1 - t).float().to(device))
    want = general_masks(x, cu, rows, sm)
    assert torch.equal((want[:, 0] > -math.inf).cpu(), e > 0)
    got = sampling_masks(x, cu, sm, target_rows=rows)
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))


def test_decreasing_counts_stay_inside_the_scratch(device):
    """Cumulative draft counts that decrease list rows more than once: the plan keeps to its
    room.  (The masks of such a batch mean nothing; the call reads and writes in bounds.)"""
    P, V, guard = 64, 65536, 1 << 20
    x = torch.randn(P, V, device=device)
    cu = torch.tensor([P if r % 2 == 0 else 0 for r in range(P)], dtype=torch.int32, device=device)
    ones = torch.ones(P, device=device)
    top_p, top_k = ones * 0.9, torch.full((P,), V, device=device)
    top_k[::3] = 20
    need = nat.lib().mvsd_constraints_scratch_bytes(P, V)
    buffer = torch.full((need + guard,), 0xA5, dtype=torch.uint8, device=device)
    masks = torch.empty(P + 64, 4, device=device).fill_(7.0)
    args = nat.RejectionArgs(
        target_logits=x.data_ptr(), target_dtype=nat.F32, target_stride=V, target_num_rows=P,
        cu_num_draft_tokens=cu.data_ptr(), temperature=ones.data_ptr(), all_greedy=0,
        apply_temperature=1, batch_size=P, num_tokens=P, vocab_size=V, top_k=top_k.data_ptr(),
        top_p=top_p.data_ptr())
    nat.check(nat.lib().mvsd_sampling_masks_split(args, masks.data_ptr(), buffer.data_ptr(), need,
                                                  nat.stream_of(x.device)),
              "mvsd_sampling_masks_split")
    assert (buffer[need:] == 0xA5).all() and (masks[P:] == 7.0).all()
