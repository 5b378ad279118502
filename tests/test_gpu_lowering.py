"""Rows under penalties that only lower (csrc/select_lowering.h) against the oracle, where that
select changes its form: rows whose leading ids were all drawn before (none of them may enter the
bound), flat and peaked rows with a row sum, more listed ids above the bound than the queue holds
(the slice is taken again), more chunks of listed ids than the notes hold (the bitmap is walked),
rows that start inside a group of eight ids, and the map of listed ids however it was written.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import lily_sampler as LS
import lily_workloads as W
import oracle as O
from gpu_util import check_row_against_oracle, dev, o_params, run_rows
from test_gpu_stream import make_sampler


@pytest.fixture(scope="module", params=[1, 3], ids=lambda s: f"slices{s}")
def sampler(request):
    s = make_sampler(request.param)
    yield s
    s.close()


def _logits(rng, rows, vocab, flat, bf16):
    x = rng.normal(0.0, 2.0, (rows, vocab))
    if not flat:
        heavy = rng.random((rows, vocab)) < 0.1
        x = np.where(heavy, rng.standard_t(3.0, (rows, vocab)) * 4.0, x)
    x = x.astype(np.float32)
    return W.to_bf16_bits(x) if bf16 else x


def _scratch(sampler, rng, vocab, ids, how):
    """A scratch that counted `ids` 1 to 6 times each, the first 40 of them many times."""
    counts = np.zeros(vocab, dtype=np.uint32)
    counts[ids] = rng.integers(1, 7, len(ids))
    counts[ids[:40]] += rng.integers(0, 120, len(ids[:40])).astype(np.uint32)
    sc = LS.SamplerScratch(sampler, vocab)
    if how == "history":
        hist = rng.permutation(np.repeat(np.arange(vocab), counts)).astype(np.int32)
        sc.add_history(torch.from_numpy(hist).to(dev()))
        return sc, counts
    sc.write_counts(torch.from_numpy(counts.view(np.int32)))
    if how == "copy":
        other = LS.SamplerScratch(sampler, vocab)
        other.add_history(torch.arange(min(vocab, 500), dtype=torch.int32, device=dev()))
        other.copy_counts_from(sc)
        return other, counts
    return sc, counts


# 8 192 bf16 / 4 096 f32 ids are a block; an odd vocabulary starts its rows anywhere in eight ids.
@pytest.mark.parametrize("vocab", [997, 8192, 16_384 + 1, 40_005, 151_936])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("flat", [False, True])
def test_rows_whose_leading_ids_were_drawn_before(sampler, vocab, bf16, flat):
    rng = np.random.default_rng(vocab * 4 + 2 * bf16 + flat)
    cases = [(0, "history"), (40, "history"), (700, "write"), (3000, "copy"), (20_000, "write")]
    rows = len(cases)
    x = _logits(rng, rows, vocab, flat, bf16)
    xf = W.bf16_bits_to_f32(x) if bf16 else x
    scratch, counts = [], []
    for r, (n, how) in enumerate(cases):
        leading = np.argsort(-xf[r], kind="stable")[:min(n, vocab - 1)]
        sc, c = _scratch(sampler, rng, vocab, leading, how)
        scratch.append(sc)
        counts.append(c)
    kw = [dict(temperature=[0.7, 1.0, 0.4][r % 3], top_k=[50, 64, 3][r % 3], top_p=0.95, min_p=0.01, repetition_penalty=1.1,
               presence_penalty=0.3, frequency_penalty=[0.2, 0.02][r % 2], seed=70 + r) for r in range(rows)]
    stats = torch.zeros(4, dtype=torch.int32, device=dev())
    for logprobs in (False, True):
        sampler.set_path_stats(stats)
        for step in range(2):
            r = run_rows(sampler, x, kw, [step] * rows, scratch=scratch, logprobs=logprobs)
            for i in range(rows):
                d = O.sample(xf[i], counts[i], o_params(**kw[i]), step, want_logprob=True)
                check_row_against_oracle(r, i, d)
                if logprobs:
                    assert abs(r.logprobs[i] - d.logprob) <= 1e-5 * max(1.0, abs(d.logprob)), (i, r.logprobs[i], d.logprob)
        sampler.set_path_stats(None)
    # Every slice by the streaming selects (the smallest row aside: its slices hold few more ids than k).
    if vocab > 997:
        assert stats[2].item() == 0, stats.tolist()
    for i in range(rows):
        assert np.array_equal(scratch[i].read_counts().numpy().view(np.uint32), counts[i])
        scratch[i].close()


# One block a slice (8 192 bf16 / 4 096 f32 ids, and less than a whole one), either side of the shares
# of elements above the sum's cut - seven eighths with enough of them far up, 31 / 32 - from which on
# a slice is taken as a flat one.
@pytest.mark.parametrize("share", [0.0, 0.5, 0.87, 0.88, 0.96, 0.968, 0.97, 0.98, 1.0])
@pytest.mark.parametrize("short,far_up", [(0, 1.0), (0, 0.002), (517, 1.0)])
@pytest.mark.parametrize("bf16", [False, True])
def test_slices_of_one_block_at_the_share_that_counts_as_flat(sampler, share, short, far_up, bf16):
    slices = sampler.slices_for(1, 20, 1 << 20, bf16)
    vocab = (8192 if bf16 else 4096) * slices - short
    rng = np.random.default_rng(int(1000 * share) + bf16)
    rows, temperature = 8, 0.4
    # the cut lies (log2(V) + 21) T ln 2 below the largest value: 20 - 9.3 ... 9.9
    x = rng.uniform(-9.0, 8.0, (rows, vocab)).astype(np.float32)
    above = rng.permuted(np.tile(np.arange(vocab) < share * vocab, (rows, 1)), axis=1)
    # (the upper quarter of the way to 20 begins at 17.5)
    up = rng.random((rows, vocab)) < far_up
    x[above] = np.where(up, rng.uniform(11.5, 19.0, (rows, vocab)), rng.uniform(11.5, 17.0, (rows, vocab)))[above]
    x[:, 77] = 20.0
    x = W.to_bf16_bits(x) if bf16 else x
    xf = W.bf16_bits_to_f32(x) if bf16 else x
    scratch, counts = zip(*[_scratch(sampler, rng, vocab, np.argsort(-xf[r], kind="stable")[5:5 + 60 * r], "write")
                            for r in range(rows)])
    kw = [dict(temperature=temperature, top_k=20, top_p=0.95, repetition_penalty=1.05, presence_penalty=0.1,
               frequency_penalty=0.01, seed=r) for r in range(rows)]
    r = run_rows(sampler, x, kw, [3] * rows, scratch=list(scratch), logprobs=True)
    for i in range(rows):
        d = O.sample(xf[i], counts[i], o_params(**kw[i]), 3, want_logprob=True)
        check_row_against_oracle(r, i, d)
        assert abs(r.logprobs[i] - d.logprob) <= 1e-5 * max(1.0, abs(d.logprob)), (i, r.logprobs[i], d.logprob)
        scratch[i].close()


# Slices of 10 to 19 blocks (one of 7 with three slices) whose share of elements above the sum's cut
# brings the notes from a tenth of their place to all of it within four blocks.
@pytest.mark.parametrize("share", [0.02, 0.04, 0.06, 0.08, 0.1, 0.14, 0.3, 0.6, 0.86])
@pytest.mark.parametrize("bf16", [False, True])
def test_notes_that_fill_up_are_handed_over_before_they_overflow(sampler, share, bf16):
    vocab, rows, temperature = (151_936 if bf16 else 80_004), 4, 0.4
    rng = np.random.default_rng(int(1000 * share) + bf16)
    # the cut lies (log2(V) + 21) T ln 2 = 10.4 ... 10.6 below the largest value, which block 0 holds
    x = rng.uniform(-9.0, 8.0, (rows, vocab)).astype(np.float32)
    above = rng.random((rows, vocab)) < share
    # (thinning out upwards: the queue of chunks above the k-th value is not what fills)
    x[above] = np.minimum(11.5 + rng.exponential(0.7, int(above.sum())), 19.9).astype(np.float32)
    x[:, 77] = 20.0
    x = W.to_bf16_bits(x) if bf16 else x
    xf = W.bf16_bits_to_f32(x) if bf16 else x
    scratch, counts = zip(*[_scratch(sampler, rng, vocab, rng.permutation(vocab)[:500 * r], "write") for r in range(rows)])
    kw = [dict(temperature=temperature, top_k=20, top_p=0.95, repetition_penalty=1.05, presence_penalty=0.1,
               frequency_penalty=0.01, seed=r) for r in range(rows)]
    stats = torch.zeros(4, dtype=torch.int32, device=dev())
    sampler.set_path_stats(stats)
    r = run_rows(sampler, x, kw, [3] * rows, scratch=list(scratch), logprobs=True)
    sampler.set_path_stats(None)
    for i in range(rows):
        d = O.sample(xf[i], counts[i], o_params(**kw[i]), 3, want_logprob=True)
        check_row_against_oracle(r, i, d)
        assert abs(r.logprobs[i] - d.logprob) <= 1e-5 * max(1.0, abs(d.logprob)), (i, r.logprobs[i], d.logprob)
        scratch[i].close()
    # every slice by the streaming select, none of them twice (which would leave a reason here)
    assert stats.tolist()[1:] == [0, 0, 0], stats.tolist()
