"""Rows that draw among many candidates (k > 64; a request without top_k gets the reference's cap
of 1024, src/kernels/sample.rs:17 and :326-331) through the launches that spread such a
row over as many workgroups as a row of few candidates: a bound from the lanes' maxima, then
the values that reach it.

Ids, candidates, probabilities and kept counts bit-exact against the oracle, the
log-probability within 1e-5 (relative, floor 1), the counts of penalised ids as the oracle
leaves them.  Which way a launch went shows in the path statistics: a row drawn this way adds
one to its entry, a row drawn by the other kernels one per workgroup.
"""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import lily_sampler as LS
import lily_workloads as W
import oracle as O
from gpu_util import check_row_against_oracle, dev, o_params, run_rows

LOGPROB_RTOL = 1e-5


@pytest.fixture(scope="module")
def sampler():
    s = LS.Sampler(0)
    yield s
    s.close()


def _with_stats(sampler, fn):
    stats = torch.zeros(4, dtype=torch.int32, device=dev())
    sampler.set_path_stats(stats)
    try:
        out = fn()
    finally:
        sampler.synchronize()
        sampler.set_path_stats(None)
    return out, stats.cpu().numpy()


def _check_logprob(got, want, what):
    if np.isfinite(want):
        assert abs(got - want) <= LOGPROB_RTOL * max(1.0, abs(want)), (what, got, want)
    else:
        assert got == -np.inf, what


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("use_plan", [False, True], ids=["inline", "plan"])
def test_plain_rows_of_many_candidates(sampler, bf16, use_plan):
    """Rows of every k above the streaming select's, heavy tails, a row with fewer finite
    values than k, a vocabulary that leaves partial chunks at both ends of the slices."""
    rng = np.random.default_rng(71 + bf16)
    rows, vocab = 5, 151_937 if not bf16 else 151_939
    x = (rng.standard_t(5, (rows, vocab)) * 2.5).astype(np.float32)
    x[2, rng.random(vocab) < 0.997] = -np.inf          # ~450 finite values: fewer than k
    x[4, rng.integers(0, vocab, 2000)] = -np.inf
    if bf16:
        x = W.to_bf16_bits(x)
    assert sampler.slices_for(rows, 1024, vocab) > 1
    for trial, k in enumerate((0, 65, 200, 777)):
        kw = [dict(temperature=0.7 + 0.1 * r, top_k=k, top_p=0.95, min_p=0.01, seed=300 + r) for r in range(rows)]
        r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [trial] * rows, logprobs=True,
                                                         use_plan=use_plan))
        assert stats[0] == 0 and stats[1] + stats[2] == rows, stats   # one count a row: the two launches
        for i in range(rows):
            d = O.sample(x[i], None, o_params(**kw[i]), trial, want_logprob=True)
            check_row_against_oracle(r, i, d)
            _check_logprob(r.logprobs[i], d.logprob, (k, i))


def test_prefix_sums_that_leave_their_binade_and_round_on_ties(sampler):
    """The left-to-right f32 sums of up to 1 024 weights are formed 64 at a time by integer
    additions while the running sum stays in one binade and no weight lies exactly half a last
    place above a multiple of it, and by the chain of real additions otherwise.  Rows that force
    either way: hundreds of ids at the row's largest value (weights of exactly 1: the sum walks
    through nine binades on integers), a flat row (the sum crosses a binade every few blocks and
    weights within a few binades of the sum tie often), a peaked row (one binade, no ties after
    the first block), and steps of one bf16 ulp (weights in a handful of exact ratios).  The
    kept counts and the probabilities are bit-exact against the oracle, so is every draw."""
    rng = np.random.default_rng(4242)
    vocab = 151_936
    x = np.empty((4, vocab), dtype=np.float32)
    x[0] = rng.normal(0, 1, vocab)
    x[0, rng.choice(vocab, 700, replace=False)] = 9.0
    x[1] = rng.normal(0, 0.05, vocab)
    x[2] = rng.normal(0, 1, vocab)
    x[2, 77] = 30.0
    x[3] = np.round(rng.normal(0, 3, vocab) * 8) / 8
    for trial, (t, top_p) in enumerate(((1.0, 0.999), (0.7, 0.9), (1.3, 0.97))):
        kw = [dict(temperature=t, top_k=0, top_p=top_p, seed=900 + r) for r in range(4)]
        r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [trial] * 4, logprobs=True))
        assert stats[0] == 0 and stats[1] + stats[2] == 4, stats
        for i in range(4):
            d = O.sample(x[i], None, o_params(**kw[i]), trial, want_logprob=True)
            check_row_against_oracle(r, i, d)
            _check_logprob(r.logprobs[i], d.logprob, (trial, i))


def test_penalised_rows_over_decode_steps(sampler):
    """Lowering penalties (repetition >= 1, presence and frequency >= 0) on the ids that matter
    most: the lanes' maxima, the row's sum and the candidates are taken on penalised worth.
    Three steps, the counts moving with the draws; a last call with a penalty that may raise
    a value goes the other kernels' way and draws what the oracle draws as well."""
    rng = np.random.default_rng(72)
    rows, vocab = 4, 151_936
    x = rng.normal(0, 3, (rows, vocab)).astype(np.float32)
    kw = [dict(temperature=0.6, top_k=0, top_p=0.95, min_p=0.0, seed=77 + r, repetition_penalty=1.2,
               presence_penalty=0.4, frequency_penalty=0.3) for r in range(rows)]
    scratch, counts = [], []
    for r in range(rows):
        best = np.argsort(-x[r])[:400].astype(np.int32)
        hh = np.concatenate([rng.integers(0, vocab, 3000).astype(np.int32), np.repeat(best[:40], 5), best])
        sc = LS.SamplerScratch(sampler, vocab)
        sc.add_history(torch.from_numpy(hh).to(dev()))
        scratch.append(sc)
        counts.append(np.bincount(hh, minlength=vocab).astype(np.uint32))
    for step in range(3):
        r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [step] * rows, scratch=scratch,
                                                         logprobs=True, use_plan=step == 1))
        assert stats[1] == rows and stats[2] == 0, stats
        for i in range(rows):
            d = O.sample(x[i], counts[i], o_params(**kw[i]), step, want_logprob=True)   # bumps the counts
            check_row_against_oracle(r, i, d)
            _check_logprob(r.logprobs[i], d.logprob, (step, i))
    kw[1] = dict(kw[1], repetition_penalty=0.8)
    r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [3] * rows, scratch=scratch, logprobs=True))
    assert stats[1] > rows, stats
    for i in range(rows):
        d = O.sample(x[i], counts[i], o_params(**kw[i]), 3, want_logprob=True)
        check_row_against_oracle(r, i, d)
    for i in range(rows):
        assert np.array_equal(scratch[i].read_counts().numpy().view(np.uint32), counts[i]), i
        scratch[i].close()


def test_more_values_at_the_bound_than_the_list_holds(sampler):
    """A constant row, a row of a few distinct values and a row in ascending order: every lane's
    maximum ties or the bound lets most of the row through, the row's list overflows, and the
    workgroup that finishes the row takes the select that is right for any input."""
    rng = np.random.default_rng(73)
    rows, vocab = 4, 100_003
    x = rng.normal(0, 1, (rows, vocab)).astype(np.float32)
    x[0, :] = 0.25
    x[1] = rng.integers(-1, 2, vocab) / 4.0
    x[2] = np.linspace(-3, 3, vocab, dtype=np.float32)
    kw = [dict(temperature=1.1, top_k=0, top_p=0.99, min_p=0.0, seed=9 + r) for r in range(rows)]
    r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [5] * rows, logprobs=True))
    assert stats[2] >= 2 and stats[1] + stats[2] == rows, stats
    for i in range(rows):
        d = O.sample(x[i], None, o_params(**kw[i]), 5, want_logprob=True)
        check_row_against_oracle(r, i, d)
        _check_logprob(r.logprobs[i], d.logprob, i)


def test_sixty_four_rows_and_the_way_of_the_other_kernels(sampler):
    """64 bf16 rows at k = 1024 (8 or 16 workgroups a row: the bound is then the median of the
    lanes' maxima); the same call on a sampler that has this way switched off draws the same."""
    c = W.config4(rows=64)
    x = c["logits"]
    rows, vocab = x.shape
    kw = c["params"]
    r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [2] * rows, logprobs=True))
    assert stats[1] == rows and stats[2] == 0, stats
    old = os.environ.get("LILY_SAMPLER_WIDE")
    os.environ["LILY_SAMPLER_WIDE"] = "0"
    try:
        other = LS.Sampler(0)
    finally:
        if old is None:
            os.environ.pop("LILY_SAMPLER_WIDE", None)
        else:
            os.environ["LILY_SAMPLER_WIDE"] = old
    try:
        r2, stats2 = _with_stats(other, lambda: run_rows(other, x, kw, [2] * rows, logprobs=True))
    finally:
        other.close()
    assert stats2[1] > rows, stats2
    assert np.array_equal(r.ids, r2.ids) and np.array_equal(r.cand_ids, r2.cand_ids)
    assert np.all(np.abs(r.logprobs - r2.logprobs) <= LOGPROB_RTOL * np.maximum(1.0, np.abs(r2.logprobs)))   # (the rows' sums are grouped differently)
    for i in range(0, rows, 7):
        d = O.sample(x[i], None, o_params(**kw[i]), 2, want_logprob=True)
        check_row_against_oracle(r, i, d)
        _check_logprob(r.logprobs[i], d.logprob, i)


def test_random_launches_of_rows_of_many_candidates(sampler):
    """Forty seeded launches: 1 to 23 rows, vocabularies that leave partial chunks at the slices'
    ends, f32 and bf16, k from 65 to 1024, Gaussian, heavy-tailed and peaked rows, rows that are
    mostly -inf, lowering penalties over histories that hold the rows' best ids, with and
    without a log-probability, as a call and as a plan."""
    rng = np.random.default_rng(2024)
    went = 0
    for case in range(40):
        rows = int(rng.integers(1, 24))
        vocab = int(rng.choice([32_003, 50_021, 100_003, 151_936, 151_937, 151_939, 200_001]))
        bf16 = bool(rng.integers(0, 2))
        k = int(rng.choice([0, 65, 100, 300, 777, 1024]))
        pen, logprob, use_plan = (bool(rng.integers(0, 2)) for _ in range(3))
        kind = int(rng.integers(0, 3))
        if kind == 0:
            x = rng.normal(0, 3, (rows, vocab)).astype(np.float32)
        elif kind == 1:
            x = (rng.standard_t(3, (rows, vocab)) * 2).astype(np.float32)
        else:
            x = rng.normal(0, 0.5, (rows, vocab)).astype(np.float32)
            x[:, rng.integers(0, vocab, 50)] += 12.0
        if rng.integers(0, 4) == 0:
            x[rng.integers(0, rows), rng.random(vocab) < 0.99] = -np.inf
        xf = x
        if bf16:
            x = W.to_bf16_bits(x)
            xf = W.bf16_bits_to_f32(x)
        kw = []
        for r in range(rows):
            d = dict(temperature=float(rng.uniform(0.3, 1.5)), top_k=k, top_p=float(rng.choice([0.8, 0.95, 1.0])),
                     min_p=float(rng.choice([0.0, 0.01])), seed=int(rng.integers(0, 1 << 30)))
            if pen:
                d.update(repetition_penalty=float(rng.choice([1.0, 1.1, 1.5])),
                         presence_penalty=float(rng.choice([0.0, 0.5])),
                         frequency_penalty=float(rng.choice([0.0, 0.2])))
            kw.append(d)
        scratch = counts = None
        if pen:
            scratch, counts = [], []
            for r in range(rows):
                best = np.argsort(-xf[r])[:int(rng.integers(10, 600))].astype(np.int32)
                hh = np.concatenate([rng.integers(0, vocab, int(rng.integers(0, 5000))).astype(np.int32),
                                     np.repeat(best[:20], int(rng.integers(1, 6))), best])
                sc = LS.SamplerScratch(sampler, vocab)
                sc.add_history(torch.from_numpy(hh).to(dev()))
                scratch.append(sc)
                counts.append(np.bincount(hh, minlength=vocab).astype(np.uint32))
        step = int(rng.integers(0, 100))
        r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [step] * rows, scratch=scratch,
                                                         logprobs=logprob, use_plan=use_plan))
        went += int(stats[1] + stats[2] == rows)
        for i in range(rows):
            d = O.sample(x[i], counts[i] if pen else None, o_params(**kw[i]), step, want_logprob=logprob)
            check_row_against_oracle(r, i, d)
            if logprob:
                _check_logprob(r.logprobs[i], d.logprob, (case, i))
        if pen:
            for i in range(rows):
                assert np.array_equal(scratch[i].read_counts().numpy().view(np.uint32), counts[i]), (case, i)
                scratch[i].close()
    assert went >= 30, went   # (a launch of one or two rows has too few slices for some k)


@pytest.mark.parametrize("rows,vocab,bf16", [(1, 32_003, True), (4, 40_001, False), (8, 248_320, False), (26, 151_936, False),
                                             (27, 151_936, False), (53, 151_937, True), (54, 151_937, True)])
def test_bounds_over_the_slices(sampler, rows, vocab, bf16):
    """Rows without top_k either side of the most workgroups that one launch takes (26 and 27 rows in 38
    slices, 53 and 54 in 19), in slices cut finer than a block, and in the most slices there are: rows of Gaussian
    logits, which need no exhaustive select; the best 1 100 all in the row's first ids, or spread evenly; all but a contiguous
    seventh -inf, so that most waves have nothing to name; penalties on the best."""
    rng = np.random.default_rng(rows + vocab)
    x = rng.normal(0, 2, (rows, vocab)).astype(np.float32)
    kw = [dict(temperature=0.8, top_k=0, top_p=0.97, seed=700 + r) for r in range(rows)]
    checked = sorted({0, rows // 2, rows - 1})
    fmt = W.to_bf16_bits if bf16 else lambda a: a
    xs = fmt(x)
    r, stats = _with_stats(sampler, lambda: run_rows(sampler, xs, kw, [1] * rows, logprobs=True))
    assert stats[0] == 0 and stats[1] == rows and stats[2] == 0, stats
    for i in checked:
        d = O.sample(xs[i], None, o_params(**kw[i]), 1, want_logprob=True)
        check_row_against_oracle(r, i, d)
        _check_logprob(r.logprobs[i], d.logprob, i)
    for i in range(rows):
        if i % 3 == 0:
            x[i, :1100] += 9.0
        elif i % 3 == 1:
            x[i, :vocab // 3] = -np.inf
            x[i, vocab // 3 + vocab // 7:] = -np.inf
        else:
            x[i, ::vocab // 1100] += 9.0
    xs = fmt(x)
    hist = [np.argsort(-x[i])[:300].astype(np.int32) for i in range(rows)]
    scratch, counts = [], [np.bincount(hh, minlength=vocab).astype(np.uint32) for hh in hist]
    for hh in hist:
        sc = LS.SamplerScratch(sampler, vocab)
        sc.add_history(torch.from_numpy(hh).to(dev()))
        scratch.append(sc)
    pkw = [dict(k, repetition_penalty=1.2, presence_penalty=0.5) if i % 2 else k for i, k in enumerate(kw)]
    r, stats = _with_stats(sampler, lambda: run_rows(sampler, xs, pkw, [2] * rows, scratch=scratch, logprobs=True))
    assert stats[0] == 0 and stats[1] + stats[2] == rows, stats
    for i in sorted({*checked, min(1, rows - 1), min(2, rows - 1)}):
        d = O.sample(xs[i], counts[i], o_params(**pkw[i]), 2, want_logprob=True)
        check_row_against_oracle(r, i, d)
        _check_logprob(r.logprobs[i], d.logprob, i)


@pytest.mark.parametrize("rows,vocab,bf16", [(32, 32_003, True), (33, 32_003, True), (64, 32_003, False), (70, 66_585, True), (40, 9_001, False),
                                             (128, 66_585, True)])
def test_bounds_over_fewer_slices(sampler, rows, vocab, bf16):
    """The same where short rows are cut for four lanes to each of the k (512 workgroups) and for two, in one launch
    and, past 1 024 workgroups, in two."""
    test_bounds_over_the_slices(sampler, rows, vocab, bf16)


@pytest.mark.parametrize("looks", ["0,8192", "8192,0", "1,1"], ids=["no key", "no maxima", "one look"])
@pytest.mark.parametrize("rows,bf16", [(2, False), (6, False), (6, True), (20, True)])
def test_slices_that_stop_waiting_for_each_other(monkeypatch, rows, bf16, looks):
    """A launch whose slices look for the words of their rows' other slices never, or once, in either wait (the second one
    belongs to rows with too many waves of -inf), in workgroups of sixteen waves (up to 128 of them) and of four: the rows go to the
    exhaustive select, and the next launch of the same sampler finds every word as it has to be."""
    vocab = 151_937
    rng = np.random.default_rng(rows + bf16)
    x = rng.normal(0, 2, (rows, vocab)).astype(np.float32)
    x[1::2, :vocab // 4] = -np.inf
    x[1::2, vocab // 4 + vocab // 2:] = -np.inf
    x = W.to_bf16_bits(x) if bf16 else x
    kw = [dict(temperature=0.8, top_k=0, top_p=0.97, seed=40 + r) for r in range(rows)]
    monkeypatch.setenv("LILY_SAMPLER_WIDE_LOOKS", looks + ",1")
    s = LS.Sampler(0)
    gave_up = {"0,8192": (rows, rows), "8192,0": (rows // 2, rows // 2), "1,1": (0, rows)}[looks]
    for launch, (least, most) in enumerate((gave_up, (0, 0), (0, 0))):
        xs = x if launch < 2 else np.roll(x, 1, axis=0)   # (the rows that are half -inf change places with the others)
        r, stats = _with_stats(s, lambda: run_rows(s, xs, kw, [launch] * rows, logprobs=True, use_plan=rows > 8))
        assert stats[0] == 0 and stats[1] + stats[2] == rows and least <= stats[2] <= most, (launch, stats)
        for i in range(rows):
            d = O.sample(xs[i], None, o_params(**kw[i]), launch, want_logprob=True)
            check_row_against_oracle(r, i, d)
            _check_logprob(r.logprobs[i], d.logprob, (launch, i))
    s.close()


@pytest.mark.parametrize("rows", [1, 4, 40], ids=["sixteen waves", "one launch", "two launches"])
def test_values_that_share_a_quotient(sampler, rows):
    """Thousands of ids at 1.75 and at the float below it, whose quotients by the temperature are the same: the ids decide,
    whichever value the bound is."""
    vocab = 151_936
    rng = np.random.default_rng(rows)
    value, temperature = np.float32(1.75), np.float32(0.75)
    below = np.nextafter(value, np.float32(0))
    assert value / temperature == below / temperature
    x = rng.random((rows, vocab)).astype(np.float32) * np.float32(0.5)
    at = np.sort(rng.choice(vocab, 3600, replace=False))
    x[:, at[::2]], x[:, at[1::2]] = below, value
    if rows > 1:
        x[-1, at] = np.where(np.arange(3600) < 1800, below, value)
    kw = [dict(temperature=0.75, top_k=0, top_p=1.0, seed=8 + r) for r in range(rows)]
    r, stats = _with_stats(sampler, lambda: run_rows(sampler, x, kw, [3] * rows))
    assert stats[0] == 0 and stats[1] == rows and stats[2] == 0, stats
    for i in sorted({0, rows - 1}):
        check_row_against_oracle(r, i, O.sample(x[i], None, o_params(**kw[i]), 3))


@pytest.mark.parametrize("masked", [False, True], ids=["two-launches", "merged-slices"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_sort_of_many_candidates(sampler, bf16, masked):
    """The sort by counted bins where it can go wrong: candidates on both sides of zero, all below
    it, an outlier that puts all others into one bin and a range past the
    largest float (the radix select takes over), a bin of
    just as many equal values as a bin may hold and one more, fewer than k candidates, and k just
    above 64.  `masked`: about 3 000 allowed ids a row, whose four slices are merged."""
    rng = np.random.default_rng(77 + bf16)
    vocab = 151_936
    x = np.full((8, vocab), -np.inf, dtype=np.float32)
    some = rng.choice(vocab, 3000, replace=False)
    x[0, some] = rng.normal(0, 1, 3000)
    x[1, some] = -rng.random(3000) - 0.25
    x[2, some] = rng.normal(3, 1, 3000)
    x[2, some[0]] = 1.0e30
    x[3, some] = rng.normal(0, 1, 3000)
    x[3, some[1]] = 2.2e38
    x[3, some[2]] = -2.2e38
    x[4, some] = 1.0 + np.arange(3000) / 4096.0
    x[4, some[500:628]] = 1.5
    x[5] = x[4]
    x[5, some[628]] = 1.5
    x[6, some[:400]] = rng.normal(2, 3, 400)
    x[7, some] = rng.standard_t(3, 3000) * 4
    if bf16:
        x = W.to_bf16_bits(x)
    allow = np.zeros((8, (vocab + 31) // 32), dtype=np.uint32)
    np.bitwise_or.at(allow, (slice(None), some >> 5), (1 << (some & 31)).astype(np.uint32))
    for trial, k in enumerate((0, 65, 700)):
        kw = [dict(temperature=1.0, top_k=k, top_p=0.98, seed=500 + r) for r in range(8)]
        r = run_rows(sampler, x, kw, [trial] * 8, allow=allow if masked else None, logprobs=True)
        for i in range(8):
            d = O.sample(x[i], None, o_params(**kw[i]), trial, allow=allow[i] if masked else None, want_logprob=True)
            check_row_against_oracle(r, i, d)
            _check_logprob(r.logprobs[i], d.logprob, (k, i))


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_sort_with_more_empty_places_than_candidates(sampler, bf16):
    """Masked rows whose four slices hand over some 375 candidates each in 1 024 places, so that most
    of what the sort is given is empty: candidates so close together that an empty place's distance
    from them, in bins, is past any integer, and on both sides of zero, where it is no number."""
    rng = np.random.default_rng(79 + bf16)
    vocab, n = 151_936, 1500
    x = np.full((3, vocab), -np.inf, dtype=np.float32)
    some = rng.choice(vocab, n, replace=False)
    x[0, some] = 3.0 + rng.permutation(n).astype(np.float32) * 2.0 ** -22    # (one f32 step apart)
    x[1, some] = -1.0 - rng.permutation(n).astype(np.float32) * 2.0 ** -14
    x[2, some] = rng.normal(0, 1, n)
    if bf16:
        x = W.to_bf16_bits(x)
    allow = np.zeros((3, (vocab + 31) // 32), dtype=np.uint32)
    np.bitwise_or.at(allow, (slice(None), some >> 5), (1 << (some & 31)).astype(np.uint32))
    kw = [dict(temperature=1.0, top_k=0, top_p=0.98, seed=600 + r) for r in range(3)]
    r = run_rows(sampler, x, kw, [0] * 3, allow=allow)
    for i in range(3):
        check_row_against_oracle(r, i, O.sample(x[i], None, o_params(**kw[i]), 0, allow=allow[i]))


@pytest.mark.parametrize("masked", [False, True], ids=["one launch", "masked"])
@pytest.mark.parametrize("n", [1200, 3000, 8200])
def test_sort_by_sixteen_waves(sampler, n, masked):
    """The sort of sixteen waves on values around zero: outliers on both sides, infinities, values near zero with one
    outlier (they share a bin, which is sorted by exchanges with what precedes it), 300 equal ones ahead of the rest, behind the
    best and across the k-th, all equal.  `masked`: so many allowed ids; else about as many as reach the row's
    bound, of a launch over one row."""
    rng = np.random.default_rng(n)
    vocab = 151_936
    some = rng.choice(vocab, n, replace=False)
    x = np.full((8, vocab), -np.inf, dtype=np.float32)
    x[:, some] = rng.normal(0, 1, (8, n))
    x[0, some[:6]] = 300, -300, 80, 2.0e38, -2.0e38, -80
    x[1, some[:2]] = np.inf, 50
    x[2, some] *= 1.0e-4
    x[2, some[0]] = 0.9
    order = some[np.argsort(-x[3, some])]
    x[3, order[:300]] = 5.0
    x[4, some[np.argsort(-x[4, some])][100:400]] = 1.0e-3
    x[5, some[np.argsort(-x[5, some])][900:1200]] = 0.0
    x[6, some] = 1.0
    x[7, some] = rng.standard_t(2, n) * 4
    allow = np.zeros((8, (vocab + 31) // 32), dtype=np.uint32)
    np.bitwise_or.at(allow, (slice(None), some >> 5), (1 << (some & 31)).astype(np.uint32))
    for trial, k in enumerate((0, 300)):
        kw = [dict(temperature=1.0, top_k=k, top_p=0.99, seed=700 + i) for i in range(8)]
        whole = run_rows(sampler, x, kw, [trial] * 8, allow=allow) if masked else None
        for i in range(8):
            d = O.sample(x[i], None, o_params(**kw[i]), trial, allow=allow[i] if masked else None)
            if masked:
                check_row_against_oracle(whole, i, d)
            else:
                check_row_against_oracle(run_rows(sampler, x[i:i + 1], kw[i:i + 1], [trial]), 0, d)


@pytest.mark.parametrize("rows,vocab,bf16", [(1, 50_257, True), (2, 60_001, False), (6, 50_257, True), (6, 151_936, False), (60, 151_936, True)])
@pytest.mark.parametrize("pen", [False, True], ids=["plain", "penalties"])
def test_clusters_of_many_candidates(sampler, rows, vocab, bf16, pen):
    """More values at the row's bound than its list holds, by sixteen waves, by four, behind one launch and two: clusters of neighbours
    that lead by far, one value everywhere, all but a few of one value, rows that fall all along; k of 1 024, 700 and 65."""
    rng = np.random.default_rng(rows + vocab)
    x = rng.normal(0, 2, (rows, vocab)).astype(np.float32)
    kinds = 6
    for i in range(rows):
        kind = (i + (0 if rows > 1 else 1)) % kinds
        if kind == 0:
            x[i, 300:6300] += 9.0
        elif kind == 1:
            x[i, vocab // 2:vocab // 2 + 9000] += 9.0
        elif kind == 2:
            x[i, :] = 1.5
        elif kind == 3:
            x[i, 7:] = -2.0
        elif kind == 4:
            x[i] = -np.sort(-x[i])
        else:
            x[i, 100:100 + vocab // 3] += 5.0
    xs = W.to_bf16_bits(x) if bf16 else x
    more = dict(repetition_penalty=1.1, presence_penalty=0.25, frequency_penalty=0.125) if pen else {}
    for trial, k in enumerate((0, 700, 65)):
        kw = [dict(temperature=0.75, top_k=k, top_p=0.99, seed=900 + i, **more) for i in range(rows)]
        hist = rng.integers(0, 8000, (rows, 600)).astype(np.int32)
        scratch = None
        if pen:
            scratch = []
            for i in range(rows):
                sc = LS.SamplerScratch(sampler, vocab)
                sc.add_history(torch.from_numpy(hist[i]).to(dev()))
                scratch.append(sc)
        r = run_rows(sampler, xs, kw, [trial] * rows, scratch=scratch, logprobs=True, use_plan=trial == 1)
        for i in range(min(rows, 2 * kinds)):
            counts = np.bincount(hist[i], minlength=vocab).astype(np.uint32) if pen else None
            d = O.sample(xs[i], counts, o_params(**kw[i]), trial, want_logprob=True)
            check_row_against_oracle(r, i, d)
            _check_logprob(r.logprobs[i], d.logprob, (k, i))
        for sc in scratch or []:
            sc.close()
