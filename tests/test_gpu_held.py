"""Rows of few candidates in slices that a workgroup holds in registers (rows_held.hip), a block at a time
(rows_blocks.hip, LILY_SAMPLER_HELD=blocks) and through the streaming selects (LILY_SAMPLER_HELD=0): sizes around a block and two (4 096 / 8 192 f32
ids, twice that in bf16), rows that start inside a 16-byte piece, penalties of either sign over sparse and
dense histories, masks and bias lists, ties by the thousand, NaN and infinite logits, forced ids, drafts
longer than a wave.  Bit-exact against the oracle; log-probabilities at the bar of the other tests."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import lily_sampler as LS
import lily_workloads as W
import oracle as O
from gpu_util import both_params, check_row_against_oracle, dev, o_params, run_rows

ROWS = 8


def _sampler(monkeypatch, held, slices=0):
    monkeypatch.setenv("LILY_SAMPLER_HELD", held)
    monkeypatch.setenv("LILY_SAMPLER_SLICES", str(slices))
    return LS.Sampler(0)


def _rows(rng, vocab, bf16):
    x = rng.normal(0, 3, (ROWS, vocab)).astype(np.float32)
    x[1] = 1.5                                                        # one value: ties by the thousand
    x[2] = np.round(x[2])
    x[3, rng.random(vocab) < 0.998] = -np.inf
    x[4, rng.random(vocab) < 0.3] = np.nan
    x[5, vocab // 2:vocab // 2 + 300] = np.linspace(20, 21, len(x[5, vocab // 2:vocab // 2 + 300]), dtype=np.float32)
    x[6] = -np.inf
    return W.to_bf16_bits(x) if bf16 else x


def _check(r, x, kw, step, lp, counts=None, **ext):
    clean = np.where(np.isnan(x), -np.inf, x) if x.dtype == np.float32 else x.copy()
    if x.dtype == np.uint16:
        clean[(clean & 0x7fff) > 0x7f80] = 0xff80
    for i in range(len(x)):
        own = {k: v[i] for k, v in ext.items() if v[i] is not None and not (k == "bias" and not v[i])}
        d = O.sample(clean[i], None if counts is None else counts[i], o_params(**kw[i]), step, want_logprob=lp, **own)
        if "forced" in own:
            assert r.ids[i] == own["forced"]
        else:
            check_row_against_oracle(r, i, d)
        if lp and np.isfinite(d.logprob):
            assert abs(r.logprobs[i] - d.logprob) <= 1e-5 * max(1.0, abs(d.logprob)), (i, r.logprobs[i], d.logprob)


@pytest.mark.parametrize("held", ["1", "blocks", "0"], ids=["held", "blocks", "streamed"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("vocab", [1, 9, 4097, 8190, 16_381, 24_601, 65_543, 131_099])
def test_plain_rows(monkeypatch, held, bf16, vocab):
    rng = np.random.default_rng(vocab)
    x = _rows(rng, vocab, bf16)
    for slices in (0, max(1, vocab * (1 if bf16 else 2) // 16_384)):   # one block a slice, and about two
        s = _sampler(monkeypatch, held, slices)
        for trial, k in enumerate((2, 20, 64)):
            kw = [dict(temperature=0.7, top_k=k, top_p=0.97, min_p=0.01, seed=60 + i) for i in range(ROWS)]
            for lp in (False, True):
                for use_plan in (False, True):   # (a plan's rows may go a block at a time)
                    _check(run_rows(s, x, kw, [trial] * ROWS, logprobs=lp, use_plan=use_plan), x, kw, trial, lp)
        s.close()


@pytest.mark.parametrize("held", ["1", "blocks", "0"], ids=["held", "blocks", "streamed"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("history", [40, 3000, 60_000])
def test_rows_under_penalties(monkeypatch, held, bf16, history):
    vocab = 40_009
    rng = np.random.default_rng(history)
    x = _rows(rng, vocab, bf16)
    for slices in (0, 3 if bf16 else 6, 1):
        s = _sampler(monkeypatch, held, slices)
        hist = rng.integers(0, vocab, (ROWS, history)).astype(np.int32)
        hist[:, :history // 2] = rng.integers(0, 50, (ROWS, history // 2))
        for pen in (dict(repetition_penalty=1.1, presence_penalty=0.3, frequency_penalty=0.0625),
                    dict(repetition_penalty=0.9, presence_penalty=-0.5, frequency_penalty=0.03125)):
            for lp in (False, True):
                sc, counts = [], []
                for i in range(ROWS):
                    t = LS.SamplerScratch(s, vocab)
                    t.add_history(torch.from_numpy(hist[i]).to(dev()))
                    sc.append(t)
                    counts.append(np.bincount(hist[i], minlength=vocab).astype(np.uint32))
                kw = [dict(temperature=0.8, top_k=33, top_p=0.95, seed=7 + i, **pen) for i in range(ROWS)]
                r = run_rows(s, x, kw, [4] * ROWS, scratch=sc, logprobs=lp, use_plan=True)
                _check(r, x, kw, 4, lp, counts)
                for i in range(ROWS):
                    assert np.array_equal(sc[i].read_counts().numpy(), counts[i]), i   # (the oracle counted its draw)
                    sc[i].close()
        s.close()


@pytest.mark.parametrize("held", ["1", "blocks", "0"], ids=["held", "blocks", "streamed"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_rows_with_masks_bias_lists_and_forced_ids(monkeypatch, held, bf16):
    vocab = 50_021
    rng = np.random.default_rng(5)
    x = _rows(rng, vocab, bf16)
    x[4] = x[0]
    allow = np.stack([W.allow_mask(rng, vocab, frac=f) for f in (0.0005, 0.02, 0.02, 0.1, 0.1, 0.5, 0.02, 0.9)])
    bias = [[(int(i), float(d)) for i, d in zip(rng.integers(0, vocab, 30), rng.choice([-5.0, 5.0, 0.5], 30))]
            for _ in range(ROWS)]
    bias[0] += [(0, 4.0), (vocab - 1, 4.0), (vocab - 1, 4.0)]
    bias[7] = []
    forced = [None] * ROWS
    forced[3] = 77
    for slices in (0, 4 if bf16 else 7):
        s = _sampler(monkeypatch, held, slices)
        hist = rng.integers(0, vocab, (ROWS, 2000)).astype(np.int32)
        for use in (dict(allow=True), dict(bias=True), dict(allow=True, bias=True, forced=True, pen=True)):
            pen = dict(repetition_penalty=1.2, presence_penalty=0.1, frequency_penalty=0.2) if use.get("pen") else {}
            for lp in (False, True):
                sc = counts = None
                if pen:
                    sc, counts = [], []
                    for i in range(ROWS):
                        t = LS.SamplerScratch(s, vocab)
                        t.add_history(torch.from_numpy(hist[i]).to(dev()))
                        sc.append(t)
                        counts.append(np.bincount(hist[i], minlength=vocab).astype(np.uint32))
                kw = [dict(temperature=0.8, top_k=50, top_p=0.95, seed=9 + i, **pen) for i in range(ROWS)]
                ext = dict(allow=allow if use.get("allow") else None, bias=bias if use.get("bias") else None,
                           forced=forced if use.get("forced") else None)
                r = run_rows(s, x, kw, [1] * ROWS, scratch=sc, logprobs=lp, **ext)
                _check(r, x, kw, 1, lp, counts, **{k: v for k, v in ext.items() if v is not None})
        s.close()


@pytest.mark.parametrize("held", ["1", "blocks", "0"], ids=["held", "blocks", "streamed"])
@pytest.mark.parametrize("draft_k", [20, 0], ids=["20 drafted from", "all drafted from"])
def test_verify_pass(monkeypatch, held, draft_k):
    """Drafts from 20 and from 1 024 candidates (the latter's distribution is longer than a wave), verified
    among 20, three rows a pass with the acceptance behind them."""
    s = _sampler(monkeypatch, held)
    rng = np.random.default_rng(3)
    v, m = 30_011, 3
    head = rng.normal(0, 1.2, (m, v)).astype(np.float32)
    trunk = (head + rng.normal(0, 0.4, (m, v))).astype(np.float32)
    t_head, t_trunk = torch.from_numpy(head).to(dev()), torch.from_numpy(trunk).to(dev())
    lp, op = both_params(temperature=1.0, top_k=20, top_p=0.95, seed=77)
    dp = LS.SamplingParams.greedy(temperature=1.0, top_k=draft_k, top_p=1.0, seed=77)
    dop = O.params(temperature=1.0, top_k=draft_k, top_p=1.0, seed=77)
    scratch, dists = LS.SamplerScratch(s, v), LS.DraftDists(s, m)
    ids = torch.zeros(m, dtype=torch.int32, device=dev())
    out = torch.zeros(m, dtype=torch.int32, device=dev())
    ctrl = torch.zeros(LS.ctrl_words(m - 1), dtype=torch.int32, device=dev())
    outcomes = set()
    for step in range(0, 60, m):
        for j in range(m - 1):
            s.sample_draft_f32(t_head[j], scratch, dp, LS.draft_step(step + j), ids[j + 1:j + 2], dists.slot(j))
        s.spec_verify(t_trunk, scratch, lp, step, dists, ids, out, ctrl, pos0=10, ratio=4, chain=m - 1)
        s.synchronize()
        drafted, got = ids.cpu().numpy(), out.cpu().numpy()
        for j in range(m - 1):
            d = O.sample(head[j], None, dop, O.lib().lo_draft_step(step + j))
            assert drafted[j + 1] == d.chosen
            p_ids, p_pr = O.kept(trunk[j], op)
            q_ids, q_pr = O.kept(head[j], dop)
            want, acc, zero, gap = O.spec(p_ids, p_pr, q_ids, q_pr, int(drafted[j + 1]), op.seed, step + j)
            assert zero or got[j] == want, (step, j)
            outcomes.add(acc)
        assert got[m - 1] == O.sample(trunk[m - 1], None, op, step + m - 1).chosen
        acc = 0
        while acc + 1 < m and got[acc] == drafted[acc + 1]:
            acc += 1
        assert int(ctrl.cpu()[0]) == acc
    assert outcomes == {True, False}
    scratch.close()
    dists.close()
    s.close()


@pytest.mark.parametrize("held", ["1", "0"], ids=["masked", "other"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("vocab", [33, 2051, 70_001])
def test_masked_rows_of_many_candidates(monkeypatch, held, bf16, vocab):
    """A workgroup a row over the mask's words (rows_masked.hip), and the selects it replaces: masks that admit
    nothing, a few ids, what the sort holds (8 192) and a little more, and nearly all (left to the
    launch behind); equal values by the thousand; bias lists, penalties and a forced id; inline and from a table."""
    rng = np.random.default_rng(vocab)
    rows = 9
    x = np.concatenate([_rows(rng, vocab, False), rng.normal(0, 2, (1, vocab)).astype(np.float32)])
    x[4] = x[0]
    x[6] = x[7]
    allow = np.zeros((rows, (vocab + 31) // 32), dtype=np.uint32)
    for i, admitted in enumerate((0.02, 0.05, 0.13, 0.6, 8192 / vocab, 8300 / vocab, 0.0, 0.97, 0.3)):
        ids = np.flatnonzero(rng.random(vocab) < admitted)
        if i in (4, 5):
            ids = rng.choice(vocab, min(vocab, 8192 + 108 * (i - 4)), replace=False)
        np.bitwise_or.at(allow[i], ids >> 5, (1 << (ids & 31)).astype(np.uint32))
    bias = [[(int(i), float(d)) for i, d in zip(rng.integers(0, vocab, 30), rng.choice([-5.0, 5.0, 0.5], 30))]
            for _ in range(rows)]
    bias[2] = []
    forced = [None] * rows
    forced[0] = 1
    xs = W.to_bf16_bits(x) if bf16 else x
    s = _sampler(monkeypatch, held)
    hist = rng.integers(0, vocab, (rows, 700)).astype(np.int32)
    for trial, (k, lp, few) in enumerate(((0, True, False), (300, False, True), (65, True, True))):
        sc, counts = [], []
        for i in range(rows):
            t = LS.SamplerScratch(s, vocab)
            t.add_history(torch.from_numpy(hist[i]).to(dev()))
            sc.append(t)
            counts.append(np.bincount(hist[i], minlength=vocab).astype(np.uint32))
        n = 8 if few else rows   # (up to eight rows travel with the launch)
        kw = [dict(temperature=0.8, top_k=k, top_p=0.95, seed=9 + i, repetition_penalty=1.2, presence_penalty=0.1,
                   frequency_penalty=0.2) for i in range(n)]
        ext = dict(allow=allow[:n], bias=bias[:n], forced=(forced if lp else [None] * rows)[:n])
        r = run_rows(s, xs[:n], kw, [trial] * n, scratch=sc[:n], logprobs=lp, **ext)
        _check(r, xs[:n], kw, trial, lp, counts[:n], **ext)
        for t in sc:
            t.close()
    s.close()


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("vocab", [9001, 70_001, 262_144])
@pytest.mark.parametrize("run", [1, 96], ids=["one by one", "in runs"])
def test_masks_that_scatter_and_masks_that_cluster(monkeypatch, bf16, vocab, run):
    """Masks of a few ids, just what the sort and the list of ids hold and one more, as many words as the rule for
    clusters takes and some more, all ids; scattered ids and runs, over every kind of row: equal values by the
    thousand, mostly and wholly -inf, NaN; bias lists, penalties and a forced id."""
    rng = np.random.default_rng(vocab + run)
    x = _rows(rng, vocab, False)
    xs = W.to_bf16_bits(x) if bf16 else x
    words = (vocab + 31) // 32
    masks = np.zeros((ROWS, words), dtype=np.uint32)
    most = 32 * (350 + vocab // 170)
    for i, n in enumerate((3, 8191, 8193, 16_384, 16_385, most - 64, most + 64, vocab)):
        n = min(n, vocab)
        if run == 1 or n == vocab:
            ids = rng.choice(vocab, n, replace=False)
        else:
            starts = np.sort(rng.choice(vocab // run, min(-(-n // run), vocab // run), replace=False)) * run
            ids = (starts[:, None] + np.arange(run)).ravel()[:n]
        np.bitwise_or.at(masks[i], ids >> 5, (1 << (ids & 31)).astype(np.uint32))
    bias = [[(int(i), float(d)) for i, d in zip(rng.integers(0, vocab, 30), rng.choice([-5.0, 5.0, 0.5], 30))]
            for _ in range(ROWS)]
    hist = rng.integers(0, vocab, (ROWS, 2000)).astype(np.int32)
    pen = dict(repetition_penalty=1.2, presence_penalty=0.1, frequency_penalty=0.2)
    s = _sampler(monkeypatch, "1")
    for trial in range(ROWS):
        lp = trial % 2 == 0
        allow = np.roll(masks, trial, axis=0)
        kw = [dict(temperature=0.8, top_k=200 if trial % 4 == 3 else 0, top_p=0.95, seed=9 + i, **(pen if trial % 4 == 2 else {}))
              for i in range(ROWS)]
        sc = counts = None
        if trial % 4 == 2:
            sc, counts = [], []
            for i in range(ROWS):
                t = LS.SamplerScratch(s, vocab)
                t.add_history(torch.from_numpy(hist[i]).to(dev()))
                sc.append(t)
                counts.append(np.bincount(hist[i], minlength=vocab).astype(np.uint32))
        ext = dict(allow=allow, bias=bias if trial % 3 else [[]] * ROWS,
                   forced=[i if trial == 4 and i % 2 else None for i in range(ROWS)])
        r = run_rows(s, xs, kw, [trial] * ROWS, scratch=sc, logprobs=lp, use_plan=trial % 4 == 1, **ext)
        _check(r, xs, kw, trial, lp, counts, **ext)
        for t in sc or []:
            t.close()
    s.close()


@pytest.mark.parametrize("slices", [40, 64])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_more_slices_than_a_wave_merges(monkeypatch, bf16, slices):
    """205 rows a block at a time, k = 64, asked for in more slices than one wave merges (2 048 entries a row):
    every id of the row can be drawn all the same."""
    vocab, rows = 131_099, 205
    rng = np.random.default_rng(slices)
    x = rng.normal(0, 3, (rows, vocab)).astype(np.float32)
    x = W.to_bf16_bits(x) if bf16 else x
    s = _sampler(monkeypatch, "1", slices)
    kw = [dict(temperature=0.7, top_k=64, top_p=0.97, seed=60 + i) for i in range(rows)]
    for lp in (False, True):
        _check(run_rows(s, x, kw, [5] * rows, logprobs=lp, use_plan=True), x, kw, 5, lp)
    s.close()


def test_row_beyond_four_gibibytes(monkeypatch):
    """An f32 row of more than 2^30 ids in a plan: its bytes are not counted in 32 bits."""
    vocab = (1 << 30) + 4099
    s = _sampler(monkeypatch, "1")
    x = torch.randn(1, vocab, dtype=torch.float32, device=dev())
    best = [(1 << 30) + 7, vocab - 1, 5]
    for at, value in zip(best, (22.0, 21.5, 21.0)):
        x[0, at] = value
    out = torch.full((1,), -1, dtype=torch.int32, device=dev())
    ids = torch.full((1, LS.SAMPLE_K_CAP), -1, dtype=torch.int32, device=dev())
    torch.cuda.synchronize()
    plan = s.plan(x, [LS.SamplingParams.greedy(temperature=1.0, top_k=3, top_p=1.0, seed=1)], [0], out, dbg_ids=ids)
    plan.run(0)
    s.synchronize()
    assert ids[0, :3].tolist() == best and out.item() in best
    plan.close()
    s.close()
    del x
    torch.cuda.empty_cache()


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("raising", [False, True], ids=["lowering", "raising"])
def test_dense_histories_stay_a_block_at_a_time(monkeypatch, bf16, raising):
    """Rows of which a twentieth to all of the ids are listed, spread evenly or crowded into the first tenth of the
    vocabulary (where a tokenizer puts what is frequent): no slice is given up to the exhaustive select."""
    vocab = 131_099
    shares = [0.05, 0.1, 0.12, 0.13, 0.16, 0.2, 0.24, 0.25, 0.3, 0.4, 0.6, 1.0]
    crowded = [0.3, 0.6, 0.9, 1.0]   # of the first tenth
    rows = len(shares) + len(crowded)
    rng = np.random.default_rng(8)
    x = rng.normal(0, 2, (rows, vocab)).astype(np.float32)
    x = W.to_bf16_bits(x) if bf16 else x
    counts = np.zeros((rows, vocab), dtype=np.uint32)
    for i, share in enumerate(shares + crowded):
        n = vocab if i < len(shares) else vocab // 10
        counts[i, rng.choice(n, int(share * n), replace=False)] = 1
        counts[i, rng.integers(0, n, 200)] += 1
    s = _sampler(monkeypatch, "blocks", 5)
    scratch = []
    for i in range(rows):
        t = LS.SamplerScratch(s, vocab)
        t.add_history(torch.from_numpy(np.repeat(np.arange(vocab, dtype=np.int32), counts[i])).to(dev()))
        scratch.append(t)
    stats = torch.zeros(4, dtype=torch.int32, device=dev())
    pen = (dict(repetition_penalty=0.95, presence_penalty=-0.1, frequency_penalty=0.0625) if raising else
           dict(repetition_penalty=1.05, presence_penalty=0.25, frequency_penalty=0.125))
    for k in (20, 64):
        for lp in (True, False):
            kw = [dict(temperature=0.8, top_k=k, top_p=0.95, seed=7 + i, **pen) for i in range(rows)]
            stats.zero_()
            torch.cuda.synchronize()
            s.set_path_stats(stats)
            r = run_rows(s, x, kw, [3] * rows, scratch=scratch, logprobs=lp, use_plan=True)
            s.set_path_stats(None)
            _check(r, x, kw, 3, lp, counts)
            assert stats.cpu().tolist()[:3] == [5 * rows, 0, 0], (k, lp)
            for i in range(rows):   # (the oracle counted its draw)
                assert np.array_equal(scratch[i].read_counts().numpy(), counts[i]), i
    for t in scratch:
        t.close()
    s.close()


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("rows,vocab", [(3, 4099), (3, 8205), (20, 9001), (70, 20_000), (100, 32_003), (299, 9001), (301, 9001)])
def test_masked_rows_in_more_slices(monkeypatch, bf16, rows, vocab):
    """Masks over rows a little longer than a block, in as many slices as are asked for of such rows, as the launch has room
    for, and in two; the first of the masks admits nothing, the next ones one id, all ids, the last eight; one row draws a forced id."""
    rng = np.random.default_rng(rows + vocab)
    x = rng.normal(0, 3, (rows, vocab)).astype(np.float32)
    x[1] = 1.5
    allow = np.stack([W.allow_mask(rng, vocab, frac=0.02) for _ in range(rows)])
    allow[0] = 0
    allow[1] = 0
    allow[1, vocab // 64] = 1
    allow[2] = 0xffffffff
    if vocab % 32:
        allow[2, -1] = (1 << vocab % 32) - 1
    if rows > 3:
        allow[3] = 0
        for i in range(vocab - 8, vocab):
            allow[3, i >> 5] |= np.uint32(1 << (i & 31))
    xs = W.to_bf16_bits(x) if bf16 else x
    kw = [dict(temperature=0.8, top_k=(50, 64, 3, 20)[i % 4], top_p=0.95, seed=40 + i) for i in range(rows)]
    forced = [i if i == rows // 2 and i > 3 else None for i in range(rows)]
    s = _sampler(monkeypatch, "1")
    for lp in (False, True):
        r = run_rows(s, xs, kw, [2] * rows, allow=allow, forced=forced, logprobs=lp)
        some = sorted({*range(min(6, rows)), rows // 2, rows - 1})
        for i in some:
            if forced[i] is not None:
                assert r.ids[i] == forced[i]
                continue
            d = O.sample(xs[i], None, o_params(**kw[i]), 2, allow=allow[i], want_logprob=lp)
            check_row_against_oracle(r, i, d)
            if lp and np.isfinite(d.logprob):
                assert abs(r.logprobs[i] - d.logprob) <= 1e-5 * max(1.0, abs(d.logprob)), (i, r.logprobs[i], d.logprob)
    s.close()


CLUSTERS = ((0, 40, 9.0), (1000, 300, 9.0), (0, 1000, 30.0), (9000, 3000, 9.0), (700, 12_000, 5.0))


def _with_stats(s, fn):
    stats = torch.zeros(4, dtype=torch.int32, device=dev())
    s.set_path_stats(stats)
    try:
        out = fn()
    finally:
        s.synchronize()
        s.set_path_stats(None)
    return out, stats.cpu().numpy()


@pytest.mark.parametrize("held", ["1", "blocks"], ids=["held", "blocks"])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("pen", [False, True], ids=["plain", "penalties"])
def test_clusters_of_likely_ids(monkeypatch, held, bf16, pen):
    """Neighbouring ids that lead by far, some forty up to twelve thousand of them, at the row's start and inside: some waves
    of a slice hold nothing else, others none, and all of the cluster reaches the bound of those.  No slice is
    given up for it.  With penalties on ids of the clusters, log-probabilities and more slices than a block needs; rows that rise
    and fall all along are drawn rightly too, whichever way."""
    vocab = 50_021
    rng = np.random.default_rng(77)
    x = rng.normal(0, 2, (len(CLUSTERS) + 2, vocab)).astype(np.float32)
    for i, (at, n, lift) in enumerate(CLUSTERS):
        x[i, at:at + n] += lift
    x[-2].sort()
    x[-1] = -np.sort(-x[-1])
    xs = W.to_bf16_bits(x) if bf16 else x
    rows = len(x)
    more = dict(repetition_penalty=1.1, presence_penalty=0.2, frequency_penalty=0.1) if pen else {}
    for slices in (0, 3, 16):
        s = _sampler(monkeypatch, held, slices)
        for k, lp in ((64, True), (20, False), (50, True)):
            kw = [dict(temperature=0.9, top_k=k, top_p=0.99, seed=60 + i, **more) for i in range(rows)]
            hist = rng.integers(0, 4000, (rows, 1500)).astype(np.int32)
            for n in (rows, len(CLUSTERS)):
                sc = counts = None
                if pen:
                    sc, counts = [], [np.bincount(hist[i], minlength=vocab).astype(np.uint32) for i in range(n)]
                    for i in range(n):
                        t = LS.SamplerScratch(s, vocab)
                        t.add_history(torch.from_numpy(hist[i]).to(dev()))
                        sc.append(t)
                # (the blocks' way takes resident batches only)
                r, stats = _with_stats(s, lambda: run_rows(s, xs[:n], kw[:n], [3] * n, scratch=sc, logprobs=lp, use_plan=True))
                _check(r, xs[:n], kw[:n], 3, lp, counts)
                assert n == rows or stats[2] == 0, (slices, k, stats)
                for t in sc or []:
                    t.close()
        s.close()


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("vocab", [20_011, 50_257])
def test_masks_in_clusters(monkeypatch, bf16, vocab):
    """Masks of runs of 16 to 1 000 ids, 5 to 60 % of them admitted: waves of a slice with hundreds of values beside waves with none.
    No slice is given up for it."""
    rng = np.random.default_rng(vocab)
    rows = 12
    x = rng.normal(0, 2, (rows, vocab)).astype(np.float32)
    allow = np.zeros((rows, (vocab + 31) // 32), dtype=np.uint32)
    for i in range(rows):
        run, frac = (16, 64, 250, 1000)[i % 4], (0.05, 0.2, 0.6)[i % 3]
        on = np.repeat(rng.random(vocab // run + 1) < frac, run)[:vocab]
        ids = np.nonzero(on)[0]
        np.bitwise_or.at(allow[i], ids >> 5, (1 << (ids & 31)).astype(np.uint32))
    xs = W.to_bf16_bits(x) if bf16 else x
    for slices in (0, 13):
        s = _sampler(monkeypatch, "1", slices)
        for k in (20, 50, 64):
            kw = [dict(temperature=0.8, top_k=k, top_p=0.95, seed=80 + i) for i in range(rows)]
            r, stats = _with_stats(s, lambda: run_rows(s, xs, kw, [5] * rows, allow=allow, logprobs=True))
            _check(r, xs, kw, 5, True, allow=allow)
            assert stats[2] == 0, (slices, k, stats)
        s.close()


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("share", [1.0, 0.06, -0.3], ids=["open", "one by one", "in runs"])
def test_masked_sums_of_small_terms(monkeypatch, bf16, share):
    """One id carries the row, the others add a 50th in terms of 2^-24 to 2^-22 of it, near half a step of its sum in f32: as a sum of f32
    values in order the log-probability is off by 1e-5; every term's own error is below 2^-21 of it, so that 1e-7 holds
    with the result's own rounding (of the rest's 0.02 and of the result, below 2e-8 each)."""
    vocab = 248_320
    rng = np.random.default_rng(11)
    x = rng.normal(0, 0.01, (4, vocab)).astype(np.float32)
    lead = 1234
    x[:, lead] = 15.5, 16.0, 16.5, 17.0
    on = rng.random(vocab) < share if share > 0 else np.repeat(rng.random(vocab // 64) < -share, 64)
    on[lead] = True
    x[:, lead] += np.float32(np.log(on.sum() / vocab))
    ids = np.nonzero(on)[0]
    allow = np.zeros((4, (vocab + 31) // 32), dtype=np.uint32)
    np.bitwise_or.at(allow, (slice(None), ids >> 5), (1 << (ids & 31)).astype(np.uint32))
    xs = W.to_bf16_bits(x) if bf16 else x
    kw = [dict(temperature=1.0, top_k=0, top_p=0.5, seed=i) for i in range(4)]
    s = _sampler(monkeypatch, "1")
    r = run_rows(s, xs, kw, [0] * 4, allow=allow, logprobs=True)
    for i in range(4):
        d = O.sample(xs[i], None, o_params(**kw[i]), 0, allow=allow[i], want_logprob=True)
        check_row_against_oracle(r, i, d)
        assert d.chosen == lead and abs(r.logprobs[i] - d.logprob) <= 1e-7, (i, r.logprobs[i], d.logprob)
    s.close()
