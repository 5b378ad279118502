"""Rows cut into slices: the one-wave merge and draw of rows of few candidates (k <= 64), on both
sides of the limits at which it lists the slices' candidates, merges them list by list or leaves
them (more than 2 048 places) to the whole workgroup; and launches of greedy rows.  Bit-exact against the oracle."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import lily_sampler as LS
import lily_workloads as W
import oracle as O
from gpu_util import check_row_against_oracle, dev, ls_params, o_params, run_rows, upload_logits


def _sampler(slices):
    old = os.environ.get("LILY_SAMPLER_SLICES")
    os.environ["LILY_SAMPLER_SLICES"] = str(slices)
    try:
        return LS.Sampler(0)
    finally:
        if old is None:
            os.environ.pop("LILY_SAMPLER_SLICES", None)
        else:
            os.environ["LILY_SAMPLER_SLICES"] = old


def _rows(rng, rows, vocab, bf16):
    x = rng.normal(0, 3, (rows, vocab)).astype(np.float32)
    x[1] = np.round(x[1])                                 # ties by the hundred at every value
    x[2, rng.random(vocab) < 0.9995] = -np.inf            # fewer finite values than k, slices without one
    x[3, :] = -np.inf
    x[4, vocab // 2:vocab // 2 + 300] = np.linspace(20, 21, 300, dtype=np.float32)   # one slice holds them all
    return W.to_bf16_bits(x) if bf16 else x


@pytest.mark.parametrize("slices", [2, 3, 4, 8, 9, 32, 33, 64])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_rows_of_few_candidates_over_slices(slices, bf16):
    s = _sampler(slices)
    rng = np.random.default_rng(slices + 100 * bf16)
    vocab = 131_075
    x = _rows(rng, 5, vocab, bf16)
    for trial, k in enumerate((2, 16, 20, 33, 63, 64)):
        kw = [dict(temperature=0.7, top_k=k, top_p=0.97, seed=60 + r) for r in range(5)]
        for lp in (False, True):
            r = run_rows(s, x, kw, [trial] * 5, logprobs=lp)
            for i in range(5):
                d = O.sample(x[i], None, o_params(**kw[i]), trial, want_logprob=lp)
                check_row_against_oracle(r, i, d)
                if lp and np.isfinite(d.logprob):
                    assert abs(r.logprobs[i] - d.logprob) <= 1e-5 * max(1.0, abs(d.logprob)), (k, i)
    s.close()


@pytest.mark.parametrize("slices", [3, 4, 31, 64])
@pytest.mark.parametrize("ks", [(64, 2, 33, 20, 7), (63, 61, 5, 48, 32), (31, 3, 30, 2, 17)])
def test_rows_of_different_k_over_slices(slices, ks):
    """A slice's list has as many places as the launch's largest k asks for, and is turned within
    them: rows whose lists fill a few of them only."""
    s = _sampler(slices)
    rng = np.random.default_rng(slices)
    x = _rows(rng, 5, 131_075, False)
    kw = [dict(temperature=0.7, top_k=k, top_p=0.97, seed=90 + r) for r, k in enumerate(ks)]
    r = run_rows(s, x, kw, [3] * 5)
    for i in range(5):
        check_row_against_oracle(r, i, O.sample(x[i], None, o_params(**kw[i]), 3))
    s.close()


@pytest.mark.parametrize("rows", [1, 8, 9, 600])
@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_launches_of_greedy_rows(rows, bf16):
    """Inline and from a table, in slices and whole; the first of equal maxima, rows of -inf and of
    NaN, rows that start inside a 16-byte piece."""
    s = LS.Sampler(0)
    rng = np.random.default_rng(rows)
    vocab = 20_011
    x = np.round(rng.normal(0, 2, (rows, vocab))).astype(np.float32)
    x[0, ::3] = np.nan
    if rows > 3:
        x[1, :] = -np.inf
        x[2, :] = np.nan
        x[3, :vocab - 1] = -np.inf
    if bf16:
        x = W.to_bf16_bits(x)
    logits = upload_logits(x)
    out = torch.full((rows,), -1, dtype=torch.int32, device=dev())
    p = [ls_params()] * rows
    torch.cuda.synchronize()
    plan = s.plan(logits, p, [0] * rows, out)
    got = []
    for _ in range(2):
        plan.run(0)
        s.synchronize()
        got.append(out.cpu().numpy().copy())
        out.fill_(-1)
        torch.cuda.synchronize()
    keep = s.sample_rows(logits, p, [0] * rows, out)
    s.synchronize()
    got.append(out.cpu().numpy())
    del keep
    f = W.bf16_bits_to_f32(x) if bf16 else x
    f = np.where(np.isnan(f), -np.inf, f)
    want = np.array([np.argmax(f[r]) for r in range(rows)])
    for ids in got:
        for r in range(rows):
            if not np.isfinite(f[r]).any():
                # (nothing to choose: the first id that is no NaN, or id 0)
                assert ids[r] == 0, (r, ids[r])
            else:
                assert ids[r] == want[r], (r, ids[r], want[r])
    plan.close()
    s.close()
