"""The work that a program has this library do, as cases that can be timed and compared.

Two halves of one decode step: the draws from logits that are there already (one row up to a
batch of 1 024, f32 and bf16, plain, under penalties, under masks and bias lists, and the
speculative step), and the language-model head in front of them with the draws from its
summaries (a few rows over bf16 weights or affine codes, a ragged batch, a batch of 1 024).
Sizes are those of the benchmark and the tests, and of the reference's vocabulary (248 320).

A case is a dict of plain values; `kind` says which call it is:
  greedy     lily_sample_f32 of one greedy row (the exact argmax)
  single     lily_sample_f32 of one sampled row
  rows       a resident plan of a batch, run once a step
  spec       one speculative step: the draft draws, the verify pass, the acceptance
  head       lily_lm_head_sample_rows: logits, summaries and draws in one call
`penalties`: 0 none; 1 those of the decode configuration over a history as text has it (a few ids
make up most of it); 2 those of the throughput configuration over ids spread evenly.
"""
import math
import os
import sys

import torch

# The library is looked for where the program runs, as an import of an installed package would be.
sys.path.insert(0, os.path.join(os.getcwd(), "lily-qwen3.8-flash-next_amd", "python"))

import lily_sampler as LS  # noqa: E402

DEVICE = "cuda"
VOCAB = 151_936
VOCAB_LARGE = 248_320
# As in the benchmark, the steps take this many resident sets of logits (or of hidden states) in
# turn: a decode step never reads the logits of the step before it.
SETS = 8
# A request under penalties writes this many tokens; then its slot takes the next request, whose
# counts start from its own prompt again.
REQUEST_TOKENS = 4096


def listed():
    return [
        # A request with temperature 0 decoded alone: the shortest call there is.
        dict(name="greedy_b1", kind="greedy", vocab=VOCAB),
        # One chat request decoded alone with the usual settings.
        dict(name="sample_b1", kind="single", vocab=VOCAB, top_k=20, penalties=0, history=0),
        # The default batch of a local server: four conversations under penalties.
        dict(name="decode_b4", kind="rows", rows=4, vocab=VOCAB, dtype="f32", shape="normal3", top_k=20, penalties=1,
             history=8192, mask=0, logprob=0),
        # The same for requests that name no top_k (1 024 candidates a row) and want log-probabilities.
        dict(name="decode_b4_no_top_k", kind="rows", rows=4, vocab=VOCAB, dtype="f32", shape="normal3", top_k=0,
             penalties=0, history=0, mask=0, logprob=1),
        # Speculative decoding of one request: two drafts proposed, three rows verified.
        dict(name="spec_m3", kind="spec", rows=3, vocab=VOCAB, top_k=20, penalties=0, history=0),
        # A server's busy batch, ragged, at the reference's vocabulary, under penalties over running text.
        dict(name="rows_b200_large_vocab", kind="rows", rows=200, vocab=VOCAB_LARGE, dtype="bf16", shape="normal2",
             top_k=50, penalties=1, history=3000, mask=0, logprob=1),
        # Constrained decoding (tool calls, a grammar): masks, bias lists, forced tokens, no top_k.
        dict(name="constrained_b64", kind="rows", rows=64, vocab=VOCAB, dtype="bf16", shape="normal2", top_k=0,
             penalties=0, history=0, mask=1, logprob=1),
        # Throughput serving: the headline batch, its history spread evenly over the vocabulary.
        dict(name="throughput_b1024", kind="rows", rows=1024, vocab=VOCAB, dtype="bf16", shape="mixture", top_k=64,
             penalties=2, history=2048, mask=0, logprob=1),
        # The head and the draws of the default batch over the reference's 4-bit head, f32 logits.
        dict(name="head_q4_b4", kind="head", rows=4, vocab=VOCAB, d=4096, weights="q4", logits="f32", top_k=20,
             penalties=1, history=2048, logprob=1),
        # The same over bf16 weights.
        dict(name="head_bf16_b4", kind="head", rows=4, vocab=VOCAB, d=4096, weights="bf16", logits="bf16", top_k=64,
             penalties=0, history=0, logprob=0),
        # A ragged middle batch over the 8-bit head at a smaller width: between a decode step and a batch.
        dict(name="head_q8_b50", kind="head", rows=50, vocab=VOCAB, d=2560, weights="q8", logits="f32", top_k=50,
             penalties=0, history=0, logprob=1),
        # Throughput serving with the head in the call.
        dict(name="head_bf16_b1024", kind="head", rows=1024, vocab=VOCAB, d=4096, weights="bf16", logits="bf16",
             top_k=64, penalties=0, history=0, logprob=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _any_vocab(rng):
    """The two vocabularies of real use, or any size from 32 000 on, odd ones among them."""
    return rng.choice([VOCAB, VOCAB_LARGE, _log_int(rng, 32_000, VOCAB_LARGE), _log_int(rng, 32_000, VOCAB_LARGE)])


def draw(rng):
    kind = rng.choice(["greedy", "single", "spec", "rows", "rows", "rows", "rows", "head", "head", "head"])
    if kind == "greedy":
        return dict(kind="greedy", vocab=_any_vocab(rng) - rng.randrange(5))
    if kind == "single":
        penalties = rng.choice([0, 1])
        return dict(kind="single", vocab=_any_vocab(rng) - rng.randrange(5),
                    top_k=rng.choice([0, _log_int(rng, 2, 64), 20, 50]), penalties=penalties,
                    history=_log_int(rng, 64, 16_384) if penalties else 0)
    if kind == "spec":
        return dict(kind="spec", rows=rng.randint(2, 6), vocab=_any_vocab(rng),
                    top_k=rng.choice([20, _log_int(rng, 2, 64)]), penalties=rng.randrange(2), history=2048)
    vocab = _any_vocab(rng)
    if kind == "rows":
        rows = _log_int(rng, 1, 1024)
        mask = 1 if rng.random() < 0.25 else 0
        penalties = 0 if mask else rng.choice([0, 1, 2])
        # No top_k asks for 1 024 candidates of each row, masks for a pass of their own: batches of
        # such requests stay within what the largest listed case costs.
        top_k = rng.choice([0, _log_int(rng, 2, 64), 20, 50, 64])
        if mask or top_k == 0:
            rows = max(1, rows // 8)
        rows = min(rows, 1024 * VOCAB // vocab)
        logprob = rng.randrange(2)
        shape = rng.choice(["normal3", "normal2", "mixture"])
        if logprob and rows < 16:
            shape = "normal2"  # (a few dominated rows would give log-probabilities of 0 and nothing to compare)
        return dict(kind="rows", rows=rows, vocab=vocab, dtype=rng.choice(["f32", "bf16"]) if rows <= 256 else "bf16",
                    shape=shape, top_k=top_k, penalties=penalties,
                    history=_log_int(rng, 64, 8192) if penalties else 0, mask=mask, logprob=logprob)
    weights = rng.choice(["bf16", "q4", "q8"])
    d = 256 * rng.randint(4, 20)
    rows = _log_int(rng, 1, 512)
    # no more than the largest listed head: 1 024 rows x 4 096 x 151 936
    rows = max(1, min(rows, int(1024 * 4096 * VOCAB * 0.6 / (d * vocab))))
    vocab -= vocab % 8  # rows of logits at multiples of 16 bytes
    penalties = rng.choice([0, 1, 2])
    return dict(kind="head", rows=rows, vocab=vocab, d=d, weights=weights,
                logits="f32" if weights != "bf16" else rng.choice(["bf16", "f32"]), top_k=rng.choice([20, 50, 64]),
                penalties=penalties, history=_log_int(rng, 64, 4096) if penalties else 0,
                logprob=rng.randrange(2) if weights != "bf16" and rows >= 4 else 0)


# ---- inputs ---------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _logits(g, rows, vocab, shape, dtype):
    """N(0, 3^2) with a few leading ids a row, N(0, 2^2), or 90 % N(0, 2^2) and 10 % Student-t(3) x 4."""
    out = torch.empty(rows, vocab, dtype=torch.float32 if dtype == "f32" else torch.bfloat16, device=DEVICE)
    for r in range(0, rows, 64):
        n = min(64, rows - r)
        x = torch.randn(n, vocab, generator=g, device=DEVICE)
        if shape == "mixture":
            chi = sum(torch.randn(n, vocab, generator=g, device=DEVICE).square() for _ in range(3)) / 3
            heavy = torch.rand(n, vocab, generator=g, device=DEVICE) < 0.1
            x = torch.where(heavy, 4.0 * x / chi.sqrt(), 2.0 * x)
        elif shape == "normal3":
            x *= 3.0
            at = torch.randint(0, vocab, (n, 8), generator=g, device=DEVICE)
            x.scatter_(1, at, x.gather(1, at) + 9.0)
        else:
            x *= 2.0
        out[r:r + n] = x
    return out


def _history(g, rows, n, vocab, evenly):
    """Ids spread evenly, or with P(rank) ~ rank^-1.1 and the ranks spread over the vocabulary."""
    if evenly:
        return torch.randint(0, vocab, (rows, n), generator=g, device=DEVICE).to(torch.int32)
    rank = torch.arange(1, vocab + 1, dtype=torch.float64, device=DEVICE)
    cdf = rank.pow(-1.1).cumsum(0)
    u = torch.rand(rows, n, generator=g, device=DEVICE, dtype=torch.float64) * cdf[-1]
    ids = torch.searchsorted(cdf, u).clamp_(max=vocab - 1)
    step = 100_003  # a prime, so no vocabulary here divides it
    start = torch.randint(0, vocab, (rows, 1), generator=g, device=DEVICE)
    return ((ids * step + start) % vocab).to(torch.int32)


def _turned(x):
    """The sets: rows handed to other requests and turned along the vocabulary."""
    rows, vocab = x.shape
    return [x] + [torch.roll(x, shifts=(131 * j % rows, vocab // 5 * j + 7 * j), dims=(0, 1)).contiguous()
                  for j in range(1, SETS)]


def _scratches(sampler, history, vocab):
    out = []
    for row in history:
        sc = LS.SamplerScratch(sampler, vocab)
        sc.add_history(row)
        out.append(sc)
    return out


def _next_request(state):
    for sc, row in zip(state["scratches"], state["history"]):
        sc.reset_counts()
        sc.add_history(row)


def _allow_masks(g, rows, vocab):
    """About 2 % of the ids allowed, in runs of up to 64; packed 32 ids a word."""
    runs = max(1, vocab * 2 // 100 // 32)
    words = (vocab + 31) // 32
    at = torch.randint(0, vocab, (rows, runs), generator=g, device=DEVICE)
    length = torch.randint(1, 65, (rows, runs), generator=g, device=DEVICE)
    edge = torch.zeros(rows, words * 32 + 1, dtype=torch.int32, device=DEVICE)
    one = torch.ones_like(at, dtype=torch.int32)
    edge.scatter_add_(1, at, one)
    edge.scatter_add_(1, (at + length).clamp_(max=vocab), -one)
    bits = (edge.cumsum(1)[:, :-1] > 0)
    bits[:, vocab:] = False
    weight = (1 << torch.arange(32, device=DEVICE, dtype=torch.int64))
    packed = (bits.view(rows, words, 32).to(torch.int64) * weight).sum(2)
    return torch.where(packed >= 2 ** 31, packed - 2 ** 32, packed).to(torch.int32).contiguous()


def _params(case, row, seed):
    kw = dict(temperature=0.8, top_k=case["top_k"], top_p=0.95, seed=1000 * seed + row)
    if case.get("mask"):
        kw.update(temperature=1.0, top_p=0.9)
    if case["penalties"] == 1:
        kw.update(temperature=0.6, min_p=0.05, repetition_penalty=1.05, presence_penalty=0.3, frequency_penalty=0.2)
    if case["penalties"] == 2:
        kw.update(top_p=0.9, repetition_penalty=1.1, presence_penalty=0.2, frequency_penalty=0.1)
    return LS.SamplingParams.greedy(**kw)


def _quantise(w, bits, group):
    """Affine codes of bf16 weights, in groups of a row: q * scale + bias."""
    vocab, d = w.shape
    per = 32 // bits
    codes = torch.empty(vocab, d // per, dtype=torch.int32, device=DEVICE)
    scales = torch.empty(vocab, d // group, dtype=torch.bfloat16, device=DEVICE)
    biases = torch.empty_like(scales)
    shift = (bits * torch.arange(per, device=DEVICE, dtype=torch.int32))
    for v in range(0, vocab, 16_384):
        part = w[v:v + 16_384].float().view(-1, d // group, group)
        low, high = part.amin(2), part.amax(2)
        scale = ((high - low) / ((1 << bits) - 1)).clamp_min(1e-8).to(torch.bfloat16)
        bias = low.to(torch.bfloat16)
        q = ((part - bias.float()[..., None]) / scale.float()[..., None]).round_().clamp_(0, (1 << bits) - 1)
        q = q.to(torch.int32).view(-1, d // per, per)
        codes[v:v + 16_384] = (q << shift).sum(2, dtype=torch.int32)  # wraps into the sign bit as the packing wants
        scales[v:v + 16_384], biases[v:v + 16_384] = scale, bias
    return LS.QuantWeights(codes, scales, biases, group, bits)


def _head_weights(g, hidden, vocab):
    """Logits of a real head's shape: a bulk N(0, 2^2), a heavy-tailed tenth of the ids, and a
    handful of ids for every hidden state whose weights point along it."""
    n_hidden, d = hidden.shape
    w = torch.empty(vocab, d, dtype=torch.bfloat16, device=DEVICE)
    for v in range(0, vocab, 16_384):
        n = min(16_384, vocab - v)
        part = torch.randn(n, d, generator=g, device=DEVICE) * (2.0 / d ** 0.5)
        chi = sum(torch.randn(n, 1, generator=g, device=DEVICE).square() for _ in range(3)) / 3
        t3 = torch.randn(n, 1, generator=g, device=DEVICE).abs() / chi.sqrt()
        heavy = torch.rand(n, 1, generator=g, device=DEVICE) < 0.1
        w[v:v + n] = part * torch.where(heavy, 0.7 * t3.clamp(max=3.0), torch.ones_like(t3))
    each = max(1, min(40, vocab // (2 * n_hidden)))
    ids = torch.randperm(vocab, generator=g, device=DEVICE)[:n_hidden * each].view(n_hidden, each)
    for r in range(0, n_hidden, 128):
        i = ids[r:r + 128]
        gain = (torch.rand(i.shape, generator=g, device=DEVICE) * 0.7 + 0.3) * (6.0 / d)
        w[i] = (w[i].float() + gain[..., None] * hidden[r:r + 128, None, :].float()).to(torch.bfloat16)
    return w


_SAMPLER = []


def _sampler():
    """A program's one sampler, on the stream its tensors live on."""
    if not _SAMPLER:
        _SAMPLER.append(LS.Sampler(0))
    return _SAMPLER[0]


def prepare(case, seed):
    s, g = _sampler(), _generator(seed)
    kind, vocab, rows = case["kind"], case["vocab"], case.get("rows", 1)
    state = dict(kind=kind, sampler=s, step=0, rows=rows, scratches=[], history=[])
    if case.get("penalties"):
        requests, evenly = 1 if kind == "spec" else rows, case["penalties"] == 2
        state["history"] = list(_history(g, requests, case["history"], vocab, evenly))
        state["scratches"] = _scratches(s, state["history"], vocab)
    if kind in ("greedy", "single"):
        state.update(x=[t[0] for t in _turned(_logits(g, 1, vocab, "normal3", "f32"))],
                     params=LS.SamplingParams.greedy() if kind == "greedy" else _params(case, 0, seed),
                     scratch=state["scratches"][0] if state["scratches"] else None,
                     out=torch.zeros(1, dtype=torch.int32, device=DEVICE))
    elif kind == "spec":
        target = _turned(_logits(g, rows, vocab, "normal3", "f32"))
        draft = [t + 0.5 * torch.randn(rows, vocab, generator=g, device=DEVICE) for t in target]
        p = _params(case, 0, seed)
        tokens = torch.randint(0, vocab, (rows,), generator=g, device=DEVICE).to(torch.int32)
        state.update(target=target, draft=draft, params=p, draft_params=LS.draft_params(p),
                     scratch=state["scratches"][0] if state["scratches"] else LS.SamplerScratch(s, vocab),
                     dists=LS.DraftDists(s, rows), tokens=tokens,
                     verified=torch.zeros(rows, dtype=torch.int32, device=DEVICE),
                     ctrl=torch.zeros(LS.ctrl_words(rows - 1), dtype=torch.int32, device=DEVICE))
    else:
        ids = torch.zeros(rows, dtype=torch.int32, device=DEVICE)
        params = [_params(case, r, seed) for r in range(rows)]
        more = {}
        if state["scratches"]:
            more["scratch"] = state["scratches"]
        if case["logprob"]:
            more["out_logprobs"] = torch.zeros(rows, dtype=torch.float32, device=DEVICE)
        out = [ids] + ([more["out_logprobs"]] if case["logprob"] else [])
        if kind == "rows":
            if case["mask"]:
                more["allow"] = _allow_masks(g, rows, vocab)
                at = torch.randint(0, vocab, (rows, 32), generator=g, device=DEVICE).tolist()
                delta = (torch.randint(0, 2, (rows, 32), generator=g, device=DEVICE) * 10.0 - 5.0).tolist()
                more["bias"] = [sorted(dict(zip(a, b)).items()) for a, b in zip(at, delta)]
                forced = torch.randint(0, 4 * vocab, (rows,), generator=g, device=DEVICE).tolist()
                more["forced"] = [f if f < vocab else None for f in forced]  # one row in four
            x = _turned(_logits(g, rows, vocab, case["shape"], case["dtype"]))
            state.update(x=x, plans=[s.plan(t, params, [0] * rows, ids, **more) for t in x], out=out)
        else:
            hidden = torch.randn(SETS, rows, case["d"], generator=g, device=DEVICE).to(torch.bfloat16)
            w = _head_weights(g, hidden.view(SETS * rows, case["d"]), vocab)
            if case["weights"] != "bf16":
                w = _quantise(w, 4 if case["weights"] == "q4" else 8, 64)
            logits = torch.zeros(rows, vocab, dtype=torch.float32 if case["logits"] == "f32" else torch.bfloat16,
                                 device=DEVICE)
            tiles = (vocab + LS.LOGIT_TILE_COLS - 1) // LS.LOGIT_TILE_COLS
            tile_max = torch.zeros(rows, tiles, dtype=torch.float32, device=DEVICE)
            tile_sum = torch.zeros(rows, tiles, dtype=torch.float32, device=DEVICE)
            state.update(hidden=list(hidden), w=w, logits=logits, tile_max=tile_max, tile_sum=tile_sum, ids=ids,
                         params=params, more=more, out=out + [logits, tile_max, tile_sum])
    return state


# ---- one pass -------------------------------------------------------------------------------

def run(state):
    s, kind, step = state["sampler"], state["kind"], state["step"]
    at = step % SETS
    state["step"] = step + 1
    if step % REQUEST_TOKENS == REQUEST_TOKENS - 1:
        _next_request(state)
    if kind in ("greedy", "single"):
        s.sample_f32(state["x"][at], state["scratch"], state["params"], step, state["out"])
        return state["out"]
    if kind == "rows":
        state["plans"][at].run(step)
        return state["out"]
    if kind == "spec":
        m, tokens, draft = state["rows"], state["tokens"], state["draft"][at]
        base = step * m
        for j in range(m - 1):
            s.sample_draft_f32(draft[j], state["scratch"], state["draft_params"], LS.draft_step(base + j),
                               tokens[j + 1:j + 2], state["dists"].slot(j))
        s.spec_verify(state["target"][at], state["scratch"], state["params"], base, state["dists"], tokens,
                      state["verified"], state["ctrl"], pos0=100, ratio=4, chain=m - 1)
        return [tokens, state["verified"], state["ctrl"]]
    s.lm_head_sample_rows(state["hidden"][at], state["w"], state["logits"], state["tile_max"], state["tile_sum"],
                          state["params"], [step] * state["rows"], state["ids"], **state["more"])
    return state["out"]


# ---- what a pass cannot do without, and how close two of them are ---------------------------

def work(case):
    kind, vocab = case["kind"], case["vocab"]
    if kind in ("greedy", "single"):
        return {"bytes": 4 * vocab + 4 * case.get("history", 0) + 4, "flops": 0}
    if kind == "spec":
        return {"bytes": (2 * case["rows"] - 1) * 4 * vocab, "flops": 0}
    rows = case["rows"]
    if kind == "rows":
        row = vocab * (4 if case["dtype"] == "f32" else 2) + 4 * case["history"] + 4 + 4 * case["logprob"]
        if case["mask"]:
            row += (vocab + 31) // 32 * 4 + 32 * 8
        return {"bytes": rows * row, "flops": 0}
    d, tiles = case["d"], (vocab + LS.LOGIT_TILE_COLS - 1) // LS.LOGIT_TILE_COLS
    bits = {"bf16": 16, "q4": 4, "q8": 8}[case["weights"]]
    weights = vocab * d * bits // 8 + (0 if bits == 16 else vocab * (d // 64) * 4)
    row = 2 * d + vocab * (4 if case["logits"] == "f32" else 2) + 8 * tiles + 4 * case["history"] + 4
    return {"bytes": weights + rows * row, "flops": 2 * rows * d * vocab}


def tolerance(case):
    if case["kind"] == "head":
        # The order of the f32 sums is free; two orders were compared (1 024 rows, d 4 096). bf16
        # logits differ by a step of bf16 in 3e-4 of the places (rel 7e-5), the summaries follow
        # them (a largest value one step off moves its tile's sum: rel 2e-4, at most 0.036), and a
        # draw that lies on such an edge may take its neighbour. f32 logits lie within rel 4e-7 and
        # at most 2.1e-5 of the product in f64, and a log-probability divides that by a temperature.
        if case["logits"] == "bf16":
            return {"rel": 8e-4, "max": 0.15, "differ": 0.01}
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    if case.get("logprob"):
        # the bar of the tests against the f64 oracle
        return {"rel": 1e-5, "max": 4e-5, "differ": 0.0}
    return "exact"
