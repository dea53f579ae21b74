"""Performance cases of the token sampler: what serving programs have it do.

A case is one call of a public entry point on logits of one shape:

* ``greedy``  -- argmax_rows: temperature 0 requests;
* ``token``   -- PreparedCall, the token alone (a decode loop's call);
* ``kept``    -- PreparedCall, the token and the kept ids (speculative and
  constrained decoding look at the kept set);
* ``scores``  -- PreparedCall with the kept probabilities and the row
  statistics (requests that ask for log-probabilities);
* ``host``    -- Sampler.sample on one row of host logits (a CPU-resident
  caller's decode step: copy in, sample, copy out).

The logits come from five families, those of the benchmark's configurations
(llz/workloads.py) drawn on the device: ``boost`` (N(0, 2) with a few strong
tokens), ``zipf`` (N(0, 2.5) with a Zipf offset: a model's usual head and
tail), ``gumbel`` (a heavy tail with 20 strong tokens), ``flat`` (N(0, 0.3):
high-entropy rows) and ``mixed`` (N(0, 2), every other row with one dominant
token).
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "llama.zig_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import llz  # noqa: E402

KEPT_CAP = 64  # kept ids / probabilities asked for per row

# the sampling chains, by name: temperature, top-k, top-p, min-p, typical-p
CHAINS = {
    "default": (0.8, 0, 0.9, 0.0, 1.0),    # SamplerConfig's defaults
    "filters": (1.0, 40, 0.95, 0.05, 1.0),  # top-k, top-p and min-p
    "topk": (0.7, 50, 0.9, 0.0, 1.0),      # top-k and top-p
    "typical": (0.7, 0, 1.0, 0.0, 0.95),   # typical-p alone
    "nucleus": (1.2, 0, 0.9, 0.0, 1.0),    # a hot nucleus: wide kept sets
    "full": (0.8, 50, 0.9, 0.02, 0.98),    # every filter
}


def _case(name, call, rows, vocab, chain="default", logits="zipf", *, pad=0, window=0, softcap=0.0, scale=1.0):
    """rows x vocab logits, rows vocab + pad apart; window: the repetition
    penalty's window (0: off) over a history of as many tokens; softcap and
    scale: the decode loop's post-processing of the final logits."""
    case = {"call": call, "rows": rows, "vocab": vocab, "chain": chain, "logits": logits, "pad": pad,
            "window": window, "softcap": softcap, "scale": scale}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # greedy requests of a small batch; an odd vocabulary, rows unaligned
        _case("greedy-32x50021", "greedy", 32, 50021),
        # one sequence decoded with the default chain: the smallest sampling call
        _case("decode-1", "token", 1, 128256, "default", "boost"),
        # the same from host logits with the default repetition penalty
        _case("decode-1-host", "host", 1, 128256, "default", "boost", window=32),
        # a few sequences of a model that soft-caps and scales its final
        # logits, with the default repetition penalty
        _case("decode-4-post", "token", 4, 128256, "default", "boost", window=32, softcap=30.0, scale=0.5),
        # a batch over a small odd vocabulary with the penalty, kept ids asked for
        _case("kept-97x32003", "kept", 97, 32003, "topk", "zipf", window=32),
        # an ordinary batch over a large vocabulary
        _case("serve-64x151936", "token", 64, 151936, "filters", "zipf"),
        # the benchmark's headline batch
        _case("serve-256", "token", 256, 128256, "filters", "zipf"),
        # the same batch with the default chain (no min-p)
        _case("default-256", "token", 256, 128256, "default", "zipf"),
        # the headline batch with kept probabilities and row statistics
        _case("scores-256", "scores", 256, 128256, "filters", "zipf"),
        # typical-p alone over a heavy tail (wide kept sets, entropy)
        _case("typical-256x151936", "token", 256, 151936, "typical", "gumbel"),
        # high-entropy rows over the largest vocabulary: nuclei of most of the row
        _case("nucleus-1024x256000", "token", 1024, 256000, "nucleus", "flat"),
        # the largest batch, every filter on
        _case("full-4096", "token", 4096, 128256, "full", "mixed"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(("greedy", "token", "token", "token", "kept", "scores", "host"))
    chain, logits = rng.choice((
        ("default", "boost"), ("default", "zipf"), ("filters", "zipf"), ("filters", "boost"), ("topk", "zipf"),
        ("topk", "mixed"), ("full", "mixed"), ("full", "zipf"), ("typical", "gumbel"), ("nucleus", "flat")))
    vocab = _log_int(rng, 16000, 262144)
    if rng.random() < 0.5:  # many models round the vocabulary up; many do not
        vocab = -(-vocab // 64) * 64
    # elements of a batch: within what the listed case of this kind has
    most = 256 * 151936 if chain == "typical" else 1024 * 256000 if chain == "nucleus" else 1 << 27
    if call == "scores":
        most = min(most, 1 << 25)
    rows = 1 if call == "host" else _log_int(rng, 1, min(4096, most // vocab))
    pad = -vocab % 64 if call != "host" and rng.random() < 0.3 else 0  # rows padded to 64 logits
    window = rng.choice((0, 0, 32, 48, 200)) if call != "greedy" else 0
    softcap, scale = rng.choice(((0.0, 1.0), (0.0, 1.0), (0.0, 0.5), (30.0, 1.0), (30.0, 0.5)))
    if call == "host" or chain in ("typical", "nucleus"):
        softcap, scale = 0.0, 1.0
    return _case(None, call, rows, vocab, chain, logits, pad=pad, window=window, softcap=softcap, scale=scale)


def _config(case):
    t, k, p, mp, ty = CHAINS[case["chain"]]
    return llz.SamplerConfig(temperature=t, top_k=k, top_p=p, min_p=mp, typical_p=ty,
                             repetition_window=case["window"], repetition_penalty=1.1 if case["window"] else 1.0)


def _post(case):
    if case["softcap"] <= 0.0 and case["scale"] == 1.0:
        return None
    return llz.LogitPost(final_logit_softcapping=case["softcap"], logit_scale=case["scale"])


def _strong(x, count, by, g):
    """Add `by` to `count` random positions of every row."""
    at = torch.randint(x.shape[1], (x.shape[0], count), generator=g, device=x.device)
    x.scatter_add_(1, at, torch.full(at.shape, by, device=x.device))


def _logits(case, seed, device):
    rows, vocab, kind = case["rows"], case["vocab"], case["logits"]
    g = torch.Generator(device=device).manual_seed(seed)
    full = torch.empty((rows, vocab + case["pad"]), dtype=torch.float32, device=device)
    x = full[:, :vocab]
    step = max(1, (1 << 25) // vocab)  # rows at a time, so that temporaries stay small
    for r in range(0, rows, step):
        y = torch.empty((min(step, rows - r), vocab), dtype=torch.float32, device=device)
        if kind == "gumbel":
            y.exponential_(generator=g).clamp_(min=1e-30).log_().mul_(-1.5)
            _strong(y, 20, 8.0, g)
        else:
            y.normal_(0.0, {"boost": 2.0, "zipf": 2.5, "flat": 0.3, "mixed": 2.0}[kind], generator=g)
            if kind == "boost":
                _strong(y, 8, 12.0, g)
            elif kind == "zipf":
                rank = torch.rand(y.shape, generator=g, device=device).argsort(1).add_(1)
                y.sub_(rank.to(torch.float32).log_(), alpha=1.1)
            elif kind == "mixed":
                _strong(y[(r + 1) % 2::2], 1, 20.0, g)
        x[r:r + step] = y
    if case["pad"]:
        full[:, vocab:] = -1e30  # the padding columns of an LM head
    u = torch.rand(rows, generator=g, device=device).clamp_(min=2.0 ** -30)
    prev = torch.randint(vocab, (rows, case["window"]), generator=g, device=device).to(torch.int32)
    return x, u, prev


def prepare(case, seed):
    if case["call"] == "host":
        x, _, prev = _logits(case, seed, torch.device("cpu"))
        return {"sampler": llz.Sampler(_config(case)), "x": np.ascontiguousarray(x[0].numpy()),
                "prev": prev[0].numpy().astype(np.uint32)}
    dev = torch.device("cuda:0")
    x, u, prev = _logits(case, seed, dev)
    if case["call"] == "greedy":
        return {"greedy": True, "x": x, "post": _post(case)}
    ids, probs = case["call"] in ("kept", "scores"), case["call"] == "scores"
    call = llz.PreparedCall(case["rows"], case["vocab"], _config(case), dev, kept_cap=KEPT_CAP if ids else 0,
                            probs=probs, stats=probs, post=_post(case), prev_tokens=prev if case["window"] else None)
    if ids:  # entries past a row's kept count are never written: defined values there
        call.result.kept_ids.fill_(-1)
    if probs:
        call.result.kept_probs.zero_()
    return {"call": call, "x": x, "u": u}


def run(state):
    if "sampler" in state:
        return state["sampler"].sample(state["x"], state["prev"])
    if "greedy" in state:
        return llz.argmax_rows(state["x"], post=state["post"])
    r = state["call"](state["x"], state["u"])
    out = {"tokens": r.tokens, "consumed": r.consumed}
    if r.kept_ids is not None:
        out.update(kept_count=r.kept_count, kept_ids=r.kept_ids)
    if r.kept_probs is not None:
        out.update(kept_probs=r.kept_probs, row_stats=r.row_stats)
    return out


def work(case):
    rows, vocab = case["rows"], case["vocab"]
    per_row = 4 * vocab + 4  # the logits in, the token out
    if case["call"] != "greedy":
        per_row += 4 + 1 + 4 * case["window"]  # the uniform and the history in, the draw flag out
    if case["call"] in ("kept", "scores"):
        per_row += 4 + 4 * KEPT_CAP
    if case["call"] == "scores":
        per_row += 4 * KEPT_CAP + 16
    # a compare for the maximum; the scale, the exponential and the sum
    return {"bytes": rows * per_row, "flops": rows * vocab * (1 if case["call"] == "greedy" else 5)}


def tolerance(case):
    # the sampler's contract: tokens, kept sets, probabilities and statistics
    # are the reference chain's sequential f32 results, bit for bit
    return "exact"


def exact(case, seed):
    """Kept probabilities and row statistics in float64.  Tokens, draw flags
    and kept sets are decisions of the f32 chain and have no such value, so a
    call that returns nothing else has none."""
    if case["call"] != "scores":
        return None
    dev = torch.device("cuda:0")
    x, _, prev = _logits(case, seed, dev)
    t, k, top_p, min_p, typical = (float(np.float32(v)) if isinstance(v, float) else v for v in CHAINS[case["chain"]])
    rows, vocab = case["rows"], case["vocab"]
    probs = torch.zeros((rows, KEPT_CAP), dtype=torch.float64, device=dev)
    stats = torch.zeros((rows, 4), dtype=torch.float64, device=dev)
    step = max(1, (1 << 23) // vocab)
    for r in range(0, rows, step):
        v = x[r:r + step].double()
        if case["softcap"] > 0.0:
            v = torch.tanh(v / case["softcap"]) * case["softcap"]
        if case["scale"] != 1.0:
            v = v / case["scale"]
        if case["window"]:
            at = prev[r:r + step].long()
            w = v.gather(1, at)
            rp = float(np.float32(1.1))
            v.scatter_(1, at, torch.where(w > 0.0, w / rp, w * rp))
        m = v.amax(1, keepdim=True)
        e = torch.exp((v - m) / t)
        total = e.sum(1, keepdim=True)
        p, order = torch.sort(e / total, dim=1, descending=True, stable=True)
        kept = torch.ones_like(p, dtype=torch.bool)
        if 0 < k < vocab:
            kept[:, k:] = False
        if 0.0 < top_p < 1.0:
            kept &= (p * kept).cumsum(1) <= top_p
        if min_p > 0.0:
            kept &= p >= p[:, :1] * min_p
        if 0.0 < typical < 1.0:
            surprise = -torch.log(p.clamp(min=1e-300))
            h = (p * surprise).sum(1, keepdim=True)
            away = torch.argsort((surprise - h).abs(), dim=1, stable=True)
            cum = (p * kept).gather(1, away).cumsum(1)
            kept &= torch.zeros_like(kept).scatter_(1, away, cum <= typical)
            # the sampler reports the entropy only where the kept set depends on it
            stats[r:r + step, 2:3] = h
        n = min(KEPT_CAP, vocab)
        first = torch.argsort((~kept).to(torch.int8), dim=1, stable=True)[:, :n]
        probs[r:r + step, :n] = p.gather(1, first) * kept.gather(1, first)
        stats[r:r + step, 0:1] = m
        stats[r:r + step, 1:2] = total
        stats[r:r + step, 3:4] = (p * kept).sum(1, keepdim=True)
    return {"tokens": None, "consumed": None, "kept_count": None, "kept_ids": None, "kept_probs": probs,
            "row_stats": stats}
