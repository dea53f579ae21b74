"""Rows at the ends of the f32 range, against the oracle: masks of very large
negative and of the type's lowest values, beside -inf masks and alone, maxima
near the largest float, and an infinite temperature.  A maximum times
log2(e) / T that overflows must not turn the estimates of -inf logits, or of
positions past the row's end, into NaN."""
import dataclasses

import numpy as np
import pytest

import llz
import oracle_lib as O
from llz.workloads import Params

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LOW = np.finfo(np.float32).min
FILTERS = Params(1.0, 40, 0.95, 0.05, 1.0, 0, 1.0)
DEFAULT = Params(0.8, 0, 0.9, 0.0, 1.0, 0, 1.0)


def _same(a, b):
    """Bit for bit, any NaN like any other."""
    a, b = np.atleast_1d(np.asarray(a, np.float32)), np.atleast_1d(np.asarray(b, np.float32))
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


def _check(x, params, *, post=None, offset=0, exact=False):
    rows, n = x.shape
    u = llz.rng_uniforms(11, rows)
    flat = torch.zeros(rows * n + offset, dtype=torch.float32, device="cuda")
    xd = flat[offset:].view(rows, n)
    xd.copy_(torch.from_numpy(x))
    r = llz.sample_rows(xd, llz.SamplerConfig.of(params), torch.from_numpy(u).cuda(), post=post, kept_cap=64,
                        probs=exact, stats=exact, path=True)
    torch.cuda.synchronize()
    tok, con = r.tokens.cpu().numpy().view(np.uint32), r.consumed.cpu().numpy()
    kc, ids = r.kept_count.cpu().numpy().view(np.uint32), r.kept_ids.cpu().numpy().view(np.uint32)
    xs = x if post is None else O.logit_post(x, post.final_logit_softcapping, post.logit_scale)
    for i in range(rows):
        o = O.sample_row(xs[i], params, u[i])
        ctx = (i, hex(int(r.row_path[i].item()) & 0xFFFFFFFF))
        assert (tok[i], con[i], kc[i]) == (o.token, o.consumed, o.kept_count), ctx
        k = min(o.kept_count, 64)
        assert np.array_equal(ids[i, :k], o.kept_ids()[:k]), ctx
        if exact:
            st = r.row_stats[i].cpu().numpy()
            assert _same(st[[0, 1, 3]], [o.max_logit, o.sum, o.total]), ctx
            assert st[2] == 0.0 or _same(st[2], o.entropy), ctx
            assert _same(r.kept_probs[i, :k].cpu().numpy(), o.probs[ids[i, :k]]), ctx


def _masked(n, low, seed=0):
    """Rows whose waves first meet nothing but the mask `low`."""
    g = np.random.default_rng([n, seed])
    x = g.normal(0.0, 2.0, size=(6, n)).astype(np.float32)
    head = min(n // 2, 16384)
    x[0, :head] = low                      # every wave's first segments
    x[1, :n - 300] = low
    x[2, :] = low                          # nothing left but the mask
    x[3, :head] = low
    x[3, head::2] = -np.inf                # both masks in a row
    x[4, ::2] = low
    x[4, 1::2] = -np.inf
    x[4, n // 3] = np.float32(3.0)
    x[5, :head:2] = -np.inf
    x[5, 1:head:2] = low
    return x


@pytest.mark.parametrize("exact", [False, True], ids=["token", "exact"])
@pytest.mark.parametrize("n,offset", [(129028, 0), (151936, 0), (200003, 1)])
@pytest.mark.parametrize("low,t,scale", [(-1e38, 0.25, 1.0), (-3e38, 1.0, 1.0), (LOW, 0.7, 2.0), (LOW, 1.0, 1.0),
                                         (LOW, 40.0, 1.0)])
def test_long_rows_low_masks(n, offset, low, t, scale, exact):
    _check(_masked(n, np.float32(low)), dataclasses.replace(FILTERS, temperature=t),
           post=llz.LogitPost(0.0, scale) if scale != 1.0 else None, offset=offset, exact=exact)


@pytest.mark.parametrize("n", [129028, 151937])
def test_long_rows_infinite_temperature(n):
    x = np.random.default_rng(n).normal(0.0, 2.0, size=(3, n)).astype(np.float32)
    x[1, n // 2] = -np.inf  # (-inf - max) / inf: NaN, in the reference too
    x[2, 3] = -np.inf
    for p in (FILTERS, DEFAULT):
        for exact in (False, True):
            _check(x, dataclasses.replace(p, temperature=float("inf")), exact=exact)


@pytest.mark.parametrize("exact", [False, True], ids=["token", "exact"])
@pytest.mark.parametrize("n", [3, 2000, 4099, 50000, 129024, 129028])
def test_largest_finite_maxima(n, exact):
    """A maximum beyond 3e38 is a number, not an infinity."""
    x = np.full((3, n), LOW, np.float32)
    x[1] = np.random.default_rng(n).normal(0.0, 2.0, n)
    x[1, n // 2] = -LOW
    x[2] = np.float32(3.2e38)
    for p in (FILTERS, DEFAULT, dataclasses.replace(FILTERS, temperature=60.0)):
        _check(x, p, exact=exact)


@pytest.mark.parametrize("exact", [False, True], ids=["token", "exact"])
@pytest.mark.parametrize("n,offset", [(2049, 0), (4100, 0), (4099, 1), (32003, 0), (128256, 0), (129021, 1)])
@pytest.mark.parametrize("low,t,scale", [(-1e38, 0.25, 1.0), (-3e38, 1.0, 1.0), (LOW, 0.7, 2.0), (LOW, 40.0, 1.0)])
def test_resident_rows_low_masks(n, offset, low, t, scale, exact):
    _check(_masked(n, np.float32(low)), dataclasses.replace(FILTERS, temperature=t),
           post=llz.LogitPost(0.0, scale) if scale != 1.0 else None, offset=offset, exact=exact)


@pytest.mark.parametrize("n", [5, 1000, 2048, 2049, 4100, 129021, 129024])
def test_resident_rows_infinite_temperature(n):
    x = np.random.default_rng(n).normal(0.0, 2.0, size=(3, n)).astype(np.float32)
    x[2, n // 2] = -np.inf  # (-inf - max) / inf: NaN, in the reference too
    for p in (FILTERS, DEFAULT):
        _check(x, dataclasses.replace(p, temperature=float("inf")))
