"""Rows beyond the single pass's residency (129024 logits) on k_long, against
the oracle: the shortest and longest such rows, remainders and unaligned rows,
token-only and exact calls, every transform, penalised positions past segment
512, special values, candidate buffers that fill and overflow; and typical-p
decided from the candidate list, inside it and past it."""
import dataclasses

import numpy as np
import pytest

import llz
import oracle_lib as O
from llz.workloads import Params

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FILTERS = Params(1.0, 40, 0.95, 0.05, 1.0, 0, 1.0)
DEFAULT = Params(0.8, 0, 0.9, 0.0, 1.0, 0, 1.0)
FULL = Params(0.8, 50, 0.9, 0.02, 0.98, 0, 1.0)
TYPICAL = Params(0.7, 0, 1.0, 0.0, 0.95, 0, 1.0)


def _rows(n, seed):
    g = np.random.default_rng([n, seed])
    x = g.normal(0.0, 2.5, size=(8, n)).astype(np.float32)
    x -= (1.1 * np.log(g.permuted(np.tile(np.arange(1, n + 1), (8, 1)), axis=1))).astype(np.float32)
    x[1, -1] = 30.0                              # the maximum is the row's last logit
    x[2] = np.sort(x[2])                         # the running maximum rises to the end: buffers refiltered
    x[3] = np.float32(0.5)                       # all equal: buffers overflow
    x[4, :n // 2] = -np.inf
    x[5, g.integers(0, n, 3)] = np.nan
    x[6, 7] = np.inf
    x[7] = g.normal(0.0, 2.0, n).astype(np.float32)
    x[7, ::9973] += 14.0
    return x


def _same(a, b):
    """Bit for bit, any NaN like any other."""
    a, b = np.atleast_1d(np.asarray(a, np.float32)), np.atleast_1d(np.asarray(b, np.float32))
    nan = np.isnan(a)
    return np.array_equal(nan, np.isnan(b)) and np.array_equal(a[~nan].view(np.uint32), b[~nan].view(np.uint32))


def _check(x, params, *, post=None, prev=None, offset=0, pad=0, exact=False):
    rows, n = x.shape
    u = llz.rng_uniforms(5, rows)
    flat = torch.zeros(rows * (n + pad) + offset, dtype=torch.float32, device="cuda")
    xd = flat[offset:].view(rows, n + pad)[:, :n]
    xd.copy_(torch.from_numpy(x))
    pv = None if prev is None else torch.from_numpy(prev.astype(np.int32)).cuda()
    llz.debug_set_split(1)
    try:
        r = llz.sample_rows(xd, llz.SamplerConfig.of(params), torch.from_numpy(u).cuda(), pv, post=post, kept_cap=64,
                            probs=exact, stats=exact, path=True)
        torch.cuda.synchronize()
    finally:
        llz.debug_set_split(0)
    tok, con = r.tokens.cpu().numpy().view(np.uint32), r.consumed.cpu().numpy()
    kc, ids = r.kept_count.cpu().numpy().view(np.uint32), r.kept_ids.cpu().numpy().view(np.uint32)
    xs = x if post is None else O.logit_post(x, post.final_logit_softcapping, post.logit_scale)
    for i in range(rows):
        o = O.sample_row(xs[i], params, u[i], prev_tokens=None if prev is None else prev[i])
        ctx = (i, hex(int(r.row_path[i].item()) & 0xFFFFFFFF))
        assert (tok[i], con[i], kc[i]) == (o.token, o.consumed, o.kept_count), ctx
        k = min(o.kept_count, 64)
        assert np.array_equal(ids[i, :k], o.kept_ids()[:k]), ctx
        if exact:
            st, pr = r.row_stats[i].cpu().numpy(), r.kept_probs[i, :k].cpu().numpy()
            assert _same(st[[0, 1, 3]], [o.max_logit, o.sum, o.total]), ctx
            assert st[2] == 0.0 or _same(st[2], o.entropy), ctx
            assert _same(pr, o.probs[ids[i, :k]]), ctx
    return r.row_path.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("n,offset,pad", [(129028, 0, 0), (129025, 1, 0), (131075, 3, 5), (151936, 0, 0),
                                          (262143, 2, 1), (262144, 0, 0), (262145, 1, 0)])
@pytest.mark.parametrize("params", [FILTERS, DEFAULT, FULL], ids=["filters", "default", "full"])
def test_long_rows_token_call(n, offset, pad, params):
    path = _check(_rows(n, 1), params, offset=offset, pad=pad)
    if params is FILTERS and n <= 262144:
        assert path[0] & llz.PATH_TOKEN_ONLY and path[1] & llz.PATH_TOKEN_ONLY


def test_long_rows_exact_call():
    _check(_rows(140001, 2), FILTERS, exact=True)


@pytest.mark.parametrize("n", [129028, 200003])
@pytest.mark.parametrize("post,window", [((0.0, 0.5), 0), ((30.0, 0.5), 0), ((0.0, 1.0), 40), ((30.0, 1.0), 64),
                                         ((0.0, 1.0), 200)])
def test_long_rows_transforms(n, post, window):
    x = _rows(n, 3)
    g = np.random.default_rng(n)
    prev, params = None, FILTERS
    if window:
        params = dataclasses.replace(FILTERS, repetition_window=window, repetition_penalty=1.3)
        prev = g.integers(0, n + 50, size=(x.shape[0], window)).astype(np.uint32)
        prev[:, 0] = np.nanargmax(x, axis=1)
        prev[:, 1] = n - 1
        prev[:, 2] = prev[:, 0]
    _check(x, params, post=llz.LogitPost(*post), prev=prev)


@pytest.mark.parametrize("n", [4099, 60000, 129028, 151936])
def test_typical_alone(n):
    """A heavy tail with strong tokens cuts inside the list; flatter rows past it."""
    g = np.random.default_rng(n)
    x = g.gumbel(0.0, 1.5, size=(6, n)).astype(np.float32)
    for r in range(3):
        x[r, g.choice(n, 20, replace=False)] += np.float32(8.0)
    x[4] = g.normal(0.0, 0.3, n).astype(np.float32)
    x[5] = np.round(x[5])  # many equal devs
    path = _check(x, TYPICAL)
    assert not np.any(path[:3] & llz.PATH_FULL_SORT), path
    assert path[4] & llz.PATH_FULL_SORT
    for p in (0.3, 0.999):
        _check(x, dataclasses.replace(TYPICAL, typical_p=p), exact=True)


@pytest.mark.parametrize("n,pad", [(4096, 0), (30001, 0), (50000, 3), (129024, 0)])
@pytest.mark.parametrize("params", [FILTERS, DEFAULT, FULL, dataclasses.replace(DEFAULT, top_k=50)],
                         ids=["filters", "default", "full", "topk"])
def test_more_rows_than_cus(n, pad, params):
    """k_tok over 300 rows: decided, flooded (all equal, flat), NaN, infinite
    and penalised rows, more candidates than the list holds under top-k."""
    rows = 300
    g = np.random.default_rng(n)
    base = _rows(n, 4)
    base = np.concatenate([base, g.normal(0.0, 2.0, size=(4, n)).astype(np.float32),
                           g.normal(0.0, 0.3, size=(1, n)).astype(np.float32)])
    pick = g.integers(0, base.shape[0], rows)
    pick[:base.shape[0]] = np.arange(base.shape[0])
    x = base[pick]
    u = llz.rng_uniforms(9, rows)
    for window in (0, 32):
        p = dataclasses.replace(params, repetition_window=window, repetition_penalty=1.2 if window else 1.0)
        prev = g.integers(0, n, size=(rows, 32)).astype(np.uint32)
        flat = torch.empty(rows, n + pad, dtype=torch.float32, device="cuda")
        flat[:, :n].copy_(torch.from_numpy(x))
        r = llz.sample_rows(flat[:, :n], llz.SamplerConfig.of(p), torch.from_numpy(u).cuda(),
                            torch.from_numpy(prev.astype(np.int32)).cuda(), kept_cap=64, probs=False, path=True)
        torch.cuda.synchronize()
        tok, con, kc, _ = _oracle_rows(x, p, u, prev)
        assert np.array_equal(r.tokens.cpu().numpy().view(np.uint32), tok)
        assert np.array_equal(r.consumed.cpu().numpy(), con)
        assert np.array_equal(r.kept_count.cpu().numpy().view(np.uint32), kc)
        path = r.row_path.cpu().numpy().view(np.uint32)
        assert not np.any(path & 0x80000000)


def _oracle_rows(x, p, u, prev):
    tok, con, kept = O.sample_rows(x, p, u, prev_tokens=prev, threads=16)
    return tok, con, kept, None


@pytest.mark.parametrize("params,n", [(FILTERS, 20000), (FULL, 20000), (DEFAULT, 20000), (FILTERS, 131076)],
                         ids=["token rows", "k_tok", "claimed rows", "claimed long rows"])
def test_replayed_calls_of_more_rows_than_cus(params, n):
    """A captured call's replays carry one epoch: every replay samples every
    row of the logits it finds, also beyond the grid."""
    rows = 800 if n < 100000 else 300
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.empty(rows, n, device="cuda")
    u = torch.rand(rows, generator=g, device="cuda")
    call = llz.PreparedCall(rows, n, llz.SamplerConfig.of(params), "cuda:0")
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        captured = llz.PreparedCall(rows, n, llz.SamplerConfig.of(params), "cuda:0", stream=side)
        x.normal_(0.0, 2.5, generator=g)
        captured(x, u)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            captured(x, u)
    for _ in range(4):
        x.normal_(0.0, 2.5, generator=g)
        torch.cuda.synchronize()
        want = call(x, u)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured.result.tokens, want.tokens)
        assert torch.equal(captured.result.consumed, want.consumed)


def test_replays_list_undecided_rows_anew():
    """k_tok's list of undecided rows is one replay's own: rows left undecided
    by one replay and decided by the next are not sampled a second time."""
    rows, n = 600, 20000  # (every filter: k_tok's call at any number of rows)
    side = torch.cuda.Stream()
    x = torch.empty(rows, n, device="cuda")
    u = torch.rand(rows, device="cuda")
    cfg = llz.SamplerConfig.of(FULL)
    eager = llz.PreparedCall(rows, n, cfg, "cuda:0")
    with torch.cuda.stream(side):
        captured = llz.PreparedCall(rows, n, cfg, "cuda:0", stream=side)
        x.normal_(0.0, 2.5)
        captured(x, u)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            captured(x, u)
    # the workspace's last section: the list's length, then (256 bytes on) the list
    section = captured.workspace[-(-(-(256 + rows * 4) // 256) * 256):]
    length, rows_listed = section[:8].view(torch.int64), section[256:256 + rows * 4].view(torch.int32)
    hot = torch.empty(rows, n, device="cuda").normal_(0.0, 2.5)
    flat = torch.full((rows, n), 0.5, device="cuda")  # every row's candidates overflow its buffers
    half = torch.where(torch.arange(rows, device="cuda")[:, None] % 2 == 0, hot, flat)
    for logits, left in ((flat, rows), (hot, 0), (half, rows // 2), (hot, 0), (flat, rows)):
        x.copy_(logits)
        rows_listed.fill_(-1)
        torch.cuda.synchronize()
        want = eager(x, u).tokens.clone()
        captured.result.tokens.fill_(-5)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured.result.tokens, want)
        assert length.item() == 0
        listed = rows_listed[rows_listed >= 0].sort().values
        assert torch.equal(listed, listed.unique())
        assert left <= listed.numel() <= left + rows // 50  # (a few hot rows' cuts are too close to call)


@pytest.mark.parametrize("n,pad", [(4096, 0), (9001, 2)])
def test_many_rows_without_typical(n, pad):
    """k_tok's calls without typical-p: eight rounds of rows and more."""
    rows = 8 * 256 + 37
    g = np.random.default_rng(n)
    base = np.concatenate([_rows(n, 6), g.normal(0.0, 2.0, size=(40, n)).astype(np.float32)])
    x = base[g.integers(0, base.shape[0], rows)]
    u = llz.rng_uniforms(3, rows)
    prev = g.integers(0, n, size=(rows, 32)).astype(np.uint32)
    for window in (0, 32):
        p = dataclasses.replace(FILTERS, repetition_window=window, repetition_penalty=1.2 if window else 1.0)
        flat = torch.empty(rows, n + pad, dtype=torch.float32, device="cuda")
        flat[:, :n].copy_(torch.from_numpy(x))
        r = llz.sample_rows(flat[:, :n], llz.SamplerConfig.of(p), torch.from_numpy(u).cuda(),
                            torch.from_numpy(prev.astype(np.int32)).cuda(), kept_cap=8, probs=False)
        torch.cuda.synchronize()
        tok, con, kc, _ = _oracle_rows(x, p, u, prev)
        assert np.array_equal(r.tokens.cpu().numpy().view(np.uint32), tok)
        assert np.array_equal(r.consumed.cpu().numpy(), con)
        assert np.array_equal(r.kept_count.cpu().numpy().view(np.uint32), kc)
