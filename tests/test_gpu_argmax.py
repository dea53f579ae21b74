"""Greedy rows read by several workgroups (k_argmax) against sampleArgmax
(sampler.zig:31-41) by the oracle: chunk edges and remainders, unaligned rows,
ties across chunks, NaN and infinities, and whatever the token words held
before the call (the chunks combine through them)."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _argmax(x_dev, fill):
    import llz

    rows, n = x_dev.shape
    tok = torch.full((rows,), fill, dtype=torch.int64, device="cuda").to(torch.int32)
    rc = llz.library().llz_argmax_rows(C.c_void_p(x_dev.data_ptr()), x_dev.stride(0), rows, n, None,
                                       C.c_void_p(tok.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    return tok.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("n", [1, 3, 4, 4095, 4096, 4097, 8191, 8193, 50021, 131075])
@pytest.mark.parametrize("rows,offset", [(1, 0), (3, 1), (300, 3)])
def test_argmax_chunks(n, rows, offset):
    g = np.random.default_rng([n, rows])
    x = g.integers(-40, 41, size=(rows, n)).astype(np.float32)  # many equal maxima, in every chunk
    for r in range(rows):
        k = r % 6
        if k == 1:
            x[r, g.integers(0, n, size=max(1, n // 3))] = np.nan  # NaN never wins past index 0
        elif k == 2:
            x[r, 0] = np.nan  # and is never replaced at index 0
        elif k == 3:
            x[r] = -np.inf
        elif k == 4:
            x[r] = np.where(g.random(n) < 0.5, np.float32(0.0), np.float32(-0.0))  # one value: the first index
        elif k == 5:
            x[r, g.integers(0, n)] = np.inf
    if rows >= 300:
        x[7] = np.nan
        x[8, 1:] = np.nan
        x[8, 0] = -np.inf
    want = np.array([O.lib().llz_oracle_argmax(O._fptr(x[r]), n) for r in range(rows)], np.uint32)
    flat = torch.zeros(rows * (n + 2) + 4, dtype=torch.float32, device="cuda")
    xd = flat[offset:offset + rows * (n + 2)].view(rows, n + 2)[:, :n]
    xd.copy_(torch.from_numpy(x))
    for fill in (0, n - 1, -1, n, 0x7FFFFFFF):
        assert np.array_equal(_argmax(xd, fill), want), fill


@pytest.mark.parametrize("n", [2**31 - 1, 2**31 - 4096])
def test_argmax_longest_rows(n):
    """Chunk positions past the end of the longest rows stay above it."""
    x = torch.full((1, n), -1.0, dtype=torch.float32, device="cuda")
    for at in (n - 1, n // 2):
        x[0, at] = x[0, at] + 2.0 + (n - at) * 1e-9
        assert _argmax(x, 0)[0] == at


@pytest.mark.parametrize("rows,n", [(1, 50021), (3, 131075), (300, 8193)])
def test_argmax_tokens_in_host_memory(rows, n):
    """Tokens in pinned host memory are stored, not combined through the word
    (argmax_rows and greedy rows of llz_sample_rows)."""
    import llz

    g = np.random.default_rng(n)
    x = torch.from_numpy(g.integers(-40, 41, size=(rows, n)).astype(np.float32)).cuda()
    want = np.array([O.lib().llz_oracle_argmax(O._fptr(r), n) for r in x.cpu().numpy()], np.uint32)
    tok = torch.full((rows,), -1, dtype=torch.int32, pin_memory=True)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    args = (C.c_void_p(x.data_ptr()), n, rows, n)
    assert llz.library().llz_argmax_rows(*args, None, C.c_void_p(tok.data_ptr()), st) == 0
    torch.cuda.synchronize()
    assert np.array_equal(tok.numpy().view(np.uint32), want)
    tok.fill_(n - 1)
    cfg = llz.SamplerConfig(temperature=0.0).to_c()
    assert llz.library().llz_sample_rows(*args, C.byref(cfg), None, None, 0, 0, None, C.c_void_p(tok.data_ptr()), None,
                                         None, None, 0, st) == 0
    torch.cuda.synchronize()
    assert np.array_equal(tok.numpy().view(np.uint32), want)


def test_argmax_replayed():
    import llz

    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.empty(8, 50021, device="cuda").normal_(0.0, 2.0, generator=g)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        llz.argmax_rows(x)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            tok = llz.argmax_rows(x)
    for _ in range(4):
        x.normal_(0.0, 2.0, generator=g)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(tok.long(), x.argmax(1))
