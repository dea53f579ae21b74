"""The host sampler on pinned logits and history that work queued on the
default stream still writes (a decoder's non-blocking copies): the call reads
them behind that work, as its copies on its own stream always did."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 32003, 128256])
def test_pinned_inputs_behind_default_stream(n):
    import llz

    g = np.random.default_rng(n)
    x = g.normal(0.0, 3.0, n).astype(np.float32)
    prev = g.integers(0, n, 8).astype(np.int32)
    x[int(np.argmax(x))] += 2.0
    prev[3] = int(np.argmax(x))  # the penalty moves the likeliest token
    old = np.zeros(n, np.float32)
    old[(int(np.argmax(x)) + 1) % n] = 50.0  # what a call that does not wait would sample
    cfg = llz.SamplerConfig(temperature=0.8, top_k=40, top_p=0.9, repetition_window=32, repetition_penalty=4.0)
    s = llz.Sampler(cfg)
    us = (0.1, 0.6, 0.95)
    want = [s.sample_uniform(x, u, prev.view(np.uint32)) for u in us]
    xd, pd = torch.from_numpy(x).cuda(), torch.from_numpy(prev).cuda()
    px = torch.empty(n, dtype=torch.float32, pin_memory=True)
    pp = torch.empty(8, dtype=torch.int32, pin_memory=True)
    busy = torch.zeros(1 << 28, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    for u, w in zip(us, want):
        px.copy_(torch.from_numpy(old))
        pp.zero_()
        for _ in range(20):
            busy.add_(1.0)  # some milliseconds of the default stream
        px.copy_(xd, non_blocking=True)
        pp.copy_(pd, non_blocking=True)
        assert s.sample_uniform(px, u, pp.numpy().view(np.uint32)) == w
