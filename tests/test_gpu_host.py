"""The host sampler over a decode loop's history, which grows by a token per
step: the tokens of the reference's chain with the same PRNG at every step,
and no step that pays for new buffers."""
import dataclasses
import time

import numpy as np
import pytest

import oracle_lib as O
from llz.workloads import WORKLOADS

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _logits(n, count, seed):
    g = np.random.default_rng([n, seed])
    x = g.normal(0.0, 2.0, size=(count, n)).astype(np.float32)
    x[:, g.choice(n, 6, replace=False)] += np.float32(9.0)
    return x


@pytest.mark.parametrize("window", [0, 5, 32, 64, 70, 0xFFFFFFFF])
@pytest.mark.parametrize("temperature", [0.0, 0.8])
def test_growing_history(window, temperature):
    import llz

    n, steps = 4099, 150
    p = dataclasses.replace(WORKLOADS["c1"].params, temperature=temperature, repetition_window=window,
                            repetition_penalty=1.4)
    x = _logits(n, 4, window & 0xFF)
    s = llz.Sampler(dataclasses.replace(llz.SamplerConfig.of(p), seed=7))
    o = O.Sampler(p, 7)
    hist = []
    for i in range(steps):
        t = s.sample(x[i % 4], hist)
        assert t == o.sample(x[i % 4], hist), i
        assert s.state == o.state, i
        hist.append(t)


def test_growing_history_costs_no_buffers():
    """Steps with a growing history against steps with one of constant length:
    a step that freed and allocated its pinned and device buffers would take
    several times as long."""
    import llz

    n = 128256
    x = _logits(n, 1, 1)[0]
    cfg = llz.SamplerConfig(temperature=0.8, top_k=40, top_p=0.9, min_p=0.05, repetition_window=32, repetition_penalty=1.1)

    def median(grow):
        s = llz.Sampler(cfg)
        hist = np.arange(400, dtype=np.uint32)
        s.sample(x, hist[:40])
        took = []
        for i in range(300):
            t0 = time.perf_counter()
            s.sample(x, hist[: 40 + (i if grow else 0)])
            took.append(time.perf_counter() - t0)
        return sorted(took)[150]

    fixed = median(False)
    grown = median(True)
    print(f"fixed {fixed * 1e6:.1f} us, grown {grown * 1e6:.1f} us")
    assert grown < 1.5 * fixed
