"""The exact phases on rows of odd lengths and alignments whose segments lie
partly in LDS (past 92160 logits), and candidate lists with long runs of equal
terms, every output against the oracle."""
import dataclasses

import numpy as np
import pytest

import llz
from llz.workloads import Params
from test_gpu_range import _check

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

FILTERS = Params(1.0, 40, 0.95, 0.05, 1.0, 0, 1.0)
DEFAULT = Params(0.8, 0, 0.9, 0.0, 1.0, 0, 1.0)


def _rows(n, seed):
    g = np.random.default_rng([n, seed])
    x = g.normal(0.0, 2.0, size=(5, n)).astype(np.float32)
    x[0, g.choice(n, 8, replace=False)] += np.float32(12.0)
    x[1, n - 3:] = (9.0, 11.0, 10.0)             # the largest lie in the row's last n % 4
    x[2, -1] = np.inf
    x[3, -1] = np.nan
    x[4] -= (1.1 * np.log(g.permutation(n) + 1.0)).astype(np.float32)
    return x


@pytest.mark.parametrize("exact", [False, True], ids=["token", "exact"])
@pytest.mark.parametrize("n,offset", [(92159, 0), (92161, 1), (92163, 0), (94207, 2), (100001, 3), (110594, 0),
                                      (129021, 0), (129023, 1), (129024, 3)])
@pytest.mark.parametrize("params", [FILTERS, DEFAULT], ids=["filters", "default"])
def test_unaligned_rows_past_the_registers(n, offset, params, exact):
    _check(_rows(n, 7), params, offset=offset, exact=exact)


@pytest.mark.parametrize("exact", [False, True], ids=["token", "exact"])
@pytest.mark.parametrize("count", [25, 130, 600, 1900])
@pytest.mark.parametrize("typical", [1.0, 0.9])
def test_lists_with_long_runs_of_equal_terms(count, typical, exact):
    """Runs too long for the bins of the list's sort, among others."""
    n = 50003
    g = np.random.default_rng(count)
    x = g.normal(-8.0, 1.0, size=(3, n)).astype(np.float32)
    for r in range(3):
        at = g.choice(n, count + 200, replace=False)
        x[r, at[:count]] = np.float32(1.0) if r < 2 else np.round(g.normal(1.0, 0.2, count), 1)  # one value, or a few
        x[r, at[count:]] = g.normal(1.0, 0.5, 200) if r else np.float32(0.5)
    _check(x, dataclasses.replace(DEFAULT, temperature=1.0, typical_p=typical), exact=exact)
    _check(x, dataclasses.replace(DEFAULT, temperature=1.0, typical_p=typical, top_k=count + 50, top_p=1.0), exact=exact)
