"""Whittle sum at the edges of its two-pass reduction: fewer bins than one block, one block and its
neighbours, the last size at which every bin has a thread of its own, and sizes beyond it."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

THREADS = 256 * 1024  # threads of the largest grid


@pytest.mark.parametrize("n_chan", [1, 3])
@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 1025, THREADS - 1, THREADS, THREADS + 1, 2 * THREADS + 77])
def test_whittle_reduction_edges(n, n_chan):
    from pespace_amd.core import whittle_lnl

    g = np.random.default_rng(n + 7 * n_chan)
    d = g.standard_normal((n_chan, n)) + 1j * g.standard_normal((n_chan, n))
    h = g.standard_normal((n_chan, n)) + 1j * g.standard_normal((n_chan, n))
    s = g.uniform(0.5, 2.0, (n_chan, n))
    df = 0.125
    got = whittle_lnl(torch.tensor(d, device="cuda"), torch.tensor(h, device="cuda"), torch.tensor(s, device="cuda"), df)
    x = d - h
    ref = -2.0 * df * math.fsum(((x.real * x.real + x.imag * x.imag) / s).ravel())
    # all terms have one sign: each is rounded at most five times (two differences' squares, their
    # sum, the quotient) and passes through at most n_chan * ceil(n / THREADS) + 6 + 2 + 2 + 6 + 2
    # additions and two products, each within 2^-53
    adds = n_chan * math.ceil(n / THREADS) + 18 + 2
    assert abs(float(got) - ref) <= (2 * 5 + adds) * 2.0**-53 * abs(ref)
    again = whittle_lnl(torch.tensor(d, device="cuda"), torch.tensor(h, device="cuda"), torch.tensor(s, device="cuda"), df)
    assert float(again) == float(got)
