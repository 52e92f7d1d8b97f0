"""Rows spread over the prior on a duty-cycled detector's long data: most tiles have some row that goes
bin by bin (a window edge or a mode's cut in the tile), and few rows of a work item do.

The rows of an item are found 64 at a time, and its duty flags by waves that hold several items: each row
has the value it has alone to the last bit, in items of 1 to 160 rows, small batches and large ones.  Only
the duty-cycled gradient may differ in its rounding, since an item with one row on a window's edge takes
its other rows through the window code too: 1e-11 of each parameter's largest component.  lnL is the
oracle's to 1e-10, as in test_gpu_panels."""

import numpy as np
import pytest

from tests._setup import add_to_core, make_detector, prior_rows

pytestmark = pytest.mark.gpu

T = 6.0e6
INTERP = (1e-4, 0.05, 1024)
DUTY = (3.0e6, 1.6e6, 2.0e5, 2.0e4)


@pytest.mark.parametrize("duty", [DUTY, None])
@pytest.mark.parametrize("modes", [((2, 2),), ((2, 2), (3, 3), (4, 4))])
def test_spread_rows_in_any_items(modes, duty):
    from oracle import cpu_baseline as cb
    from pespace_amd.core import LikelihoodCore
    d, labels = make_detector(orbit="Tianqin_analytic", psd_model="Tianqin_GWSpace", fmin=1e-3, fmax=0.039, T=T,
                              modes=modes, interp=INTERP, duty=duty)
    core = LikelihoodCore(modes=[f"{l}{m}" for l, m in modes], n_nodes=INTERP[2], f_node_min=INTERP[0],
                          f_node_max=INTERP[1])
    add_to_core(core, d, labels)
    assert core.panel_tiles[0] >= 512
    rows = prior_rows(900, seed=41, tc_range=(0.0, T))
    lnl, g = (x.cpu().numpy() for x in core.lnl(rows, grad=True))
    l0 = core.lnl(rows).cpu().numpy()
    assert np.all(np.isfinite(lnl)) and np.all(np.isfinite(g))
    ref = [cb.lnl_row(cb.Network([d]), cb.RowInputs(rows[i], modes, 0.0, INTERP), threads=4) for i in range(6)]
    ref = [r[0] if isinstance(r, tuple) else r for r in ref]
    np.testing.assert_allclose(lnl[:6], ref, rtol=1e-10)
    np.testing.assert_allclose(l0, lnl, rtol=1e-12)

    def same_grad(a, b):
        if duty is None:
            np.testing.assert_array_equal(a, b)
        else:
            assert np.max(np.abs(a - b) / np.abs(g).max(axis=0)) <= 1e-11

    parts = [(i, i + 1) for i in range(8)] + [(100, 165), (0, 120), (130, 430)]
    for a, b in parts:
        lp, gp = (x.cpu().numpy() for x in core.lnl(rows[a:b], grad=True))
        np.testing.assert_array_equal(lp, lnl[a:b])
        same_grad(gp, g[a:b])
        np.testing.assert_array_equal(core.lnl(rows[a:b]).cpu().numpy(), l0[a:b])
    for r in (3, 33, 64, 65, 160):
        core.set_schedule(8, 4, r)
        for n in (900, 131):
            lp, gp = (x.cpu().numpy() for x in core.lnl(rows[:n], grad=True))
            np.testing.assert_array_equal(lp, lnl[:n])
            same_grad(gp, g[:n])
            np.testing.assert_array_equal(core.lnl(rows[:n]).cpu().numpy(), l0[:n])
