"""The panel kernel against the bin-by-bin kernel on the same data.

A grid of more than 512 tiles with panels goes by panels; cut at tile ends into contexts of fewer
tiles each, all of it goes bin by bin, and the contexts' lnL and gradients add up to the whole's.

Tolerances: both sides are FP64 sums over the same bins.  The panels' truncation is ~3e-15 of the
panel's largest response and a bin's roundings are ~1e-15 of its terms; lnL is a sum of terms of one
sign: 1e-13 relative.  A gradient's sums cancel by up to three orders of magnitude (as in
test_gpu_panels): 1e-11 of each parameter's largest component over the batch.
"""

import numpy as np
import pytest

from tests._setup import ORBIT_KIND, inj_row, make_detector, particle_cloud, prior_rows

pytestmark = pytest.mark.gpu

T = 4.0e6
INTERP = (1e-4, 0.06, 1024)
TIANQIN = dict(orbit="Tianqin_analytic", psd_model="Tianqin_GWSpace", fmin=1e-3, fmax=0.05)
CASES = [
    (dict(fmax=0.05), ("22", "21", "33", "32", "44", "43")),
    (dict(TIANQIN, duty=(1.0e6, 6.0e5, 2.0e5, 3.0e4)), ("22", "33", "44")),
    (dict(orbit="Taiji_analytic", psd_model="Taiji_TDC", fmax=0.06, gen="2.0", orthogonal=False), ("22",)),
]


def _core(d, labels, modes, first, last):
    from pespace_amd.core import LikelihoodCore
    core = LikelihoodCore(modes=modes, n_nodes=INTERP[2], f_node_min=INTERP[0], f_node_max=INTERP[1])
    kind, arm, rot0, rev0 = d.orbit[:4]
    geo = dict(zip(("omega_rotation", "lambda_ref", "beta_ref"), d.orbit[4:]))
    core.add_detector(ORBIT_KIND[kind], arm, rot0, rev0, 15 if d.tdi_generation == "1.5" else 20, d.orthogonal,
                      d.f[first:last], np.stack([d.data[c] for c in labels])[:, first:last],
                      np.stack([d.psd[c] for c in labels])[:, first:last], [1 if c in d.channels else 0 for c in labels],
                      df=d.df, duty_cycle=getattr(d, "duty", None), **geo)
    return core


@pytest.mark.parametrize("case", range(len(CASES)))
def test_panels_match_bins(case):
    kw, modes = CASES[case]
    d, labels = make_detector(T=T, dt=5.0, modes=tuple((int(m[0]), int(m[1])) for m in modes), interp=INTERP, seed=90, **kw)
    near = inj_row(coalescence_time=0.7 * T)
    rows = np.vstack([particle_cloud(9, seed=91, rel=1e-3, center=near), prior_rows(6, seed=92, tc_range=(0.0, T))])
    whole = _core(d, labels, modes, 0, d.f.size)
    assert whole.panel_tiles[0] >= 512
    lnl, g = (x.cpu().numpy() for x in whole.lnl(rows, grad=True))
    step = 500 * 256
    lnl_b, g_b = 0.0, 0.0
    for a in range(0, d.f.size, step):
        part = _core(d, labels, modes, a, min(a + step, d.f.size))
        assert part.panel_tiles == [0]
        l, gr = (x.cpu().numpy() for x in part.lnl(rows, grad=True))
        lnl_b, g_b = lnl_b + l, g_b + gr
    err_l, err_g = np.abs(lnl / lnl_b - 1), np.abs(g - g_b) / np.abs(g_b).max(axis=0)
    print(f"case {case}: {whole.n_bins} bins, {whole.panel_tiles} tiles with panels, lnL {err_l.max():.1e}, "
          f"gradient {err_g.max():.1e}", flush=True)
    assert err_l.max() < 1e-13
    assert err_g.max() < 1e-11


@pytest.mark.parametrize("modes", [("22",), ("22", "33")])
@pytest.mark.parametrize("duty", [None, (1.0e6, 6.0e5, 2.0e5, 3.0e4)])
def test_lnl_alone_of_short_panels(modes, duty):
    """Where panels hold few bins lnL alone of one mode goes bin by bin and the gradient by panels (LISA
    over 3.1e6 s; TianQin's panels are longer): the same lnL up to rounding, and each the same in every
    batch, to the last bit."""
    d, labels = make_detector(T=4.0e6 if duty else 3.1e6, dt=5.0, modes=tuple((int(m[0]), int(m[1])) for m in modes), interp=INTERP, seed=93,
                              **(dict(TIANQIN, duty=duty) if duty else {}))
    core = _core(d, labels, modes, 0, d.f.size)
    assert core.panel_tiles[0] >= 512
    rows = np.vstack([particle_cloud(900, seed=94, rel=1e-3, center=inj_row(coalescence_time=0.7 * T)),
                      prior_rows(200, seed=95, tc_range=(0.0, T))])[np.random.default_rng(1).permutation(1100)]
    lnl = core.lnl(rows).cpu().numpy()
    np.testing.assert_allclose(core.lnl(rows, grad=True)[0].cpu().numpy(), lnl, rtol=1e-13)
    for a, b in ((0, 1), (3, 8), (0, 90), (100, 330), (0, 700)):
        np.testing.assert_array_equal(core.lnl(rows[a:b]).cpu().numpy(), lnl[a:b])
