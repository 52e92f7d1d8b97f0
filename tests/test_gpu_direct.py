"""lnL and gradient of contexts evaluated at every bin (n_nodes = 0) through the direct kernels
(the waveform's values per bin, its adjoint contracted bin by bin), against the kernels that read
node tables: a detector with a duty cycle that is on throughout takes those, with a window of 1.

Grids that end inside a tile, both orbit kinds, one to six modes and modes in another order, TDI 1.5
and 2.0, A/E/T and X/Y/Z, rows near the source and from the wide prior.  Tolerances: the two paths
differ in the waveform's rounding alone, a few 1e-13 of the phase's terms (up to 1e4 rad): 1e-9 rad per
bin at most, so lnL to 1e-11 of itself and the gradient, whose terms cancel by up to three orders, to
1e-8 of each parameter's largest component.
"""

import numpy as np
import pytest

from tests._setup import add_to_core, inj_row, make_detector, particle_cloud, prior_rows

pytestmark = pytest.mark.gpu

T = 655360.0
ALWAYS_ON = (4.0e12, 3.0e12, -1.0e12, 1.0)  # from long before the lightest system enters the band
TIANQIN = dict(orbit="Tianqin_analytic", psd_model="Tianqin_GWSpace", fmin=1e-3, fmax=0.0391)
HM = ((2, 2), (2, 1), (3, 3), (3, 2), (4, 4), (4, 3))
CASES = [
    ([dict(fmax=0.0391)], ((2, 2),)),
    ([dict(fmax=0.0391, gen="2.0", orthogonal=False)], ((3, 3), (2, 2))),
    ([TIANQIN], HM),
    ([dict(fmax=0.02), TIANQIN], ((2, 2), (4, 4), (2, 1))),
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_direct_matches_tables(case):
    from pespace_amd.core import LikelihoodCore
    dets, modes = CASES[case]
    cores = []
    for duty in (None, ALWAYS_ON):
        core = LikelihoodCore(modes=[f"{l}{m}" for l, m in modes], n_nodes=0)
        for i, kw in enumerate(dets):
            d, labels = make_detector(T=T, dt=5.0, modes=modes, seed=31 + i, **dict(kw, duty=duty))
            add_to_core(core, d, labels)
        cores.append(core)
    rows = np.vstack([particle_cloud(5, seed=41, rel=1e-3, center=inj_row()), prior_rows(6, seed=42 + case),
                      inj_row(mass_ratio=1.0)[None]])
    print(f"direct case {case}: bins {cores[0].n_bins}", flush=True)
    (l0, g0), (l1, g1) = [[x.cpu().numpy() for x in c.lnl(rows, grad=True)] for c in cores]
    np.testing.assert_allclose(l0, l1, rtol=1e-11)
    err = np.abs(g0 - g1) / np.abs(g1).max(axis=0)
    print(f"lnl rel {np.max(np.abs(l0 / l1 - 1)):.1e}, gradient {err.max():.1e}")
    assert err.max() < 1e-8
    np.testing.assert_array_equal(cores[0].lnl(rows).cpu().numpy(), l0)
    lp, gp = (x.cpu().numpy() for x in cores[0].lnl(rows[:1], grad=True))
    np.testing.assert_array_equal(lp, l0[:1])
    np.testing.assert_array_equal(gp, g0[:1])


@pytest.mark.parametrize("kind", ["nodes", "direct", "panels"])
def test_small_and_large_batches_agree(kind):
    """Small batches run one tile (or panel) per work item, large ones whole groups of tiles: the same
    values to the last bit on both sides of the line."""
    from pespace_amd.core import LikelihoodCore
    t = 3.0e6 if kind == "panels" else T
    d, labels = make_detector(T=t, dt=5.0, fmax=0.05)
    core = LikelihoodCore(modes=["22"], n_nodes=0 if kind == "direct" else 1024, f_node_min=1e-4, f_node_max=0.05)
    add_to_core(core, d, labels)
    rows = particle_cloud(1030, seed=51, rel=1e-3, center=inj_row(coalescence_time=0.8 * t))
    print(kind, core.n_bins, flush=True)
    lnl, g = (x.cpu().numpy() for x in core.lnl(rows, grad=True))
    for p in (1, 6, 130, 400, 600):
        lp, gp = (x.cpu().numpy() for x in core.lnl(rows[:p], grad=True))
        np.testing.assert_array_equal(lp, lnl[:p])
        np.testing.assert_array_equal(gp, g[:p])
