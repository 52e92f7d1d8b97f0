"""Networks of which one run of detectors (an orbit kind of its own) has no tile with panels while
another has: long LISA data beside short TianQin data, whose tiles all go bin by bin.

Small batches run one panel per work item there and have no such item in TianQin's run; the last
batch is large enough for items of whole groups.  Tolerances as in test_gpu_panels: lnL 1e-10
relative, gradient 2e-6 of each parameter's largest component (the oracle differentiates the node
tables by finite differences); a row's values are the same to the last bit in every batch.
"""

import numpy as np
import pytest

from tests._setup import add_to_core, inj_row, make_detector, particle_cloud

pytestmark = pytest.mark.gpu

T = 4.0e6
INTERP = (1e-4, 0.06, 1024)
MODES = ((2, 2), (3, 3))


@pytest.mark.parametrize("order", [0, 1])
def test_run_of_detectors_without_panels(order):
    from oracle import cpu_baseline as cb
    from pespace_amd.core import LikelihoodCore
    long = make_detector(T=T, modes=MODES, interp=INTERP, seed=31)
    short = make_detector(orbit="Tianqin_analytic", psd_model="Tianqin_GWSpace", fmin=1e-3, fmax=0.039, T=2.0e5,
                          modes=MODES, interp=INTERP, seed=32)
    made = [long, short] if order == 0 else [short, long]
    core = LikelihoodCore(modes=[f"{l}{m}" for l, m in MODES], n_nodes=INTERP[2], f_node_min=INTERP[0],
                          f_node_max=INTERP[1])
    for d, labels in made:
        add_to_core(core, d, labels)
    rows = particle_cloud(1000, seed=33, rel=1e-3, center=inj_row(coalescence_time=0.7 * T))
    print(f"bins {core.n_bins}", flush=True)
    lnl, g = (x.cpu().numpy() for x in core.lnl(rows, grad=True))
    net = cb.Network([d for d, _ in made])
    ref = [cb.lnl_row(net, cb.RowInputs(rows[i], MODES, 0.0, INTERP, grad=True), grad=True, threads=4)
           for i in range(4)]
    ref_l, ref_g = np.array([r[0] for r in ref]), np.stack([r[1] for r in ref])
    np.testing.assert_allclose(lnl[:4], ref_l, rtol=1e-10)
    assert np.max(np.abs(g[:4] - ref_g) / np.abs(ref_g).max(axis=0)) < 2e-6
    full = core.lnl(rows).cpu().numpy()
    np.testing.assert_allclose(full, lnl, rtol=1e-12)
    for p in (1, 16, 64):
        lp, gp = (x.cpu().numpy() for x in core.lnl(rows[:p], grad=True))
        np.testing.assert_array_equal(lp, lnl[:p])
        np.testing.assert_array_equal(gp, g[:p])
        np.testing.assert_array_equal(core.lnl(rows[:p]).cpu().numpy(), full[:p])
