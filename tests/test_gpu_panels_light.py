"""Small batches of light systems on data with panels: nearly every tile goes bin by bin, and the
bin-by-bin kernel takes more rows per work item than the host chose.  Each row has the value it has in
every other batch, whatever shares its items, to the last bit, and with the rows per item fixed."""

import numpy as np
import pytest

from tests._setup import add_to_core, inj_row, make_detector, particle_cloud

pytestmark = pytest.mark.gpu

T = 4.0e6


@pytest.mark.parametrize("modes", [("22",), ("22", "33", "44")])
def test_light_systems_in_any_batch(modes):
    from oracle import cpu_baseline as cb
    from pespace_amd.core import LikelihoodCore
    lm = tuple((int(m[0]), int(m[1])) for m in modes)
    interp = (1e-4, 0.05, 1024)
    d, labels = make_detector(T=T, modes=lm, interp=interp)
    core = LikelihoodCore(modes=modes, n_nodes=1024, f_node_min=1e-4, f_node_max=0.05)
    add_to_core(core, d, labels)
    assert core.panel_tiles[0] >= 512
    rows = particle_cloud(1000, seed=95, rel=1e-4, center=inj_row(chirp_mass=30.0, coalescence_time=0.7 * T))
    rows[40:60] = particle_cloud(20, seed=96, rel=1e-3, center=inj_row(coalescence_time=0.7 * T))
    lnl, g = (x.cpu().numpy() for x in core.lnl(rows, grad=True))
    l0 = core.lnl(rows).cpu().numpy()
    ref = [cb.lnl_row(cb.Network([d]), cb.RowInputs(rows[i], lm, 0.0, interp), threads=4) for i in (0, 50)]
    ref = [r[0] if isinstance(r, tuple) else r for r in ref]
    np.testing.assert_allclose(lnl[[0, 50]], ref, rtol=1e-10)
    for a, b in ((0, 1), (0, 8), (30, 47), (0, 64), (45, 50)):
        lp, gp = (x.cpu().numpy() for x in core.lnl(rows[a:b], grad=True))
        np.testing.assert_array_equal(lp, lnl[a:b])
        np.testing.assert_array_equal(gp, g[a:b])
        np.testing.assert_array_equal(core.lnl(rows[a:b]).cpu().numpy(), l0[a:b])
    for r in (1, 5, 48):
        core.set_schedule(8, 4, r)
        lp, gp = (x.cpu().numpy() for x in core.lnl(rows[:64], grad=True))
        np.testing.assert_array_equal(lp, lnl[:64])
        np.testing.assert_array_equal(gp, g[:64])
