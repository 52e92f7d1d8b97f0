"""HIP graphs of the batched lnL + gradient and the schedule, on contexts with panels (long data:
k_panel_class lists the bin-by-bin work on the device, batch by batch) and without (short data),
for batches whose work items are single tiles and panels and for larger ones.

Every replay equals the eager result of its rows to the last bit, also after the context's schedule
was changed (the graph keeps the tile groups that it was captured with), and a schedule may be set
while a stream is being captured.
"""

import numpy as np
import pytest
import torch

from tests._setup import add_to_core, inj_row, make_detector, particle_cloud, prior_rows

pytestmark = pytest.mark.gpu

TIANQIN = dict(orbit="Tianqin_analytic", psd_model="Tianqin_GWSpace", fmin=1e-3, fmax=0.039)


def _core(span, modes):
    from pespace_amd.core import LikelihoodCore
    core = LikelihoodCore(modes=[f"{l}{m}" for l, m in modes], n_nodes=1024, f_node_min=1e-4, f_node_max=0.05)
    for kw in (dict(), dict(TIANQIN, duty=(0.5 * span, 0.3 * span, 0.1 * span, 0.01 * span))):
        add_to_core(core, *make_detector(T=span, modes=modes, interp=(1e-4, 0.05, 1024), **kw))
    return core


@pytest.mark.parametrize("span", [4.0e6, 655360.0])
@pytest.mark.parametrize("P", [5, 1000])
def test_replays_keep_their_groups(span, P):
    core = _core(span, ((2, 2), (3, 3)))
    center = inj_row(coalescence_time=0.7 * span)
    batches = [np.vstack([particle_cloud(P - 2, seed=40 + k, rel=1e-3, center=center),
                          prior_rows(2, seed=50 + k, tc_range=(0.0, span))]) for k in range(3)]
    for per in (1, 11):  # scratch for the most groups and for the largest batch of single tiles
        core.set_schedule(per, 4)
        core.reserve(P, grad=True)
    core.pin_scratch(True)
    eager = {}
    for per in (8, 3, 11):
        core.set_schedule(per, 4)
        eager[per] = [tuple(t.clone() for t in core.lnl(rows, grad=True)) for rows in batches]
        if per != 8:  # another order of the partial sums
            assert torch.allclose(eager[per][0][0], eager[8][0][0], rtol=1e-12, atol=0.0)
    core.set_schedule(8, 4)
    x = torch.as_tensor(batches[0], device="cuda").contiguous()
    out = [(torch.empty(P, dtype=torch.float64, device="cuda"), torch.empty(P, 11, dtype=torch.float64, device="cuda"))
           for _ in range(2)]
    torch.cuda.synchronize()
    graphs = []
    for per, (lnl, g) in zip((8, 3), out):  # the second graph's schedule is set during its capture
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            core.set_schedule(per, 4)
            core.lnl(x, grad=True, out=lnl, grad_out=g)
        graphs.append(graph)
    print(f"captured span {span:g} P {P}", flush=True)
    for now in (3, 8, 11, 1):
        core.set_schedule(now, 4)
        for k in (1, 2, 0):
            x.copy_(torch.as_tensor(batches[k], device="cuda"))
            for graph, per, (lnl, g) in zip(graphs, (8, 3), out):
                lnl.fill_(np.nan)
                g.fill_(np.nan)
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(lnl, eager[per][k][0]) and torch.equal(g, eager[per][k][1]), (now, per, k)
            if now in eager:
                l_e, g_e = core.lnl(batches[k], grad=True)
                assert torch.equal(l_e, eager[now][k][0]) and torch.equal(g_e, eager[now][k][1]), (now, k)
    core.pin_scratch(False)
    del graphs


@pytest.mark.parametrize("span", [4.0e6, 655360.0])
def test_pinned_scratch_takes_a_schedule_with_fewer_groups(span):
    """Fewer tile groups need no more scratch: more batches count as small then, and those that the
    pinned sums of single tiles have no room for run in items of whole groups."""
    from pespace_amd._lib import PespaceError
    core = _core(span, ((2, 2), (3, 3)))
    P = 1000
    rows = particle_cloud(P, seed=60, rel=1e-3, center=inj_row(coalescence_time=0.7 * span))
    core.set_schedule(4, 4)
    core.reserve(P, grad=True)
    core.pin_scratch(True)
    ref = core.lnl(rows, grad=True)
    for per in (8, 64, 4096):
        core.set_schedule(per, 4)
        lnl, g = core.lnl(rows, grad=True)
        assert torch.allclose(lnl, ref[0], rtol=1e-12, atol=0.0)
        for p in (1, 150):  # batches of single tiles that fit: the same to the last bit
            l_p, g_p = core.lnl(rows[:p], grad=True)
            assert torch.equal(l_p, lnl[:p]) and torch.equal(g_p, g[:p])
    core.set_schedule(1, 4)
    with pytest.raises(PespaceError, match="pinned"):
        core.lnl(rows, grad=True)
    core.pin_scratch(False)
