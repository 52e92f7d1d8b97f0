"""pes_lnl_batch_noalloc on contexts of which one row fills the fixed array: whatever the account
(pes_lnl_batch_noalloc_bytes) accepts runs, though the buffers of a row, with the flags and groups of
the panels and the padded setup table, take more than the array.  A year of data and six modes: the
node grid that fills the array with the gradient still leaves panels of tens of bins.  One mode and
short data: no panels."""

import numpy as np
import pytest
import torch

from tests._setup import YEAR_SI, add_to_core, inj_row, make_detector, particle_cloud

pytestmark = pytest.mark.gpu
LIMIT = 64 << 20
YEAR = (dict(T=YEAR_SI, dt=5.0, fmin=0.03, fmax=0.05, inject=False), ["22", "21", "33", "32", "44", "43"])
SHORT = (dict(T=655360.0, dt=5.0, fmax=0.05), ["22"])


@pytest.mark.parametrize("data,grad", [(YEAR, True), (SHORT, True), (SHORT, False)])
def test_noalloc_one_row_fills_the_array(data, grad):
    from pespace_amd._lib import check, lib
    from pespace_amd.core import LikelihoodCore
    kw, modes = data
    d, labels = make_detector(**kw)

    def build(n_nodes):
        core = LikelihoodCore(modes=modes, n_nodes=n_nodes, f_node_min=1e-4, f_node_max=0.05)
        add_to_core(core, d, labels)
        core.n_bins  # builds the context
        return core, lib().pes_lnl_batch_noalloc_bytes(core._ctx, 1, int(grad))

    def tables(n_nodes):  # the node tables of a row, each rounded up to 256 bytes
        return sum(-(-len(modes) * (n_nodes + 1) * 8 * k // 256) * 256 for k in ((4, 16) if grad else (4,)))

    probe, other = build(1024)
    probe.close()
    other -= tables(1024)
    n = (LIMIT - other) // (len(modes) * 8 * (20 if grad else 4))
    while other + tables(n) > LIMIT:
        n -= 1
    core, need = build(n)
    assert need == other + tables(n) and LIMIT - 1024 < need <= LIMIT
    assert lib().pes_lnl_batch_noalloc_bytes(core._ctx, 2, int(grad)) > LIMIT
    row = particle_cloud(1, seed=81, rel=1e-3, center=inj_row(chirp_mass=2.0e4))
    print(core.n_bins, n, need, flush=True)
    x = torch.as_tensor(row, device="cuda")
    for per in (8, 64):
        core.set_schedule(per, 4)
        ref = core.lnl(row, grad=grad)
        l = torch.full((1,), np.nan, dtype=torch.float64, device="cuda")
        g = torch.full((1, 11), np.nan, dtype=torch.float64, device="cuda") if grad else None
        check(lib().pes_lnl_batch_noalloc(core._ctx, x.data_ptr(), 1, l.data_ptr(), g.data_ptr() if grad else None, 0,
                                          torch.cuda.current_stream().cuda_stream))
        if grad:
            assert torch.equal(l, ref[0]) and torch.equal(g, ref[1])
        else:
            assert torch.equal(l, ref)
