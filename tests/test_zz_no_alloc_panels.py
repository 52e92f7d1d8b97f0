"""pes_lnl_batch_noalloc on contexts with panels and on contexts evaluated at every bin: batches up
to the largest that is accepted (which may run in parts) give pes_lnl_batch's values to the last bit."""

import numpy as np
import pytest
import torch

from tests._setup import add_to_core, inj_row, make_detector, particle_cloud

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_nodes", [1024, 0])
@pytest.mark.parametrize("grad", [False, True])
def test_noalloc_largest_batch(n_nodes, grad):
    from pespace_amd._lib import check, lib
    from pespace_amd.core import LikelihoodCore
    t = 3.0e6 if n_nodes else 655360.0
    d, labels = make_detector(T=t, dt=5.0, fmax=0.05)
    core = LikelihoodCore(modes=["22"], n_nodes=n_nodes, f_node_min=1e-4, f_node_max=0.05)
    add_to_core(core, d, labels)
    core.n_bins  # builds the context
    limit = 64 << 20
    P = 1
    while lib().pes_lnl_batch_noalloc_bytes(core._ctx, P + 1, int(grad)) <= limit:
        P += 1
    rows = particle_cloud(P, seed=61, rel=1e-3, center=inj_row(coalescence_time=0.8 * t))
    print(n_nodes, grad, core.n_bins, P, flush=True)
    for p in (1, P):
        x = torch.as_tensor(rows[:p], device="cuda")
        l = torch.full((p,), np.nan, dtype=torch.float64, device="cuda")
        g = torch.full((p, 11), np.nan, dtype=torch.float64, device="cuda") if grad else None
        check(lib().pes_lnl_batch_noalloc(core._ctx, x.data_ptr(), p, l.data_ptr(), g.data_ptr() if grad else None, 0,
                                          torch.cuda.current_stream().cuda_stream))
        ref = core.lnl(rows[:p], grad=grad)
        if grad:
            assert torch.equal(l, ref[0]) and torch.equal(g, ref[1])
        else:
            assert torch.equal(l, ref)
