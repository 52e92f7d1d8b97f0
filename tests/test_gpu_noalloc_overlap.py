"""pes_lnl_batch and pes_lnl_batch_noalloc of one context with panels on two streams at once.

The two entry points share no scratch (the second's lies in the GPU's fixed array, its list of
bin-by-bin work in arrays of its own), so batches that overlap give the values they give alone, to the
last bit.  The two batches differ in what they leave to the bin-by-bin kernel: near and light systems.
"""

import numpy as np
import pytest
import torch

from tests._setup import add_to_core, inj_row, make_detector, particle_cloud, prior_rows

pytestmark = pytest.mark.gpu

T = 4.0e6


@pytest.mark.parametrize("grad", [False, True])
def test_two_entry_points_overlap(grad):
    from pespace_amd._lib import check, lib
    from pespace_amd.core import LikelihoodCore
    core = LikelihoodCore(modes=["22", "33"], n_nodes=1024, f_node_min=1e-4, f_node_max=0.05)
    add_to_core(core, *make_detector(T=T, modes=((2, 2), (3, 3)), interp=(1e-4, 0.05, 1024)))
    light = particle_cloud(40, seed=71, rel=1e-4, center=inj_row(chirp_mass=3.0e3, coalescence_time=0.7 * T))
    a = np.vstack([particle_cloud(200, seed=72, rel=1e-3, center=inj_row(coalescence_time=0.7 * T)),
                   prior_rows(100, seed=73, tc_range=(0.0, T))])
    xa, xb = (torch.as_tensor(r, device="cuda").contiguous() for r in (a, light))

    def buffers(n):
        return (torch.full((n,), np.nan, dtype=torch.float64, device="cuda"),
                torch.full((n, 11), np.nan, dtype=torch.float64, device="cuda"))

    def noalloc(out):
        check(lib().pes_lnl_batch_noalloc(core._ctx, xb.data_ptr(), xb.shape[0], out[0].data_ptr(),
                                          out[1].data_ptr() if grad else None, 0,
                                          torch.cuda.current_stream().cuda_stream))

    def batch(out):
        core.lnl(xa, grad=grad, out=out[0], grad_out=out[1] if grad else None)

    ref_a, ref_b = buffers(len(a)), buffers(len(light))
    batch(ref_a)
    torch.cuda.synchronize()
    noalloc(ref_b)
    torch.cuda.synchronize()
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    out_a, out_b = [buffers(len(a)) for _ in range(6)], [buffers(len(light)) for _ in range(18)]
    torch.cuda.synchronize()
    for i in range(6):
        with torch.cuda.stream(sa):
            batch(out_a[i])
        with torch.cuda.stream(sb):
            for k in range(3):
                noalloc(out_b[3 * i + k])
    torch.cuda.synchronize()
    for ref, outs in ((ref_a, out_a), (ref_b, out_b)):
        for o in outs:
            assert torch.equal(o[0], ref[0])
            assert not grad or torch.equal(o[1], ref[1])
