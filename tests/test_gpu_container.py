"""Links of supplied waveforms: read where the caller has them, or gathered into one array first.

The two ways are the same kernel on the same numbers, so their links are the same to the last bit,
whatever the arrays' types, strides and count; both against the oracle-checked kernel's own waveform
container (pes_links) to its tolerance; far or non-finite t_f takes the general formulas and is
compared with them through a mode whose amplitude is zero there.  Time domain: columns of one array
against separate arrays, bit for bit.
"""

import numpy as np
import pytest
import torch

from tests._setup import add_to_core, inj_row, make_detector

pytestmark = pytest.mark.gpu
SKY = (1.375, -1.2108, 2.659)
TIANQIN = dict(orbit="Tianqin_analytic", psd_model="Tianqin_GWSpace", fmin=1e-3, fmax=0.0391)
ON_OFF = (3.0e5, 1.5e5, 1.0e5, 1.0e4)


def _core(n_modes, **kw):
    from pespace_amd.core import LikelihoodCore
    names = ("22", "21", "33", "32", "44", "43")[:n_modes]
    core = LikelihoodCore(modes=names, n_nodes=1024, f_node_min=1e-4, f_node_max=0.05)
    d, labels = make_detector(T=655360.0, dt=5.0, inject=False, **kw)
    add_to_core(core, d, labels)
    return core


@pytest.mark.parametrize("kw", [dict(fmax=0.0391), TIANQIN, dict(TIANQIN, duty=ON_OFF), dict(fmax=0.02, duty=ON_OFF)])
@pytest.mark.parametrize("n_modes", [1, 2, 6])
def test_container_links(kw, n_modes):
    core = _core(n_modes, **kw)
    row = inj_row()
    wf = core.waveform(0, row[None])[0]  # [mode][bin][h+ re, im, hx re, im, tf]
    modes = {str(m): {"plus": torch.view_as_complex(wf[m, :, 0:2].contiguous()),
                      "cross": torch.view_as_complex(wf[m, :, 2:4].contiguous()), "tf": wf[m, :, 4].contiguous()}
             for m in range(n_modes)}
    where = (*row[7:10], row[10])
    direct = core.links_from_container(0, modes, *where)
    host = {k: {a: v.cpu().numpy() for a, v in m.items()} for k, m in modes.items()}
    assert torch.equal(torch.view_as_real(core.links_from_container(0, host, *where)), torch.view_as_real(direct))
    strided = {k: dict(m, plus=torch.stack([m["plus"], m["plus"]], 1)[:, 0]) for k, m in modes.items()}
    assert torch.equal(torch.view_as_real(core.links_from_container(0, strided, *where)), torch.view_as_real(direct))
    # the library's own links of the same waveform: its interpolated phase is the container's, and
    # 1e4 rad of it rounded on the way through h+ and hx cost 1e4 * 1.1e-16 * a few
    own = core.links(0, row[None])[0]
    err = (direct - own).abs().max(1).values / own.abs().max(1).values
    assert float(err.max()) < 2e-11


def test_container_many_modes_and_far_times():
    core = _core(1, **TIANQIN)
    row = inj_row()
    wf = core.waveform(0, row[None])[0, 0]
    m = {"plus": torch.view_as_complex(wf[:, 0:2].contiguous()),
         "cross": torch.view_as_complex(wf[:, 2:4].contiguous()), "tf": wf[:, 4].contiguous()}
    where = (*row[7:10], row[10])
    one = core.links_from_container(0, m, *where)
    nine = core.links_from_container(0, {str(i): m for i in range(9)}, *where)  # beyond the pointers' count
    # nine sums and the common factor, each rounding within 1.1e-16 of the complex value
    assert bool(((nine - 9.0 * one).abs() <= 1e-14 * (9.0 * one).abs()).all())
    # silent bins with any t_f, however far, add exactly nothing
    far = {k: v.clone() for k, v in m.items()}
    far["plus"][::2] = far["cross"][::2] = 0.0
    near = {k: v.clone() for k, v in far.items()}
    far["tf"][::4], far["tf"][2::4] = 1e300, -1e19
    a, b = core.links_from_container(0, far, *where), core.links_from_container(0, near, *where)
    assert torch.equal(torch.view_as_real(a), torch.view_as_real(b)) and torch.isfinite(torch.view_as_real(a)).all()
    # a NaN t_f gives NaN links at its bin and nowhere else
    bad = {k: v.clone() for k, v in m.items()}
    bad["tf"][5] = float("nan")
    c = torch.isnan(torch.view_as_real(core.links_from_container(0, bad, *where))).any(2)
    assert bool(c[:, 5].all()) and int(c.sum()) == 6


@pytest.mark.parametrize("n", [2, 255, 256, 257, 5000])
@pytest.mark.parametrize("wave_dt", [5.0, 1.0, 0.25])
def test_td_links_columns(n, wave_dt):
    from pespace_amd.core import td_links
    g = torch.Generator(device="cuda").manual_seed(n)
    data = torch.randn(max(n, 300), 2, dtype=torch.float64, device="cuda", generator=g)
    args = (0, 2.5e9, 0.1, 0.4)
    tail = (100.0, wave_dt, *SKY, 90.0, 5.0, n)
    a = td_links(*args, data[:, 0], data[:, 1], *tail)
    b = td_links(*args, data[:, 0].contiguous(), data[:, 1].contiguous(), *tail)
    c = td_links(*args, torch.stack([data[:, 0]] * 3, 1)[:, 0], data[:, 1], *tail)
    assert torch.equal(a, b) and torch.equal(a, c)
