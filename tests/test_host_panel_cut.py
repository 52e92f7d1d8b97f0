"""Where tiles are cut into panels (csrc/panel_cut.hpp, compiled for the host under ASan and UBSan).

Every panel keeps both bounds, a relative half-width of 1.4e-3 and 4 pi L (f_hi - f_lo) <= 3e-3, on
even grids, on grids with a gap or a change of spacing inside a tile and on logarithmic ones, with fine
and coarse node grids.  On even grids the panels of a node interval are equal to one bin.  Cutting
into equal numbers of bins alone breaks the bounds on the uneven grids, so these can tell.
"""

import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = "/opt/rocm/llvm/bin/clang++" if os.path.exists("/opt/rocm/llvm/bin/clang++") else shutil.which("clang++")
YEAR = 31557600.0
EPS, SWING, PIECES = 1.4e-3, 3.0e-3, 8


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if CXX is None:
        pytest.skip("no clang++")
    exe = str(tmp_path_factory.mktemp("cut") / "host_panel_cut")
    subprocess.run([CXX, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-I", os.path.join(ROOT, "pespace_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host_kernel", "host_panel_cut.cpp"), "-o", exe], check=True)
    return exe


def _even(lo, hi, df):
    return df * np.arange(np.ceil(lo / df), np.floor(hi / df) + 1)


def _grid(name):
    df = 1.0 / YEAR
    if name == "even":
        return _even(1e-3, 3e-3, df)
    if name == "gap":       # 1.5e-4 Hz left out, no bin of it at a tile's edge
        f = _even(0.0298, 0.0302, df)
        return f[(f < 0.02995) | (f > 0.0301)]
    if name == "notches":   # a narrow line every few hundred bins
        f = _even(4e-3, 5e-3, df)
        return f[(np.arange(f.size) % 300) > 40]
    if name == "step":      # six times the spacing from the middle of a tile on
        f = _even(2e-3, 2.01e-3, df)
        return np.concatenate([f, f[-1] + 6 * df * np.arange(1, 4000)])
    if name == "log":
        return np.geomspace(1e-3, 2e-3, 60000)
    return np.array([1e-3])  # one bin


def _widths(f, L):
    """Of the frequencies f (increasing), the width in units of each bound."""
    return max((f[-1] - f[0]) / ((f[-1] + f[0]) * EPS), 4 * np.pi * L * (f[-1] - f[0]) / SWING)


def _index_cut(f, j, L):
    """Equal numbers of bins, as many panels as the whole width of a part asks for."""
    worst, total = 0.0, 0
    for v in np.unique(j):
        g = f[j == v]
        k = max(1, min(int(np.ceil(_widths(g, L))), g.size))
        e = [g.size * i // k for i in range(k + 1)]
        worst, total = max([worst] + [_widths(g[a:b], L) for a, b in zip(e, e[1:])]), total + k
    return worst, total


@pytest.mark.parametrize("n_nodes", [1024, 64, 5])
@pytest.mark.parametrize("arm", [2.5e9, 1.7e8])
@pytest.mark.parametrize("name", ["even", "gap", "notches", "step", "log", "one"])
def test_every_panel_keeps_the_bounds(driver, tmp_path, name, arm, n_nodes):
    f, L = _grid(name), arm / 299792458.0
    u0, du = np.log(1e-4), np.log(0.06 / 1e-4) / (n_nodes - 1)
    j = np.clip(np.floor((np.log(f) - u0) / du), 0, n_nodes - 2).astype(np.int32)
    path = str(tmp_path / "grid.bin")
    with open(path, "wb") as fh:
        np.array([f.size], np.int32).tofile(fh)
        f.tofile(fh)
        j.tofile(fh)
        np.array([L]).tofile(fh)
    out = subprocess.run([driver, path], check=True, capture_output=True, text=True).stdout.splitlines()
    assert len(out) == (f.size + 255) // 256
    broken, cut = 0, 0
    for t, line in enumerate(out):
        v = np.array(line.split(), dtype=int)
        ft, jt = f[256 * t:256 * t + 256], j[256 * t:256 * t + 256]
        worst, total = _index_cut(ft, jt, L)
        broken += total <= PIECES and worst > 1.0
        assert 0 <= v[0] <= PIECES and v.size == 1 + 3 * v[0]
        if v[0] == 0:  # only where no cut into so few panels keeps the bounds
            assert total > PIECES
            continue
        cut += 1
        first, bins, node = v[1:].reshape(-1, 3).T
        assert first[0] == 0 and np.all(first[1:] == (first + bins)[:-1]) and first[-1] + bins[-1] == ft.size
        for a, n, k in zip(first, bins, node):
            assert n >= 1 and np.all(jt[a:a + n] == k)
            assert _widths(ft[a:a + n], L) <= 1.0 + 1e-9  # (the same sums in another order)
        if name == "even":
            assert v[0] == total
            for k in np.unique(node):
                assert np.ptp(bins[node == k]) <= 1
    assert cut > 0
    if name in ("gap", "step") and n_nodes < 1024 and arm > 1e9:
        assert broken > 0
