"""Argument checks of the entry points that read waveforms where the caller has them (no GPU)."""

import ctypes

from pespace_amd._lib import lib


def test_links_from_modes_needs_a_context():
    p = (ctypes.c_void_p * 1)(8)
    assert lib().pes_links_from_modes(None, 0, 1, p, p, p, 0.0, 0.0, 0.0, 0.0, 8, None) == 3


def test_td_links_strided_checks():
    orbit = (0, 2.5e9, 0.0, 0.0, 0.0, 0.0, 0.0)
    tail = (0.0, 1.0, 8, 0.1, 0.2, 0.3, 0.0, 1.0)
    f = lib().pes_td_links_strided
    assert f(*orbit, None, None, 0, *tail, 0, None, None) == 1  # stride
    assert f(*orbit, None, None, -2, *tail, 0, None, None) == 1
    assert f(*orbit, None, None, 2, *tail, 4, None, None) == 1  # NULL arrays
    assert f(*orbit, None, None, 2, *tail, 0, None, None) == 0  # nothing to do
