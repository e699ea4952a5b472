"""The 2-D loop as one graph (loops that are not resident: fdorder 10 and 12,
the resident loop switched off) against the CPU oracle, bit for bit: capture,
replays, a setter, another trace buffer and the profiled run."""
import numpy as np
import pytest

import test_gpu_cart as cart
from wavefield_imaging_amd import awefd

pytestmark = pytest.mark.gpu


def test_replays_setters_and_eager_path(orc, monkeypatch, capfd):
    monkeypatch.setenv("AWEFD_RESIDENT", "0")
    monkeypatch.setenv("AWEFD_VERBOSE", "1")
    cart.test_cart2d_graph_replays_setters_and_eager_path(orc)
    assert "resident" not in capfd.readouterr().err


@pytest.mark.parametrize("fdorder", [10, 12])
def test_replays_of_high_orders(orc, fdorder):
    par, vel, sou, rec, wav = cart._case2d(nt=61, fdorder=fdorder)
    ref, ufin, _ = orc.run("cart2d", par, vel, sou, rec, wav)
    ref2, ufin2, _ = orc.run("cart2d", par, vel * np.float32(1.125), sou, rec, wav)
    with awefd.Model("cart2d", par) as m:
        m.set_model(vel)
        m.set_sources(sou)
        m.set_receivers(rec)
        m.set_wavelet(wav)
        for rep in range(4):                         # direct, capture, replays
            np.testing.assert_array_equal(m.run()[0], ref, err_msg="run %d" % rep)
            np.testing.assert_array_equal(m.field(), ufin)
        m.set_model(vel * np.float32(1.125))
        for rep in range(3):
            np.testing.assert_array_equal(m.run()[0], ref2, err_msg="run %d" % rep)
            np.testing.assert_array_equal(m.field(), ufin2)
