"""The resident adjoint loop (every backward step in one launch) against the
loop of one launch per step, bit for bit: the same operations on the same
values, so there is no tolerance."""
import numpy as np
import pytest

from test_gpu_kept_fields import _case, _equal, _single

pytestmark = pytest.mark.gpu


def _both(case, monkeypatch):
    par, nt = case[0], case[0]["nt"]
    print("case", par, flush=True)
    monkeypatch.setenv("AWEFD_RESIDENT", "0")
    want = _single(case, 0, max(1, nt // 3))
    monkeypatch.setenv("AWEFD_RESIDENT", "1")
    got = _single(case, 0, nt)
    assert np.any(want[2]) or nt < 3
    _equal(got, want)


# a tile owns 64 - 2 nop z nodes and 8 rx rows: one tile, a tile and a node,
# several with remainders, the most rows compiled
@pytest.mark.parametrize("fdorder", [2, 4, 6, 8])
@pytest.mark.parametrize("nz,nx,nt,nb", [(30, 31, 20, 8), (45, 190, 21, 8), (97, 203, 17, 12), (300, 43, 12, 10)])
def test_tiles(nz, nx, nt, nb, fdorder, monkeypatch):
    _both(_case(nz, nx, nt, nb, fdorder=fdorder), monkeypatch)


@pytest.mark.parametrize("nz,nx,fdorder", [(900, 900, 4), (800, 1900, 4), (900, 1500, 8), (500, 1200, 6)])
def test_many_rows_per_wave(nz, nx, fdorder, monkeypatch):
    _both(_case(nz, nx, 12, 10, nsrc=6000, nrec=6000, fdorder=fdorder), monkeypatch)


@pytest.mark.parametrize("kw", [dict(dabc=False), dict(free=True), dict(expl=True), dict(optfd=True)])
def test_options(kw, monkeypatch):
    _both(_case(83, 130, 20, 9, **kw), monkeypatch)


def test_more_points_than_lanes(monkeypatch):
    """Waves with more receiver and source nodes than lanes, several points
    on one node."""
    _both(_case(40, 50, 14, 6, nsrc=900, nrec=2500), monkeypatch)


def test_a_block_that_gives_up(monkeypatch):
    case = _case(83, 130, 20, 9)
    want = _single(case, 0, 20)
    monkeypatch.setenv("AWEFD_RES_WAIT", "0")
    _equal(_single(case, 0, 20), want)
