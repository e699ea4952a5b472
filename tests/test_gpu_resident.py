"""The resident 2-D loop (every step in one launch, rims exchanged between
blocks) against the loop of one launch per step, bit for bit: the same
operations on the same values, so there is no tolerance."""
import numpy as np
import pytest

from wavefield_imaging_amd import awefd, synth

pytestmark = pytest.mark.gpu


def _case(n1, n2, nb, nt, seed, nsrc=3, dense=False, **kw):
    """Random velocity, sources anywhere on the padded grid (several on one
    node), receivers off the nodes or on every node."""
    rng = np.random.default_rng(seed)
    vel = rng.uniform(1.2e8, 3.0e8, (n2, n1)).astype(np.float32)
    lo = np.array([-nb, -nb], float)
    hi = np.array([n2 + nb - 1.01, n1 + nb - 1.01])
    sou = rng.uniform(lo, hi, (nsrc, 2))
    if nsrc > 1:
        sou[1] = sou[0]
    if dense:
        x, z = np.meshgrid(np.arange(-nb, n2 + nb - 1), np.arange(-nb, n1 + nb - 1), indexing="ij")
        rec = np.stack([x.ravel(), z.ravel()], 1) + 0.25
    else:
        rec = rng.uniform(lo, hi, (97, 2))
    par = dict(n=[n1, n2], o=[0.0, 0.0], d=[5.0, 5.0], nt=nt, dt=synth.DT, nb=nb, dabc=True, cden=True,
               fdorder=4, expl=False)
    par.update(kw)
    wav = rng.standard_normal((nt, 1 if par["expl"] else nsrc)).astype(np.float32)
    den = None if par["cden"] else rng.uniform(900.0, 2700.0, (n2, n1)).astype(np.float32)
    return par, vel, (sou * 5).astype(np.float32), (rec * 5).astype(np.float32), wav, den


def _both(case, monkeypatch, capfd, steps=None, taken=True):
    par, vel, sou, rec, wav, den = case
    print("case", par, len(sou), len(rec), steps, flush=True)
    monkeypatch.setenv("AWEFD_VERBOSE", "1")
    monkeypatch.setenv("AWEFD_RESIDENT", "0")
    tr0, _, f0 = awefd.run("cart2d", par, vel, sou, rec, wav, den=den)
    assert "resident" not in capfd.readouterr().err
    monkeypatch.setenv("AWEFD_RESIDENT", "1")
    if steps:
        monkeypatch.setenv("AWEFD_RES_STEPS", str(steps))
    tr1, _, f1 = awefd.run("cart2d", par, vel, sou, rec, wav, den=den)
    err = capfd.readouterr().err
    assert ("resident" in err) == taken, err
    if steps and taken:
        assert "%d steps per exchange" % steps in err
    assert par["nt"] == 1 or np.any(f0)   # the first row and field are those before any source
    np.testing.assert_array_equal(tr1, tr0)
    np.testing.assert_array_equal(f1, f0)


# one step owns 64 - 2 nop z nodes a tile, two 64 - 4 nop: grids of one tile,
# a tile and one node, several with a remainder, a narrow one
@pytest.mark.parametrize("steps", [1, 2])
@pytest.mark.parametrize("fdorder", [2, 4, 6, 8])
@pytest.mark.parametrize("n1,n2,nb,nt", [(40, 41, 10, 60), (45, 150, 8, 61), (97, 203, 12, 47), (300, 33, 8, 30)])
def test_tiles(n1, n2, nb, nt, fdorder, steps, monkeypatch, capfd):
    _both(_case(n1, n2, nb, nt, n1 + fdorder, fdorder=fdorder), monkeypatch, capfd, steps)


@pytest.mark.parametrize("steps", [1, 2])
@pytest.mark.parametrize("kw", [dict(dabc=False), dict(free=True), dict(optfd=True), dict(expl=True)])
def test_options(kw, steps, monkeypatch, capfd):
    _both(_case(83, 130, 9, 50, 5, **kw), monkeypatch, capfd, steps)


@pytest.mark.parametrize("fdorder", [2, 4, 6, 8])
def test_variable_density(fdorder, monkeypatch, capfd):
    _both(_case(83, 210, 9, 50, 7, cden=False, fdorder=fdorder), monkeypatch, capfd)


@pytest.mark.parametrize("steps", [1, 2])
def test_a_receiver_on_every_node(steps, monkeypatch, capfd):
    """Receivers across every seam and corner of the tiles, many per thread."""
    _both(_case(118, 131, 5, 21, 9, dense=True), monkeypatch, capfd, steps)


@pytest.mark.parametrize("steps", [1, 2])
def test_more_sources_than_lanes(steps, monkeypatch, capfd):
    case = _case(60, 40, 6, 25, 11, nsrc=400)
    _both(case, monkeypatch, capfd, steps)


@pytest.mark.parametrize("nt", [1, 2, 3])
@pytest.mark.parametrize("steps", [1, 2])
def test_few_steps(nt, steps, monkeypatch, capfd):
    _both(_case(70, 90, 6, nt, 13, nsrc=40), monkeypatch, capfd, steps)


@pytest.mark.parametrize("rx_rows", [1900, 2600])
def test_many_rows_per_wave(rx_rows, monkeypatch, capfd):
    """Tiles of 16 and more rows per wave, and the widest grid they hold."""
    _both(_case(1000, rx_rows, 10, 12, 17, nsrc=5), monkeypatch, capfd)


def test_grid_beyond_the_chip(monkeypatch, capfd):
    _both(_case(1500, 4500, 4, 3, 19, dense=False, nsrc=300), monkeypatch, capfd, taken=False)


def test_repeated_runs_and_setters(monkeypatch):
    """Runs of one handle one after the other (tags grow), with another
    source in between, equal fresh handles."""
    par, vel, sou, rec, wav, _ = _case(83, 130, 9, 40, 21)
    fresh = [awefd.run("cart2d", par, vel, s, rec, wav)[0] for s in (sou, sou[::-1].copy())]
    with awefd.Model("cart2d", par) as m:
        m.set_model(vel)
        m.set_receivers(rec)
        m.set_wavelet(wav)
        for k in (0, 0, 1, 0, 1, 1):
            m.set_sources(sou if k == 0 else sou[::-1].copy())
            np.testing.assert_array_equal(m.run()[0], fresh[k])


def test_a_block_that_gives_up(monkeypatch):
    """A wait cut short (no poll may fail): the run falls back to the loop of
    one launch per step and still gives its result."""
    par, vel, sou, rec, wav, _ = _case(83, 130, 9, 40, 23)
    want = awefd.run("cart2d", par, vel, sou, rec, wav)
    monkeypatch.setenv("AWEFD_RES_WAIT", "0")
    got = awefd.run("cart2d", par, vel, sou, rec, wav)
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[2], want[2])


# 18, 26 and 30 rows per wave at fdorder 4, and 30 at fdorder 8
@pytest.mark.parametrize("n1,n2,fdorder", [(1000, 2100, 4), (1000, 3050, 4), (1000, 3500, 4), (1001, 2777, 8)])
def test_even_row_counts(n1, n2, fdorder, monkeypatch, capfd):
    _both(_case(n1, n2, 10, 8, 29, nsrc=40, fdorder=fdorder), monkeypatch, capfd)
