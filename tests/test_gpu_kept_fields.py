"""Gradients whose forward run keeps every field against those that recompute
them from checkpoints, single shots and batches: traces, last field and
gradient bit for bit (the same steps), so there is no tolerance."""
import numpy as np
import pytest

from wavefield_imaging_amd import _lib as L
from wavefield_imaging_amd import awefd, synth

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _model(par, vel, s, rec, wav):
    m = awefd.Model("cart2d", par)
    m.set_model(vel)
    m.set_sources(s)
    m.set_receivers(rec)
    m.set_wavelet(wav)
    return m


def _case(nz, nx, nt, nb, nsrc=2, nrec=70, **kw):
    rng = np.random.default_rng(nz + nx + nt)
    par = dict(n=[nz, nx], o=[0.0, 0.0], d=[5.0, 5.0], nt=nt, dt=synth.DT, nb=nb, dabc=True, fdorder=4, expl=False)
    par.update(kw)
    vel = rng.uniform(1.2e8, 3.0e8, (nx, nz)).astype(np.float32)
    pts = [rng.uniform(-nb * 5.0, [5.0 * (nx + nb - 2), 5.0 * (nz + nb - 2)], (n, 2)).astype(np.float32)
           for n in (nsrc, nsrc, nsrc, nrec)]
    wav = rng.standard_normal((nt, 1 if par["expl"] else nsrc)).astype(np.float32)
    res = rng.standard_normal((3, nt, nrec)).astype(np.float32)
    return par, vel, pts[:3], pts[3], wav, torch.from_numpy(res).cuda()


def _single(case, k, ckpt):
    par, vel, sous, rec, wav, res = case
    with _model(par, vel, sous[k], rec, wav) as m:
        tr = torch.empty((m.nt, m.nr), device="cuda")
        g = torch.empty((par["n"][1], par["n"][0]), device="cuda")
        torch.cuda.synchronize()
        L.check(m.lib.awefd_run_ckpt(m.h, tr.data_ptr(), ckpt))
        f = m.field()
        out = []
        for _ in range(2):               # a second gradient of the same run
            L.check(m.lib.awefd_adjoint_grad(m.h, res[k].contiguous().data_ptr(), g.data_ptr()))
            out.append(g.cpu().numpy().copy())
        np.testing.assert_array_equal(out[0], out[1])
        return tr.cpu().numpy(), f, out[0]


def _batch(case, ckpt, runs=2):
    par, vel, sous, rec, wav, res = case
    ms = [_model(par, vel, s, rec, wav) for s in sous]
    b = awefd.Batch(ms)
    g = torch.empty((par["n"][1], par["n"][0]), device="cuda")
    for _ in range(runs):                # the second replays both graphs
        b.run_ckpt(ckpt)
        tr, f = [m.traces() for m in ms], [m.field() for m in ms]
        b.adjoint_grad([res[s].data_ptr() for s in range(3)], g.data_ptr())
    b.close()
    for m in ms:
        m.close()
    return tr, f, g.cpu().numpy()


def _equal(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


# runs of one step to a few passes of three; a grid inside one tile, several
# tiles with remainders; loops the resident kernel does not take (fdorder 12,
# AWEFD_RESIDENT=0)
@pytest.mark.parametrize("resident", ["1", "0"])
@pytest.mark.parametrize("nz,nx,nt,nb,kw", [
    (30, 31, 40, 6, dict()), (30, 31, 41, 6, dict(expl=True)), (97, 140, 30, 8, dict(fdorder=8)),
    (120, 75, 23, 10, dict(fdorder=2, free=True)), (61, 90, 18, 7, dict(dabc=False)), (61, 90, 19, 12, dict(fdorder=12)),
    (40, 50, 5, 6, dict()), (40, 50, 2, 6, dict()), (40, 50, 1, 6, dict()), (61, 90, 25, 7, dict(sse=False))])
def test_kept_against_recomputed(nz, nx, nt, nb, kw, resident, monkeypatch):
    monkeypatch.setenv("AWEFD_RESIDENT", resident)
    case = _case(nz, nx, nt, nb, **kw)
    few = max(1, nt // 3)
    want = _single(case, 0, few) if nt > 1 else None
    for ckpt in (0, nt, nt + 5):
        got = _single(case, 0, ckpt)
        if want is None:
            want = got
        _equal(got, want)
    if nt > 1:
        tr, f, g = _batch(case, few)
        for ckpt in (0, nt):
            t2, f2, g2 = _batch(case, ckpt)
            _equal(t2, tr)
            _equal(f2, f)
            np.testing.assert_array_equal(g2, g)
        np.testing.assert_array_equal(tr[0], want[0])
        np.testing.assert_array_equal(f[0], want[1])


def test_interval_changes_between_runs():
    """One handle, one batch: kept, recomputed, kept again."""
    case = _case(61, 90, 24, 7)
    par, vel, sous, rec, wav, res = case
    want = _batch(case, 5)
    ms = [_model(par, vel, s, rec, wav) for s in sous]
    b = awefd.Batch(ms)
    g = torch.empty((par["n"][1], par["n"][0]), device="cuda")
    for ckpt in (0, 5, 24, 7, 0):
        b.run_ckpt(ckpt)
        _equal([m.traces() for m in ms], want[0])
        b.adjoint_grad([res[s].data_ptr() for s in range(3)], g.data_ptr())
        np.testing.assert_array_equal(g.cpu().numpy(), want[2])
    b.close()
