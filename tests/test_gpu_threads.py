"""Handles of several threads at once on one GPU: resident loops (cartesian,
polar, a gradient) beside each other, beside a loop and batches that capture
graphs, and beside set-ups; each gives what it gives alone, bit for bit."""
import os
import subprocess
import sys
import threading
import traceback

import numpy as np
import pytest

import test_gpu_cart as small
import test_gpu_kept_fields as kept
import test_gpu_resident as cart
import test_gpu_resident_polar as polar
from wavefield_imaging_amd import _lib as L
from wavefield_imaging_amd import awefd

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _model(kind, par, vel, sou, rec, wav):
    m = awefd.Model(kind, par)
    m.set_model(vel)
    m.set_sources(sou)
    m.set_receivers(rec)
    m.set_wavelet(wav)
    return m


def _forward(kind, case):
    m = _model(kind, *case)
    return lambda: np.concatenate([m.run()[0].ravel(), m.field().ravel()])


def _gradient(case):
    par, vel, sous, rec, wav, res = case
    m = kept._model(par, vel, sous[0], rec, wav)
    g = torch.empty((par["n"][1], par["n"][0]), device="cuda")
    r = res[0].contiguous()

    def run():
        L.check(m.lib.awefd_run_ckpt(m.h, None, par["nt"]))
        L.check(m.lib.awefd_adjoint_grad(m.h, r.data_ptr(), g.data_ptr()))
        return np.concatenate([m.traces().ravel(), g.cpu().numpy().ravel()])

    return run


def _batch(case):
    ms = [_model("cart2d", *case), _model("cart2d", *case)]
    b = awefd.Batch(ms)

    def run():
        b.run()
        return np.stack([m.traces() for m in ms])

    return run


def test_handles_of_several_threads(monkeypatch, capfd):
    monkeypatch.setenv("AWEFD_VERBOSE", "1")
    c1, c2 = cart._case(83, 130, 9, 150, 1)[:5], cart._case(400, 700, 20, 60, 2, nsrc=9)[:5]
    graph = cart._case(83, 130, 12, 90, 3, fdorder=12)[:5]      # not resident: captured by its second run
    work = [lambda: _forward("cart2d", c1), lambda: _forward("cart2d", c1), lambda: _forward("cart2d", c2),
            lambda: _forward("spher2d", polar._case(150, 210, 9, 150)), lambda: _gradient(g1), lambda: _gradient(g1),
            lambda: _batch(c1), lambda: _forward("cart2d", graph), lambda: _forward("cart3d", small._case3d()),]
    g1 = kept._case(97, 203, 80, 12)
    torch.cuda.synchronize()
    want = [w()() for w in work]
    np.testing.assert_array_equal(want[1], want[0])
    np.testing.assert_array_equal(want[5], want[4])
    bad = []

    def loop(i):
        try:
            for k in range(16):
                if k % 4 == 0:                       # a fresh handle: its set-up beside the others' runs
                    run = work[i]()
                if not np.array_equal(run(), want[i]):
                    bad.append((i, k))
        except Exception:
            bad.append((i, traceback.format_exc()))

    threads = [threading.Thread(target=loop, args=(i,)) for i in range(len(work))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
    err = capfd.readouterr().err
    assert "resident 2-D loop" in err and "resident adjoint" in err and "off" not in err


CHILD = """
import sys
sys.path[:0] = [%r, %r]
import numpy as np
import test_gpu_kept_fields as kept
import test_gpu_resident as cart
import test_gpu_resident_polar as polar
import test_gpu_threads as t
for k, run in enumerate((t._forward("cart2d", cart._case(83, 130, 9, 150, 1)[:5]),
                         t._forward("spher2d", polar._case(150, 210, 9, 150)), t._gradient(kept._case(97, 203, 80, 12)))):
    for _ in range(3):
        out = run()
    np.save(sys.argv[1] + "/%%d.npy" %% k, out)
    print("case", k, flush=True)
"""


def test_a_second_process(tmp_path):
    """One process at a time has a card's cooperative queue: beside one that
    runs resident loops, another runs the loops of one launch per step, and
    gives the same."""
    here = os.path.dirname(os.path.abspath(__file__))
    runs = [_forward("cart2d", cart._case(83, 130, 9, 150, 1)[:5]), _forward("spher2d", polar._case(150, 210, 9, 150)),
            _gradient(kept._case(97, 203, 80, 12))]
    want = [r() for r in runs]
    child = subprocess.Popen([sys.executable, "-c", CHILD % (os.path.dirname(here), here), str(tmp_path)])
    while child.poll() is None:                          # this process's runs go on beside it
        for r, w in zip(runs, want):
            np.testing.assert_array_equal(r(), w)
    assert child.returncode == 0
    for k, w in enumerate(want):
        np.testing.assert_array_equal(np.load(tmp_path / ("%d.npy" % k)), w)
