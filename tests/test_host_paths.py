"""The host code's own paths, on the CPU: the C sources against a HIP runtime
without a GPU (hip_stub.c), which can refuse an allocation, return a launch
error or let a resident loop give up."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from wavefield_imaging_amd import _lib as L
from wavefield_imaging_amd import awefd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "wavefield_imaging_amd", "csrc")
HOST = ("awefd_api.c", "awefd_setup.c", "spher_host.c", "awefd_batch.c", "awefd_adjoint.c", "awefd_resident.c")


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libhost.so")
    subprocess.run(["gcc", "-O1", "-g", "-shared", "-fPIC", "-std=gnu99", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-Wl,-Bsymbolic", "-I", SRC, "-I", os.path.join(ROOT, "include"), "-I", "/opt/rocm/include",
                    "-o", so] + [os.path.join(SRC, f) for f in HOST] + [os.path.join(ROOT, "tests", "hip_stub.c")]
                   + ["-lm", "-lpthread"], check=True)
    return so


class Stub:
    def __init__(self, lib):
        self.lib = lib

    def reset(self, fail_at=0, fail_above=0):
        self.lib.stub_reset(C.c_long(fail_at), C.c_size_t(fail_above))

    def get(self, name):
        return C.c_long.in_dll(self.lib, "stub_" + name).value

    def set(self, name, v):
        (C.c_long if name == "fail_at" else C.c_int).in_dll(self.lib, "stub_" + name).value = v


@pytest.fixture
def stub(built, monkeypatch):
    """The binding on the stubbed library for the time of one test."""
    monkeypatch.setattr(L, "_lib", None)
    monkeypatch.setattr(L, "LIB_PATH", built)
    for k in ("AWEFD_RESIDENT", "AWEFD_RES_STEPS", "AWEFD_RES_WAIT", "AWEFD_NARROW"):
        monkeypatch.delenv(k, raising=False)
    s = Stub(L.load())
    s.reset()
    yield s
    s.reset()


def _model(nt=9, n=(30, 40), nb=4, kind="cart2d", nr=5, **kw):
    par = dict(n=list(n), o=[0.0, 0.0] if kind == "cart2d" else [3387.5e3, 0.785], d=[5.0, 5.0], nt=nt, dt=6.67e-9,
               nb=nb, expl=True)
    if kind == "spher2d":
        par["d"] = [5.0, 5.0 / 3388.5e3]
    par.update(kw)
    m = awefd.Model(kind, par)
    m.set_model(np.full(n[::-1], 1.7e8, np.float32))
    x = np.array([par["o"][i] + 3.0 * par["d"][i] for i in ((1, 0) if kind == "cart2d" else (0, 1))], np.float32)
    m.set_sources(x[None])
    m.set_receivers(np.repeat(x[None], nr, 0))
    m.set_wavelet(np.ones(nt, np.float32))
    return m


def _dev(*shape):
    """An array of the stub's device memory, which is host memory."""
    a = np.zeros(shape, np.float32)
    return a, a.ctypes.data


def _grad(m, ckpt, tr=None):
    """A checkpointed run and its gradient."""
    res, rp = _dev(m.nt, m.nr)
    g, gp = _dev(m.params.n[1], m.params.n[0])
    L.check(m.lib.awefd_run_ckpt(m.h, tr, ckpt))
    L.check(m.lib.awefd_adjoint_grad(m.h, rp, gp))


def test_refused_fields_of_every_step_leave_no_error(stub):
    """A gradient whose nt fields are refused takes ceil(sqrt(nt)) checkpoints
    instead; the refused allocation's error must not be reported by the
    launches that follow."""
    with _model(nt=100) as m:
        stub.reset(fail_above=60 * 4 * 64 * 48)      # 100 fields of 64 x 48 are, 20 and 10 are not
        _grad(m, 0)
    stub.reset()
    with _model(nt=100) as m:                        # nor after an error that a caller has seen
        stub.reset(fail_at=1)
        with pytest.raises(L.AwefdError, match="out of memory"):
            m.run()                                  # the trace buffer
        stub.set("fail_at", 0)
        m.run()


ALL = 60 * 4 * 64 * 48       # more than 60 padded fields of the default grid at once


def test_an_interval_of_every_step_without_memory_for_it(stub):
    """ckpt >= nt where the fields do not fit: the run keeps its one pair, as
    with any interval, the gradient asks for its segment, and gives it by
    recomputing once there is memory."""
    with _model(nt=100) as m:
        for ckpt in (100, 300):
            stub.reset(fail_above=ALL)
            L.check(m.lib.awefd_run_ckpt(m.h, None, ckpt))
            assert stub.get("steps") == 100
            res, rp = _dev(m.nt, m.nr)
            g, gp = _dev(40, 30)
            assert m.lib.awefd_adjoint_grad(m.h, rp, gp) == -3
            assert b"gradient buffers" in m.lib.awefd_last_error()
            stub.reset()
            L.check(m.lib.awefd_adjoint_grad(m.h, rp, gp))
            assert stub.get("steps") == 99           # the segment's recomputed fields
            assert stub.get("adjoint") == 0
            m.lib.awefd_adjoint_release(m.h)
        L.check(m.lib.awefd_run_ckpt(m.h, None, 100))
        stub.reset()
        L.check(m.lib.awefd_adjoint_grad(m.h, rp, gp))
        assert stub.get("steps") == 0 and stub.get("adjoint") == 1


def test_a_batch_that_keeps_every_step_of_some_shots_only(stub):
    ms = [_model(nt=30) for _ in range(2)]
    b = awefd.Batch(ms)
    res, rp = _dev(30, 5)
    g, gp = _dev(40, 30)
    stub.reset(fail_at=4)                            # the second shot's fields
    b.run_ckpt(30)
    assert stub.get("rows") == 0 and stub.get("recomputed") == 0
    stub.reset()
    b.adjoint_grad([rp, rp], gp)
    assert stub.get("recomputed") == 2 * 29 or stub.get("recomputed") == 29     # one launch advances both shots
    L.check(ms[0].lib.awefd_adjoint_grad(ms[0].h, rp, gp))
    assert stub.get("adjoint") == 0                  # its fields were not kept either
    stub.reset()
    b.run_ckpt(30)
    assert stub.get("rows") == 2 * 30
    stub.reset()
    b.adjoint_grad([rp, rp], gp)
    assert stub.get("recomputed") == 0
    # a default interval drops to checkpoints for every shot
    for m in ms:
        m.lib.awefd_adjoint_release(m.h)
    stub.reset(fail_at=4)
    b.run_ckpt(0)
    stub.reset()
    b.adjoint_grad([rp, rp], gp)
    assert 0 < stub.get("recomputed") < 30
    b.run_ckpt(30)
    # a shot that was run on its own without its fields does not serve a batch that kept them
    ms[1].lib.awefd_adjoint_release(ms[1].h)
    stub.reset(fail_at=2)
    L.check(ms[1].lib.awefd_run_ckpt(ms[1].h, None, 30))
    stub.reset()
    with pytest.raises(L.AwefdError, match="awefd_batch_run_ckpt"):
        b.adjoint_grad([rp, rp], gp)
    b.close()
    for m in ms:
        m.close()


def test_traces_of_more_steps_than_a_grid_has_rows(stub, monkeypatch):
    """The trace rows of a run that kept its fields are rows of a launch's
    grid, of which there are at most 65,535."""
    monkeypatch.setenv("AWEFD_RESIDENT", "0")
    nt = 140000
    with _model(nt=nt, n=(5, 5), nb=1, fdorder=2, nr=1) as m:
        tr, tp = _dev(nt, 1)
        L.check(m.lib.awefd_run_ckpt(m.h, tp, nt))
        assert stub.get("rows") == nt
        assert stub.get("max_rows") <= 65535
        np.testing.assert_array_equal(tr[:, 0], np.arange(nt, dtype=np.float32))     # row n of field n


def _passes(kind, stub, fail_at):
    """Set-up, two runs and (cart2d) a gradient with allocation `fail_at`
    refused; whether every call went through, and the allocations asked for."""
    stub.reset(fail_at=fail_at)
    try:
        with _model(kind=kind) as m:
            m.run()
            m.run()
            if kind == "cart2d":
                _grad(m, 9)
                _grad(m, 9)
    except L.AwefdError as e:
        assert "out of memory" in str(e)
        return False, stub.get("allocs")
    return True, stub.get("allocs")


@pytest.mark.parametrize("kind", ["cart2d", "spher2d"])
def test_the_resident_loops_memory_is_optional(kind, stub, monkeypatch):
    """Calls fail for the allocations that the loop of one launch per step
    needs too, and for no others."""
    failed, asked = {}, {}
    for on in ("0", "1"):
        monkeypatch.setenv("AWEFD_RESIDENT", on)
        ok, asked[on] = _passes(kind, stub, 0)
        assert ok and (stub.get("resident") > 0) == (on == "1")
        failed[on] = sum(not _passes(kind, stub, n)[0] for n in range(1, asked[on] + 1))
    assert asked["1"] > asked["0"]
    assert failed["1"] == failed["0"] > 0
    if kind == "spher2d":
        assert failed["0"] == asked["0"] - 1         # the receivers near the sources: separate launches then


@pytest.mark.parametrize("kind", ["cart2d", "spher2d"])
def test_a_model_without_the_resident_loops_memory(kind, stub):
    """Whichever allocation was refused: a run without it takes the other
    loop; with memory again (polar: and its setters called again) the resident
    one."""
    asked, lacked = _passes(kind, stub, 0)[1], 0
    for n in range(1, asked + 1):
        stub.reset(fail_at=n)
        try:
            m = _model(kind=kind)
        except L.AwefdError:
            continue
        stub.reset()
        m.traces_dev()
        stub.reset(fail_above=1)
        m.run()
        lacked += stub.get("resident") == 0
        stub.reset()
        if kind == "spher2d":
            m.set_model(np.full((40, 30), 1.7e8, np.float32))
            x = np.array([[3387.5e3, 0.785]], np.float32)
            m.set_sources(x)
            m.set_receivers(x)
        m.run()
        assert stub.get("resident") == 1
        m.close()
    assert lacked > 0


def test_shots_of_a_batch_hold_no_rims(stub, monkeypatch):
    held = []
    for on in ("0", "1"):
        monkeypatch.setenv("AWEFD_RESIDENT", on)
        before = stub.get("bytes")
        ms = [_model(nt=30) for _ in range(2)]
        b = awefd.Batch(ms)
        for m in ms:
            m.set_sources(np.array([[20.0, 20.0]], np.float32))
        res, rp = _dev(30, 5)
        g, gp = _dev(40, 30)
        b.run()
        b.run_ckpt(0)
        b.adjoint_grad([rp, rp], gp)
        held.append(stub.get("bytes") - before)
        ms[0].run()                                  # one of them alone
        _grad(ms[0], 30)
        assert stub.get("resident") == (2 if on == "1" else 0) and stub.get("adjoint") == (on == "1")
        b.close()
        for m in ms:
            m.close()
        assert stub.get("bytes") == before
        stub.reset()
    assert 0 <= held[1] - held[0] < 2 * 4096         # two shots' flags and point tables


@pytest.mark.parametrize("kind", ["cart2d", "spher2d"])
def test_launch_errors_of_a_resident_loop(kind, stub):
    """A device that cannot hold the blocks (720) or launch them together
    (801), or whose cooperative queue another process has (401): the other
    loop, from then on.  A failed device or kernel is the run's error."""
    for code in (720, 801, 401):
        with _model(kind=kind) as m:
            stub.reset()
            stub.set("launch_error", code)
            m.run()
            m.run()
            assert stub.get("resident") == 1
    with _model(kind=kind) as m:
        stub.reset()
        stub.set("launch_error", 719)                # an earlier kernel failed
        with pytest.raises(L.AwefdError, match="resident"):
            m.run()


def test_launch_errors_of_the_resident_adjoint(stub):
    with _model() as m:
        L.check(m.lib.awefd_run_ckpt(m.h, None, 9))
        res, rp = _dev(m.nt, m.nr)
        g, gp = _dev(40, 30)
        stub.set("launch_error", 719)
        assert m.lib.awefd_adjoint_grad(m.h, rp, gp) == -2
        assert b"resident adjoint" in m.lib.awefd_last_error()
        stub.set("launch_error", 720)
        for _ in range(2):
            L.check(m.lib.awefd_adjoint_grad(m.h, rp, gp))
        assert stub.get("adjoint") == 2


@pytest.mark.parametrize("kind", ["cart2d", "spher2d"])
def test_a_loop_that_gave_up_is_not_tried_again(kind, stub, monkeypatch, capfd):
    """A wait that ends takes 4 s; a handle whose blocks did not get on pays
    it once, and says so."""
    monkeypatch.setenv("AWEFD_VERBOSE", "1")
    with _model(kind=kind) as m:
        stub.reset()
        stub.set("give_up", 1)
        m.run()
        assert stub.get("resident") == 1
        m.run()
        assert stub.get("resident") == 1
    assert "resident loop off" in capfd.readouterr().err


def test_an_adjoint_that_gave_up_is_not_tried_again(stub, monkeypatch, capfd):
    monkeypatch.setenv("AWEFD_VERBOSE", "1")
    with _model() as m:
        stub.reset()
        _grad(m, 9)
        assert stub.get("resident") == 1 and stub.get("adjoint") == 1
        stub.set("give_up", 1)
        res, rp = _dev(m.nt, m.nr)
        g, gp = _dev(40, 30)
        for _ in range(2):
            L.check(m.lib.awefd_adjoint_grad(m.h, rp, gp))
        assert stub.get("adjoint") == 2
        stub.set("give_up", 0)
        _grad(m, 9)                                  # the forward loop did get on
        assert stub.get("resident") == 2 and stub.get("adjoint") == 2
    assert "resident adjoint off" in capfd.readouterr().err


@pytest.mark.parametrize("kind", ["cart2d", "spher2d"])
def test_no_call_needs_the_legacy_stream(kind, stub):
    """hipMemcpy fails, and spoils the capture, while another thread captures a
    graph: handles of other threads must get on without it."""
    stub.set("capturing", 1)
    with _model(kind=kind) as m:
        m.run(jsnap=2, snapshots=True)
        m.run()
        m.traces()
        m.field()
        if kind == "spher2d":
            return
        _grad(m, 9)
        _grad(m, 3)
    m = _model(kind=kind, cden=False)
    m.set_model(np.full((40, 30), 1.7e8, np.float32), np.full((40, 30), 900.0, np.float32))
    m.run()
    ms = [_model(nt=30) for _ in range(2)]
    b = awefd.Batch(ms)
    res, rp = _dev(30, 5)
    g, gp = _dev(40, 30)
    for depth in (1, 2, 3):
        b.set_tile(8)
        b.set_depth(depth)
        b.run()
        for ckpt in (0, 30, 4):
            b.run_ckpt(ckpt)
            b.adjoint_grad([rp, rp], gp)
    b.close()
