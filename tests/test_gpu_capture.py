"""A caller's own stream under graph capture: a run recorded by the caller
and replayed takes the system on by its steps every time, also after runs
that were not recorded, with the noise of the steps that the replay takes.

The recorded run and a run taken directly launch the same kernels, so the
state after any mix of them equals the state of an uninterrupted twin bit
for bit."""
import ctypes

import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, spec_cahn_hilliard, spec_diffusion, spec_kpz
from cupss_amd.systems import spec_gray_scott, spec_model_h

pytestmark = pytest.mark.gpu

VP = ctypes.c_void_p


def hip(name, *args):
    """A HIP runtime call of the runtime that the library itself uses."""
    fn = getattr(C.lib(), name)
    fn.restype = ctypes.c_int
    rc = fn(*args)
    assert rc == 0, "%s: HIP error %d" % (name, rc)


class Stream:
    def __init__(self):
        self.s, self.keep = VP(), []
        hip("hipStreamCreateWithFlags", ctypes.byref(self.s), ctypes.c_uint(1))

    def record(self, work):
        """The launches of work() as an executable graph (relaxed mode)."""
        g, ex = VP(), VP()
        hip("hipStreamBeginCapture", self.s, ctypes.c_int(2))
        try:
            work()
        finally:
            hip("hipStreamEndCapture", self.s, ctypes.byref(g))
        hip("hipGraphInstantiate", ctypes.byref(ex), g, None, None, ctypes.c_size_t(0))
        self.keep.append((g, ex))
        return ex

    def replay(self, ex):
        hip("hipGraphLaunch", ex, self.s)
        hip("hipStreamSynchronize", self.s)

    def close(self):
        for g, ex in self.keep:
            hip("hipGraphExecDestroy", ex)
            hip("hipGraphDestroy", g)
        hip("hipStreamDestroy", self.s)


SYSTEMS = {
    "kpz 64": (lambda: spec_kpz(64, seed=3), 0),
    "kpz 128": (lambda: spec_kpz(128, seed=3), 0),
    "kpz 128 spectral": (lambda: spec_kpz(128, seed=4), 1),
    "gray-scott 64": (lambda: spec_gray_scott(64), 0),
    "model h 128": (lambda: spec_model_h(128), 0),
    "cahn-hilliard 256x64": (lambda: spec_cahn_hilliard((256, 64, 1), seed=6), 0),
    "diffusion 64": (lambda: spec_diffusion(64, sigma=5.0), 0),
    "edwards-wilkinson 64 spectral": (lambda: spec_kpz(64, lam=0.0, seed=9), 1),
}


def make(name):
    mk, mode = SYSTEMS[name]
    s, ids = build_system(C.System, C.pres, mk())
    s.set_noise_mode(mode)
    return s, ids


@pytest.mark.parametrize("n", [2, 3])
@pytest.mark.parametrize("before", [2, 5])
@pytest.mark.parametrize("name", list(SYSTEMS))
def test_replayed_runs_go_on(name, before, n):
    print("capture", name, before, n, flush=True)
    st = Stream()
    s, ids = make(name)
    C.check(s.L.cupss_system_set_stream(s.h, st.s))
    s.step(1)
    s.step(before)
    ex = st.record(lambda: s.step(n))
    st.replay(ex)
    st.replay(ex)
    s.step(2)
    st.replay(ex)
    s.step(1)
    got = {f: s.get_real(i) for f, i in ids.items()}
    twin, tid = make(name)
    twin.step(1 + before + 2 * n + 2 + n + 1)
    for f in got:
        assert np.array_equal(got[f], twin.get_real(tid[f])), f
    s.close()
    st.close()


@pytest.mark.parametrize("before", [1, 2, 5])
@pytest.mark.parametrize("name", list(SYSTEMS))
def test_recordings_in_any_order(name, before):
    """Two recordings one after the other, a direct run before either is
    replayed, the second replayed first."""
    print("capture order", name, before, flush=True)
    st = Stream()
    s, ids = make(name)
    C.check(s.L.cupss_system_set_stream(s.h, st.s))
    s.step(1)
    s.step(before)
    two = st.record(lambda: s.step(2))
    four = st.record(lambda: s.step(4))
    if before != 2:
        s.step(1)
    st.replay(four)
    st.replay(two)
    s.step(1)
    st.replay(two)
    s.step(2)
    got = {f: s.get_real(i) for f, i in ids.items()}
    twin, tid = make(name)
    twin.step(1 + before + (before != 2) + 4 + 2 + 1 + 2 + 2)
    for f in got:
        assert np.array_equal(got[f], twin.get_real(tid[f])), f
    s.close()
    st.close()


def test_replayed_runs_of_a_batch_go_on():
    """Members with transforms, of one workgroup each and elementwise; two
    recorded runs of different lengths."""
    print("capture batch", flush=True)
    st = Stream()
    names = ["kpz 64", "kpz 128 spectral", "diffusion 64", "edwards-wilkinson 64 spectral", "model h 128"]
    b = C.Batch.__new__(C.Batch)
    b.L, b.h, b.members = C.lib(), VP(), []
    C.check(b.L.cupss_batch_create(st.s, ctypes.byref(b.h)))
    members = [make(k) for k in names]
    for s, _ in members:
        b.add(s)
    b.step(1)
    b.step(2)
    e1 = st.record(lambda: b.step(1))
    st.replay(e1)
    b.step(2)
    e4 = st.record(lambda: b.step(4))
    st.replay(e4)
    for ex in (e1, e4, e1):
        st.replay(ex)
    b.step(1)
    total = 3 + 1 + 2 + 4 + 6 + 1
    for (s, ids), k in zip(members, names):
        twin, tid = make(k)
        twin.step(total)
        for f, i in ids.items():
            assert np.array_equal(s.get_real(i), twin.get_real(tid[f])), (k, f)
    b.close()
    for s, _ in members:
        s.close()
    st.close()


def line(n, noise):
    """A Burgers-like line: one product, with or without noise."""
    x = np.sin(2 * np.pi * np.arange(n) / n).astype(np.float32)
    spec = {"dims": (n, 1, 1), "dt": 0.01, "fields": [("u", True), ("dx", False)], "implicit": {"u": [(-1.0, 1)]},
            "terms": [("u", ["u", "dx"], [(-0.5,)]), ("dx", ["u"], [(1.0, 0, 1)])], "init": {"u": x}}
    if noise:
        spec["noise"] = {"u": ((0.02,), 5)}
    return spec


def box(dims):
    """Model B with conserved noise, the real-space draw."""
    spec = spec_cahn_hilliard(dims, seed=2)
    spec["noise"] = {"phi": ((0.02, 1), 8)}
    return spec


@pytest.mark.parametrize("spec", [line(256, True), box((32, 32, 32)), box((64, 32, 16))], ids=["line", "cube", "box"])
def test_first_run_of_a_fresh_system_recorded(spec):
    """Nothing is set up inside the graph: it holds the general program."""
    print("recorded first run", spec["dims"], flush=True)
    st = Stream()
    s, ids = build_system(C.System, C.pres, spec)
    C.check(s.L.cupss_system_set_stream(s.h, st.s))
    st.replay(st.record(lambda: s.step(2)))
    twin, tid = build_system(C.System, C.pres, spec)
    twin.set_path(1)
    twin.step(2)
    for f, i in ids.items():
        assert np.array_equal(s.get_real(i), twin.get_real(tid[f])), f
    # and on by direct runs (another route: rounding apart)
    s.step(3)
    twin.step(3)
    for f, i in ids.items():
        assert np.linalg.norm(s.get_real(i) - twin.get_real(tid[f])) <= 1e-5 * np.linalg.norm(twin.get_real(tid[f])), f
    s.close()
    st.close()


def test_recorded_line_goes_on():
    st = Stream()
    s, ids = build_system(C.System, C.pres, line(512, False))
    C.check(s.L.cupss_system_set_stream(s.h, st.s))
    s.step(3)
    ex = st.record(lambda: s.step(2))
    for _ in range(3):
        st.replay(ex)
    twin, tid = build_system(C.System, C.pres, line(512, False))
    twin.step(9)
    for f, i in ids.items():
        assert np.array_equal(s.get_real(i), twin.get_real(tid[f])), f
    s.close()
    st.close()


def test_recorded_box_goes_on_between_direct_runs():
    """Direct runs between replays leave what the recorded general steps read
    as they expect it.  (The replayed steps draw the noise of the steps that
    were recorded.)"""
    spec = box((32, 32, 32))
    st = Stream()
    s, ids = build_system(C.System, C.pres, spec)
    C.check(s.L.cupss_system_set_stream(s.h, st.s))
    ex = st.record(lambda: s.step(2))
    st.replay(ex)
    s.step(2)
    st.replay(ex)
    s.step(1)
    twin, tid = build_system(C.System, C.pres, spec)
    twin.set_path(1)
    twin.step(4)
    C.check(twin.L.cupss_system_set_step(twin.h, 0))
    twin.step(2)
    C.check(twin.L.cupss_system_set_step(twin.h, 4))
    twin.step(1)
    for f, i in ids.items():
        want = twin.get_real(tid[f])
        assert np.linalg.norm(s.get_real(i) - want) <= 1e-5 * np.linalg.norm(want), f
    s.close()
    st.close()
