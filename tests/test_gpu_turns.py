"""Systems that change hands: alone, in one batch, in another, with runs of
odd and even length and reads in between.  The step counters and buffer order
on the device follow the runs only when needed, so every handover must find
them right: the state equals an uninterrupted twin's bit for bit.  A system
with stored fields starts a run that cannot continue the one before with the
general program's operations in place of a pass's: relative L2 <= 1e-5 there
(the bar between the two programs)."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2, spec_cahn_hilliard, spec_diffusion, spec_kpz
from cupss_amd.systems import spec_gray_scott, spec_model_h

pytestmark = pytest.mark.gpu

KINDS = {
    "kpz 64": (lambda: spec_kpz(64, seed=3), 0),
    "kpz 128 spectral": (lambda: spec_kpz(128, seed=4), 1),
    "gray-scott 128": (lambda: spec_gray_scott(128), 0),
    "model h 128": (lambda: spec_model_h(128), 0),
    "cahn-hilliard 32x64": (lambda: spec_cahn_hilliard((32, 64, 1), seed=6), 0),
    "diffusion 64": (lambda: spec_diffusion(64, sigma=5.0), 0),
    "edwards-wilkinson 64 spectral": (lambda: spec_kpz(64, lam=0.0, seed=9), 1),
}


STORED = ("gray-scott 128", "model h 128")


def make(name):
    mk, mode = KINDS[name]
    s, ids = build_system(C.System, C.pres, mk())
    s.set_noise_mode(mode)
    return s, ids


def same(s, ids, name, steps):
    twin, tid = make(name)
    twin.step(steps)
    for f, i in ids.items():
        for got, want in ((s.get_real(i), twin.get_real(tid[f])), (s.get_dealiased(i), twin.get_dealiased(tid[f]))):
            if name in STORED:
                assert rel_l2(got, want) <= 1e-5 or not np.any(want), (name, f, steps)
            else:
                assert np.array_equal(got, want), (name, f, steps)


@pytest.mark.parametrize("name", list(KINDS))
def test_two_batches_take_turns(name):
    print("turns", name, flush=True)
    a, b = C.Batch(autotune=False), C.Batch(autotune=False)
    other, _ = make("kpz 64")
    a.add(other)
    a.step(1)
    s, ids = make(name)
    n = 0

    def run(batch, runs, read=False):
        nonlocal n
        batch.add(s)
        for k in runs:
            batch.step(k)
            n += k
            if read:
                s.get_real(ids[list(ids)[0]])
        batch.remove(s)

    run(a, [3])
    run(b, [1, 2])
    s.step(1)
    n += 1
    same(s, ids, name, n)
    run(a, [1], True)
    run(b, [2, 1, 1], True)
    run(a, [5, 1])
    same(s, ids, name, n)
    assert other.step_count == 1 + 3 + 1 + 6
    same(other, {"h": 0}, "kpz 64", 11)
    a.close()
    b.close()


@pytest.mark.parametrize("name", list(KINDS))
def test_reads_between_runs(name):
    s, ids = make(name)
    n = 0
    for k in (1, 1, 2, 1, 3, 1):
        s.step(k)
        n += k
        same(s, ids, name, n)


def test_one_member_read_between_runs_of_a_batch():
    """Only some descriptors change between the runs."""
    b = C.Batch(autotune=False)
    members = [(k, *make(k)) for k in KINDS]
    for _, s, _ in members:
        b.add(s)
    n = 0
    for j, k in enumerate((1, 2, 1, 1, 3, 1)):
        b.step(k)
        n += k
        name, s, ids = members[j % len(members)]
        same(s, ids, name, n)
        if j == 3:
            f = C.ctypes.c_void_p()
            C.check(s.L.cupss_field_spectrum_device(s.h, ids[list(ids)[0]], C.ctypes.byref(f)))
    for name, s, ids in members:
        same(s, ids, name, n)
    b.close()
