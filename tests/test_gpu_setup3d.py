"""What a fresh 3D system's first run sets up: the tiles follow from the box
alone (no timing runs), so equal systems run equal kernels, and the fused step
works in the buffers that the system has anyway (the dealiased copies, the
product transforms, the noise and the transform scratch), whatever is read or changed between runs."""
import ctypes

import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2, spec_cahn_hilliard

pytestmark = pytest.mark.gpu


def box(dims, noise=True):
    spec = spec_cahn_hilliard(dims, seed=2)
    if noise:
        spec["noise"] = {"phi": ((0.02, 1), 8)}
    return spec


@pytest.mark.parametrize("dims,width", [
    ((32, 32, 32), 16), ((64, 64, 64), 8), ((32, 32, 128), 4), ((128, 64, 64), 8), ((256, 64, 64), 16), ((64, 256, 256), 8),
    ((128, 128, 128), 16), ((64, 64, 16), 32), ((64, 64, 8), 64), ((32, 16, 512), 4), ((32, 16, 1024), 4)])
def test_z_tiles_follow_from_the_box(dims, width):
    print("z tiles", dims, flush=True)
    for noise in (True, False):
        s, _ = build_system(C.System, C.pres, box(dims, noise))
        s.profile_kernel(True)
        s.step(2)
        assert s.kernel_time()[2] == "k_f3z<%d, %d>" % (dims[2], width)
        s.close()


def free_bytes():
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    fn = C.lib().hipMemGetInfo  # of the runtime that the library itself uses
    assert fn(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


@pytest.mark.parametrize("noise", [True, False])
def test_first_run_allocates_no_field_buffers(noise):
    s, ids = build_system(C.System, C.pres, box((128, 128, 128), noise))
    s.synchronize()
    before = free_bytes()
    s.step(3)
    s.synchronize()
    assert before - free_bytes() < 4 << 20  # one spectrum is 8.5 MB
    s.close()


def gradients(dims):
    """Four real fields, two groups of products."""
    n = dims[0] * dims[1] * dims[2]
    d = [("dx", [(1.0, 0, 1)]), ("dy", [(1.0, 0, 0, 1)]), ("dz", [(1.0, 0, 0, 0, 1)])]
    return {"dims": dims, "dt": 0.005, "fields": [("u", True)] + [(m, False) for m, _ in d],
            "implicit": {"u": [(-1.0, 1)]},
            "terms": [("u", [m, m], [(0.4,)]) for m, _ in d] + [("u", ["u", "dx"], [(0.2, 0, 1)])] +
                     [(m, ["u"], p) for m, p in d],
            "noise": {"u": ((0.02,), 17)},
            "init": {"u": np.random.default_rng(4).uniform(-0.2, 0.2, n).astype(np.float32)}}


@pytest.mark.parametrize("dims", [(32, 32, 32), (16, 64, 32)])
def test_reading_dealiased_copies_between_runs(dims):
    """Reading them changes no bit of what follows; they are the general
    program's, before a field's first update (zero) and after."""
    spec = gradients(dims)
    a, ia = build_system(C.System, C.pres, spec)
    b, ib = build_system(C.System, C.pres, spec)
    g, ig = build_system(C.System, C.pres, spec)
    g.set_path(1)
    for k in (0, 5, 1, 4):
        a.step(k)
        b.step(k)
        g.step(k)
        for f in ia:
            x, y = a.get_dealiased(ia[f]), g.get_dealiased(ig[f])
            assert np.array_equal(x, a.get_dealiased(ia[f])), f
            assert np.linalg.norm(x - y) <= 1e-5 * np.linalg.norm(y), f
    for f in ia:
        assert np.array_equal(a.get_real(ia[f]), b.get_real(ib[f])), f


def many(dims):
    """Five real fields in one product: more fields than there are buffers to
    transform them from."""
    n = dims[0] * dims[1] * dims[2]
    ops = {"a": (1.0, 0, 1), "b": (1.0, 0, 0, 1), "c": (1.0, 0, 0, 0, 1), "d": (0.5, 1)}
    return {"dims": dims, "dt": 0.002, "fields": [("u", True)] + [(m, False) for m in ops],
            "implicit": {"u": [(-1.0, 1)]},
            "terms": [("u", ["u", "a", "b", "c", "d"], [(-0.8,)])] +
                     [(m, ["u"], [p]) for m, p in ops.items()],
            "init": {"u": np.random.default_rng(6).uniform(-0.4, 0.4, n).astype(np.float32)}}


@pytest.mark.parametrize("dims", [(64, 16, 32), (64, 64, 64)])
def test_five_real_fields(dims):
    spec = many(dims)
    got = []
    for path, runs in ((0, [8]), (1, [8]), (0, [3, 1, 4])):
        s, ids = build_system(C.System, C.pres, spec)
        s.set_path(path)
        s.profile_kernel(True)
        for k in runs:
            s.step(k)
        if path == 0:
            assert s.kernel_time()[2].startswith("k_f3z<")
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[0][f], got[1][f]) <= 1e-5, f
        assert np.array_equal(got[0][f], got[2][f]), f


def test_routes_and_resets_between_runs():
    """Fused runs, general steps and a reset field in turn, against the
    general program alone."""
    spec = gradients((32, 32, 32))
    got = []
    for first in (0, 1):
        s, ids = build_system(C.System, C.pres, spec)
        s.set_path(first)
        s.step(4)
        s.set_path(1)
        s.step(2)
        s.set_path(first)
        s.step(3)
        s.set_real(ids["u"], spec["init"]["u"][::-1].copy())
        s.step(3)
        got.append({f: (s.get_real(i), s.get_dealiased(i)) for f, i in ids.items()})
    for f in got[0]:
        for x, y in zip(got[0][f], got[1][f]):
            assert rel_l2(x, y) <= 1e-5, f


def test_a_narrower_mask_after_runs():
    """A cubic term added after runs with a quadratic one narrows the dealias
    mask: nothing of the wider one is left in the real fields, so the runs
    that follow equal those of a system of both terms from the same state."""
    x = np.random.default_rng(9).uniform(-0.5, 0.5, 32 ** 3).astype(np.float32)

    def quadratic():
        s = C.System(32, 32, 32, dt=0.002)
        u = s.add_field(True)
        s.add_implicit(u, C.pres(-0.1, q2n=1))
        s.add_term(u, [u, u], [C.pres(-0.5)])
        s.set_real(u, x)
        return s, u

    a, u = quadratic()
    a.prepare()
    a.step(3)
    z = a.get_spectrum(u)
    a.add_term(u, [u, u, u], [C.pres(-1.0)])
    a.prepare()
    a.step(10)
    b, u = quadratic()
    b.add_term(u, [u, u, u], [C.pres(-1.0)])
    b.prepare()
    b.step(1)  # the field has been updated: its dealiased copy is no longer zero
    flat = np.stack([z.real, z.imag], axis=-1).astype(np.float32).ravel()
    C.check(b.L.cupss_field_set_spectrum(b.h, u, flat.ctypes.data_as(ctypes.POINTER(ctypes.c_float))))
    b.step(10)
    assert np.array_equal(a.get_real(u), b.get_real(u))
