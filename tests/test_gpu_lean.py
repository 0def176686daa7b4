"""Simple systems on the lean row and column tiles (lean_tiles.hpp): grids at
the edges of the tiles (shortest and longest rows and columns, one column
tile, the one-workgroup class 64^2 and its neighbours), each product form,
operator and noise draw the lean program holds, and systems just outside it,
against the general step program.

Bar: relative L2 <= 1e-5.  Both run the same equations with the operations
rounded differently: 10 steps of at most three transforms of 24 stages and
about 20 operations a bin, independent roundings of 6e-8: sqrt(10 * 92) * 6e-8
= 2e-6 expected."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2

pytestmark = pytest.mark.gpu


def base(dims, terms, imp, noise=None, extra=(), dt=0.01):
    n = dims[0] * dims[1]
    x0 = np.random.default_rng(9).uniform(-0.2, 0.2, n).astype(np.float32)
    s = {"dims": dims + (1,), "dt": dt, "fields": [("u", True)] + [(name, False) for name, _ in extra],
         "implicit": {"u": imp}, "terms": terms + [(name, ["u"], p) for name, p in extra], "init": {"u": x0}}
    if noise:
        s["noise"] = {"u": (noise, 21)}
    return s


DX, DY = ("dx", [(1.0, 0, 1)]), ("dy", [(1.0, 0, 0, 1)])
SYSTEMS = {
    "cubic": lambda d: base(d, [("u", ["u"] * 3, [(-1.0, 1)])], [(1.0, 1), (-1.0, 2)]),
    "gradients": lambda d: base(d, [("u", ["dx", "dx"], [(0.7,)]), ("u", ["dy", "dy"], [(0.4,)])], [(-1.0, 1)], (0.02,),
                                [DX, DY], 0.005),
    "flux": lambda d: base(d, [("u", ["u", "dx"], [(0.3, 0, 1)]), ("u", ["u", "u"], [(0.2, 0, 1)])], [(-0.5, 1)],
                           (0.01, 1), [DX]),
    "linear": lambda d: base(d, [("u", [], [(0.3,), (5.0, 1)])], [(-0.2,), (-1.0, 1), (0.1, 2), (-0.2, 3)], (0.02, 1)),
    "no implicit": lambda d: base(d, [("u", ["u", "u"], [(-0.5,)]), ("u", [], [(0.1,)])], []),
    "single term (not lean)": lambda d: base(d, [("u", ["u", "u"], [(-0.5,)]), ("u", ["u"], [(0.4, 1)])], [(-1.0, 1)]),
    "inverse q (not lean)": lambda d: base(d, [("u", ["u", "u"], [(-0.5, 1, 0, 0, 0, 1)])], [(-1.0, 1)], (0.02,)),
    "two groups (not lean)": lambda d: base(d, [("u", ["u", "u"], [(-0.5,)]), ("u", ["u"] * 3, [(0.3, 1)])], [(-1.0, 1)]),
}
DIMS = [(16, 8), (16, 64), (32, 32), (64, 64), (64, 128), (128, 128), (256, 16), (512, 256), (1024, 64), (2048, 16),
        (4096, 8), (16, 1024), (32, 2048), (16, 4096)]


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("name", sorted(SYSTEMS))
def test_lean_equals_general_program(name, dims):
    spec = SYSTEMS[name](dims)
    for mode in ((0, 1) if "noise" in spec else (0,)):
        print("lean", name, dims, "noise mode", mode, flush=True)
        got = []
        for path in (0, 1):
            s, ids = build_system(C.System, C.pres, spec)
            s.set_path(path)
            s.set_noise_mode(mode)
            s.step(7)
            s.step(3)
            got.append({f: s.get_real(i) for f, i in ids.items()})
        for f in got[0]:
            assert rel_l2(got[0][f], got[1][f]) <= 1e-5, f


def test_lean_state_changes_between_runs():
    """New state, step, prefactors and dt between runs of a lean system."""
    got = []
    for path in (0, 1):
        s, ids = build_system(C.System, C.pres, SYSTEMS["gradients"]((64, 32)))
        s.set_path(path)
        u = ids["u"]
        s.step(3)
        s.set_implicits(u, [C.pres(-2.0, q2n=1), C.pres(-0.1, q2n=2)])
        s.step(2)
        C.check(s.L.cupss_system_set_dt(s.h, 0.002))
        s.step(5)
        s.set_real(u, np.cos(np.arange(64 * 32) * 2 * np.pi / 64).astype(np.float32))
        s.step(4)
        got.append(s.get_real(u))
    assert rel_l2(got[0], got[1]) <= 1e-5
