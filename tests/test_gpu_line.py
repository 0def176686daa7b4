"""1D systems on the one-workgroup kernel (line.hip), at the edges of its
range: every transform length (the shortest ones share a wavefront, 4096
points take two), one to four transforms per stage, both noise draws, the
largest program that fits and one that does not.

Bars: relative L2 <= 1e-4 against the FP32 oracle (the repository's parity
bar), and <= 1e-5 against the general step program, which runs the same
operations in the same order: 20 steps of two transforms of at most 12 stages
and ~10 operations a bin, each rounded to 6e-8, differ by at most
20 * 34 * 6e-8 = 4e-5 if every rounding were worst case and aligned; the
roundings are independent, so sqrt(680) * 6e-8 = 1.6e-6 is expected."""
import numpy as np
import pytest

import cupss_amd as C
from oracle import oracle as O
from tests.helpers import build_system, rel_l2

pytestmark = pytest.mark.gpu


def kpz(n):
    return {"dims": (n, 1, 1), "dt": 0.005, "fields": [("h", True), ("dx", False)], "implicit": {"h": [(-1.0, 1)]},
            "terms": [("h", ["dx", "dx"], [(0.6,)]), ("dx", ["h"], [(1.0, 0, 1)])], "noise": {"h": ((0.02,), 11)},
            "init": {"h": np.zeros(n, np.float32)}}


def coupled(n):
    """Two dynamic fields, a solved constraint of their product, a coefficient field, noise on a constraint."""
    rng = np.random.default_rng(5)
    u = lambda: rng.uniform(-0.3, 0.3, n).astype(np.float32)  # noqa: E731
    return {"dims": (n, 1, 1), "dt": 0.01,
            "fields": [("u", True), ("p", False), ("v", True), ("c", False)],
            "implicit": {"u": [(-1.0, 1)], "v": [(-0.5, 1)], "p": [(1.0,), (0.5, 1)]},
            "terms": [("u", ["u", "v"], [(-0.4,)]), ("u", ["p"], [(0.3,), (0.1, 1)]), ("u", [], [(0.05,)]),
                      ("v", ["u", "u", "v"], [(0.2,)]), ("v", ["c", "u"], [(0.1, 0, 1)]),
                      ("p", ["u", "v"], [(1.0,)]), ("p", ["v"], [(1.0, 0, 1)])],
            "noise": {"p": ((0.01,), 3), "v": ((0.02, 1), 4)}, "init": {"u": u(), "v": u(), "c": u()}}


def run(spec, path, steps, mode=0):
    s, ids = build_system(C.System, C.pres, spec)
    s.set_path(path)
    s.set_noise_mode(mode)
    for k in steps:
        s.step(k)
    return {name: (s.get_real(i), s.get_dealiased(i)) for name, i in ids.items()}


@pytest.mark.parametrize("n", [2, 4, 8, 32, 128, 256, 1024, 2048, 4096])
@pytest.mark.parametrize("make", [kpz, coupled])
def test_line_equals_general_program_and_oracle(n, make):
    spec = make(n)
    print("line", make.__name__, n, flush=True)
    a, b = run(spec, 0, [20]), run(spec, 1, [20])
    o, oid = build_system(O.System, O.pres, dict(spec, precision="f32"))
    o.step(20)
    for name in a:
        scale = np.linalg.norm(b[name][0])
        if scale == 0:
            assert not np.any(a[name][0])
            continue
        assert rel_l2(a[name][0], b[name][0]) <= 1e-5, name
        assert np.linalg.norm(a[name][1] - b[name][1]) <= 1e-5 * scale, name
        assert rel_l2(a[name][0], o.get_real(oid[name])) <= 1e-4, name


@pytest.mark.parametrize("n", [2, 64, 1024, 4096])
def test_line_spectral_noise_equals_general_program(n):
    a, b = run(coupled(n), 0, [20], 1), run(coupled(n), 1, [20], 1)
    for name in a:
        assert rel_l2(a[name][0], b[name][0]) <= 1e-5, name


def test_line_runs_of_any_length_equal_one_run():
    """Odd and even runs, a parameter change and a reset between them."""
    spec = kpz(512)
    a, b = run(spec, 0, [21]), run(spec, 0, [1, 2, 1, 7, 10])
    for name in a:
        assert np.array_equal(a[name][0], b[name][0]) and np.array_equal(a[name][1], b[name][1]), name
    got = []
    for path in (0, 1):
        s, ids = build_system(C.System, C.pres, spec)
        s.set_path(path)
        s.step(5)
        s.set_implicits(ids["h"], [C.pres(-2.0, q2n=1)])
        s.step(4)
        s.set_real(ids["h"], np.sin(np.arange(512) * 2 * np.pi / 64).astype(np.float32))
        s.step(3)
        got.append(s.get_real(ids["h"]))
    assert rel_l2(got[0], got[1]) <= 1e-5


def test_line_program_too_large_for_one_workgroup():
    """Ten dealiased fields on 4096 points: the general program's launches."""
    n, rng = 4096, np.random.default_rng(6)
    names = ["u%d" % i for i in range(10)]
    spec = {"dims": (n, 1, 1), "dt": 0.01, "fields": [(m, True) for m in names],
            "implicit": {m: [(-1.0, 1)] for m in names},
            "terms": [(m, [m, names[(i + 1) % 10]], [(0.5,)]) for i, m in enumerate(names)],
            "init": {m: rng.uniform(-0.5, 0.5, n).astype(np.float32) for m in names}}
    a = run(spec, 0, [10])
    o, oid = build_system(O.System, O.pres, dict(spec, precision="f32"))
    o.step(10)
    for m in names:
        assert rel_l2(a[m][0], o.get_real(oid[m])) <= 1e-4
