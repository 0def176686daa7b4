"""Which 1D programs the one-workgroup kernel takes, and what it does with
those that only its longer lines run with several wavefronts a transform:
spectral noise, noise on a solved constraint, products of three factors.

A line of n points has n/2 complex ones: up to 512 of them one wavefront takes
a transform (lanes beyond a short one's repeat its work), 1024 take four and
2048 eight wavefronts.  The program's arrays must fit 153600 bytes of LDS.

Bars as for the other 1D tests: relative L2 <= 1e-5 against the general step
program, which runs the same operations in the same order (20 steps of at most
34 roundings a bin in a chain, sqrt(680) * 6e-8 = 1.6e-6 expected), and <= 1e-4
against the FP32 oracle (real-space noise)."""
import numpy as np
import pytest

import cupss_amd as C
from oracle import oracle as O
from tests.helpers import build_system, rel_l2
from tests.test_gpu_line import coupled, kpz

pytestmark = pytest.mark.gpu

STEPS = 20


def cubic_constraint(n):
    """A solved constraint with noise and a product of three factors."""
    x = np.random.default_rng(8).uniform(-0.5, 0.5, n).astype(np.float32)
    return {"dims": (n, 1, 1), "dt": 0.01, "fields": [("u", True), ("p", False)],
            "implicit": {"u": [(-1.0, 1)], "p": [(1.0,), (0.5, 1)]},
            "terms": [("u", ["p"], [(0.4,)]), ("p", ["u", "u", "u"], [(-1.0,)])],
            "noise": {"p": ((0.02,), 7)}, "init": {"u": x}}


def run(spec, path, mode, runs=(STEPS,)):
    s, ids = build_system(C.System, C.pres, spec)
    s.set_path(path)
    s.set_noise_mode(mode)
    for k in runs:
        s.step(k)
    return {f: (s.get_real(i), s.get_dealiased(i)) for f, i in ids.items()}, s


@pytest.mark.parametrize("make,n,mode,fits", [
    (kpz, 2, 0, True), (kpz, 1024, 0, True), (kpz, 2048, 0, True), (kpz, 4096, 0, True),
    (kpz, 2048, 1, True), (kpz, 4096, 1, True),
    (coupled, 256, 0, True), (coupled, 1024, 0, True), (coupled, 1024, 1, True),
    (coupled, 2048, 1, True), (coupled, 2048, 0, False), (coupled, 4096, 0, False), (coupled, 4096, 1, False),
    (cubic_constraint, 128, 0, True), (cubic_constraint, 2048, 0, True), (cubic_constraint, 2048, 1, True),
    (cubic_constraint, 4096, 0, True), (cubic_constraint, 4096, 1, True)])
def test_route_and_result(make, n, mode, fits):
    print("line route", make.__name__, n, mode, flush=True)
    a, s = run(make(n), 0, mode)
    assert s.stat("line_steps") == (STEPS if fits else 0)
    b, g = run(make(n), 1, mode)
    assert g.stat("line_steps") == 0
    for f in a:
        for x, y in zip(a[f], b[f]):
            assert rel_l2(x, y) <= 1e-5 or not np.any(y), f
    c, _ = run(make(n), 0, mode, (1, 2, 7, 10))
    for f in a:
        for x, y in zip(a[f], c[f]):
            assert np.array_equal(x, y), f
    if mode == 0:
        o, oid = build_system(O.System, O.pres, dict(make(n), precision="f32"))
        o.step(STEPS)
        for f in a:
            want = o.get_real(oid[f])
            assert rel_l2(a[f][0], want) <= 1e-4 or not np.any(want), f


@pytest.mark.parametrize("n,fits", [(1024, True), (4096, False)])
def test_a_program_is_laid_out_once(n, fits):
    """Not again at every call, whether it fits or not; again when it changes."""
    s, ids = build_system(C.System, C.pres, coupled(n))
    for _ in range(5):
        s.step(1)
    assert s.stat("line_plans") == 1
    s.set_implicits(ids["u"], [C.pres(-2.0, q2n=1)])
    for _ in range(3):
        s.step(1)
    assert s.stat("line_plans") == 2
    assert s.stat("line_steps") == (8 if fits else 0)


def test_unknown_counts_are_refused():
    s, _ = build_system(C.System, C.pres, kpz(64))
    with pytest.raises(C.CupssError):
        s.stat("no such count")
    assert s.stat("fused_steps") == 0
