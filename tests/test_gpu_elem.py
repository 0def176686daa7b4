"""Simple systems without transforms (diffusion and its noisy and driven
forms) on the lean elementwise kernel, and runs whose step counters the
device descriptors follow only when something needs them: one-step runs,
reads, new values and replays in between, batches in which such systems stand
beside systems with transforms.

Bars: against the general program relative L2 <= 1e-5 (13 steps of about 30
operations a bin, independent roundings of 6e-8, and one transform pair:
sqrt(13 * 30 + 40) * 6e-8 = 1.3e-6 expected); the same steps in other runs,
or in a batch, give the same bits."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2, spec_cahn_hilliard

pytestmark = pytest.mark.gpu


def spec(dims, kind):
    x0 = np.random.default_rng(3).uniform(-0.2, 0.2, dims[0] * dims[1]).astype(np.float32)
    s = {"dims": dims + (1,), "dt": 0.02, "fields": [("u", True), ("du", False)], "implicit": {"u": [(-1.0, 1), (-0.1, 3)]},
         "terms": [("du", ["u"], [(1.0, 0, 1), (0.5, 1, 0, 1)])], "init": {"u": x0}}
    if kind != "diffusion":
        s["terms"].append(("u", [], [(0.3,)]))
        s["noise"] = {"u": ((0.05, 1), 8)}
    if kind == "not lean":
        s["terms"].append(("u", ["u"], [(0.2, 1)]))
    return s


def make(sp, path=0):
    s, ids = build_system(C.System, C.pres, sp)
    s.set_path(path)
    s.set_noise_mode(1)
    return s, ids


@pytest.mark.parametrize("dims", [(16, 8), (64, 32), (256, 256), (16, 4096), (4096, 8)])
@pytest.mark.parametrize("kind", ["diffusion", "noisy", "not lean"])
def test_runs_equal_general_program_and_each_other(kind, dims):
    print("elementwise", kind, dims, flush=True)
    got = []
    for path, runs, read in ((1, [13], False), (0, [13], False), (0, [1] * 13, False), (0, [1, 2, 1, 3, 6], True)):
        s, ids = make(spec(dims, kind), path)
        for k in runs:
            s.step(k)
            if read:
                s.get_real(ids["u"])
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[1][f], got[0][f]) <= 1e-5, f
        assert np.array_equal(got[1][f], got[2][f]) and np.array_equal(got[1][f], got[3][f]), f


@pytest.mark.parametrize("graph", [0, 4])
def test_batch_of_one_step_runs(graph):
    specs = [spec((64, 32), "noisy"), spec((32, 64), "not lean"), spec((64, 64), "diffusion"),
             spec_cahn_hilliard((64, 64, 1), seed=5), spec_cahn_hilliard((128, 64, 1), seed=6)]
    batch = C.Batch(graph_steps=graph)
    members = [make(sp) for sp in specs]
    for s, _ in members:
        batch.add(s)
    for k in (1, 1, 3, 9, 1, 1, 4, 2):
        batch.step(k)
    members[3][0].get_real(members[3][1]["phi"])  # one member read: its state written back
    batch.step(1)
    batch.step(2)
    for sp, (s, ids) in zip(specs, members):
        alone, ia = make(sp)
        alone.step(25)
        for f in ids:
            assert np.array_equal(alone.get_real(ia[f]), s.get_real(ids[f])), f


def test_new_values_between_one_step_runs():
    got = []
    for path in (1, 0):
        s, ids = make(spec((64, 32), "noisy"), path)
        for _ in range(3):
            s.step(1)
        s.set_implicits(ids["u"], [C.pres(-2.0, q2n=1), C.pres(-0.05, q2n=3)])
        for _ in range(3):
            s.step(1)
        s.set_real(ids["u"], np.cos(np.arange(64 * 32) * 2 * np.pi / 64).astype(np.float32))
        for _ in range(3):
            s.step(1)
        C.check(s.L.cupss_system_set_dt(s.h, 0.01))
        for _ in range(2):
            s.step(2)
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[1][f], got[0][f]) <= 1e-5, f
