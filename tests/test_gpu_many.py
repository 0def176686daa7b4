"""Many instances of one size at once: launches of more than 4096 rows of 256
or 512 complex points take the fields of a row singly, smaller ones in pairs;
either way a member equals the system alone bit for bit (the same operations
in the same order)."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, spec_kpz
from cupss_amd.systems import spec_gray_scott

pytestmark = pytest.mark.gpu


def reactants(w, h, seed):
    """Gray-Scott on a rectangle: two real fields, one product for each."""
    spec = spec_gray_scott(8)
    rng = np.random.default_rng(seed)
    return dict(spec, dims=(w, h, 1), init={f: rng.uniform(0.2, 0.6, w * h).astype(np.float32) for f in ("u", "v")})


def slopes(w, h, seed):
    """Three real fields, three products in two groups."""
    spec = spec_kpz(8, seed=seed)
    terms = spec["terms"] + [("h", ["h", "h"], [(-0.1,)]), ("h", ["h", "iqxh"], [(0.2, 0, 1)]),
                             ("h", ["h"], [(-0.05,)])]
    x = np.random.default_rng(seed).uniform(-0.3, 0.3, w * h).astype(np.float32)
    return dict(spec, dims=(w, h, 1), terms=terms, init={"h": x})


@pytest.mark.parametrize("make", [reactants, slopes])
@pytest.mark.parametrize("w,h,members", [(512, 64, 63), (512, 64, 65), (512, 512, 9), (1024, 64, 66), (128, 128, 40),
                                         (2048, 32, 130)])
def test_members_equal_the_system_alone(make, w, h, members):
    print("many", make.__name__, w, h, members, flush=True)
    b = C.Batch(autotune=members % 2 == 0)
    keep = [build_system(C.System, C.pres, make(w, h, 5 + i % 3)) for i in range(members)]
    for s, _ in keep:
        b.add(s)
    b.step(3)
    b.step(4)
    for k in (0, 1, 2, members - 1):
        alone, aid = build_system(C.System, C.pres, make(w, h, 5 + k % 3))
        alone.step(3)
        alone.step(4)
        s, ids = keep[k]
        for f, i in ids.items():
            assert np.array_equal(s.get_real(i), alone.get_real(aid[f])), (k, f)
    b.close()
    for s, _ in keep:
        s.close()


@pytest.mark.parametrize("members", [3, 128, 129])
@pytest.mark.parametrize("mode", [0, 1])
def test_one_step_runs_of_small_simple_systems(members, mode):
    """64^2: runs of one step of up to 128 instances take two launches, longer
    ones and those of more instances one workgroup each."""
    print("one-step runs", members, mode, flush=True)
    b = C.Batch()
    keep = [build_system(C.System, C.pres, spec_kpz(64, seed=3 + i % 4)) for i in range(members)]
    for s, _ in keep:
        s.set_noise_mode(mode)
        b.add(s)
    runs = (1, 1, 4, 1, 2, 1)
    for k in runs:
        b.step(k)
    for k in (0, 1, 2, members - 1):
        for whole in ((sum(runs),), runs):
            alone, aid = build_system(C.System, C.pres, spec_kpz(64, seed=3 + k % 4))
            alone.set_noise_mode(mode)
            for n in whole:
                alone.step(n)
            s, ids = keep[k]
            for f, i in ids.items():
                assert np.array_equal(s.get_real(i), alone.get_real(aid[f])), (k, f, whole)
    b.close()
    for s, _ in keep:
        s.close()
