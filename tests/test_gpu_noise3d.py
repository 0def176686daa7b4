"""3D systems with the real-space noise draw on the fused step: boxes at the
edges of its tiles (shortest rows and lines, unequal sides, one column tile),
one to four real fields, plain and conserved noise, against the general step
program and split into runs.

Bar: relative L2 <= 1e-5 (as for the noiseless 3D step): the same operations
rounded in another order, 12 steps of up to four transforms of 21 stages and
about 20 operations a bin, independent roundings of 6e-8:
sqrt(12 * 104) * 6e-8 = 2e-6 expected."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2

pytestmark = pytest.mark.gpu


def system(dims, kind):
    n = dims[0] * dims[1] * dims[2]
    x0 = np.random.default_rng(4).uniform(-0.2, 0.2, n).astype(np.float32)
    d = [("dx", [(1.0, 0, 1)]), ("dy", [(1.0, 0, 0, 1)]), ("dz", [(1.0, 0, 0, 0, 1)])]
    if kind == "noise only":
        fields, terms, noise, d = [("u", True)], [("u", [], [(0.1,)])], (0.02,), []
    elif kind == "cubic":
        fields, terms, noise, d = [("u", True)], [("u", ["u"] * 3, [(-1.0, 1)])], (0.02, 1), []
    elif kind == "gradients":
        fields = [("u", True)] + [(m, False) for m, _ in d]
        terms, noise = [("u", [m, m], [(0.4,)]) for m, _ in d], (0.02,)
    else:  # four real fields, two groups, a single-field term
        fields = [("u", True)] + [(m, False) for m, _ in d]
        terms = [("u", [m, m], [(0.4,)]) for m, _ in d] + [("u", ["u", "dx"], [(0.2, 0, 1)]), ("u", ["dy"], [(0.1,)])]
        noise = (0.02,)
    return {"dims": dims, "dt": 0.005, "fields": fields, "implicit": {"u": [(-1.0, 1)]},
            "terms": terms + [(m, ["u"], p) for m, p in d], "noise": {"u": (noise, 17)}, "init": {"u": x0}}


@pytest.mark.parametrize("dims", [(32, 32, 32), (64, 64, 8), (16, 64, 32), (512, 8, 8), (128, 16, 64), (32, 128, 16)])
@pytest.mark.parametrize("kind", ["noise only", "cubic", "gradients", "four fields"])
def test_noise_3d_fused_equals_general(kind, dims):
    print("3D real-space noise", kind, dims, flush=True)
    spec = system(dims, kind)
    got = []
    for path, runs in ((0, [12]), (1, [12]), (0, [5, 1, 6])):
        s, ids = build_system(C.System, C.pres, spec)
        s.set_path(path)
        for k in runs:
            s.step(k)
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[0][f], got[1][f]) <= 1e-5, f
        assert np.array_equal(got[0][f], got[2][f]), f
