"""3D systems with the real-space draw: which route they take, and the row
variants of the fused one that other tests do not reach: 128 complex points
(eight elements a lane with up to three real fields), 512 and 1024 (rows over
several wavefronts).

Below 32^3 points the general program runs, bit for bit; from there on the
fused step, to the bar between the two (relative L2 <= 1e-5; see
test_gpu_noise3d.py)."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2
from tests.test_gpu_noise3d import system

pytestmark = pytest.mark.gpu


def run(spec, path, runs, mode=0):
    s, ids = build_system(C.System, C.pres, spec)
    s.set_path(path)
    s.set_noise_mode(mode)
    for k in runs:
        s.step(k)
    return {f: s.get_real(i) for f, i in ids.items()}, s.stat("fused_steps")


@pytest.mark.parametrize("dims", [(32, 32, 32), (16, 64, 32), (256, 16, 8), (256, 8, 32), (1024, 8, 8), (2048, 8, 8),
                                  (32, 1024, 8), (32, 8, 1024)])
@pytest.mark.parametrize("kind", ["noise only", "cubic", "gradients", "four fields"])
def test_fused_route_equals_general(kind, dims):
    print("3D real-space noise, route", kind, dims, flush=True)
    spec = system(dims, kind)
    # rows of more than three real fields need 32 to 1024 complex points
    fused = kind != "four fields" or 32 <= dims[0] // 2 <= 1024
    a, na = run(spec, 0, [12])
    b, nb = run(spec, 1, [12])
    c, nc = run(spec, 0, [5, 1, 6])
    assert (na, nb, nc) == ((12, 0, 12) if fused else (0, 0, 0))
    for f in a:
        assert rel_l2(a[f], b[f]) <= 1e-5, f
        assert np.array_equal(a[f], c[f]), f


@pytest.mark.parametrize("dims", [(16, 16, 16), (32, 32, 16), (16, 8, 8)])
def test_small_boxes_run_the_general_program(dims):
    spec = system(dims, "cubic")
    a, na = run(spec, 0, [12])
    b, _ = run(spec, 1, [12])
    assert na == 0
    for f in a:
        assert np.array_equal(a[f], b[f]), f
    _, ns = run(spec, 0, [12], 1)  # the spectral draw is fused at every size
    assert ns == 12
