"""What a fresh 3D system's first run sets up: the tiles follow from the box
alone (no timing runs), so equal systems run equal kernels."""
import pytest

import cupss_amd as C
from tests.helpers import build_system, spec_cahn_hilliard

pytestmark = pytest.mark.gpu


def box(dims, noise=True):
    spec = spec_cahn_hilliard(dims, seed=2)
    if noise:
        spec["noise"] = {"phi": ((0.02, 1), 8)}
    return spec


@pytest.mark.parametrize("dims,width", [
    ((32, 32, 32), 16), ((64, 64, 64), 8), ((32, 32, 128), 4), ((128, 64, 64), 8), ((256, 64, 64), 16),
    ((128, 128, 128), 16), ((64, 64, 16), 32), ((64, 64, 8), 64), ((32, 16, 512), 4), ((32, 16, 1024), 4)])
def test_z_tiles_follow_from_the_box(dims, width):
    print("z tiles", dims, flush=True)
    for noise in (True, False):
        s, _ = build_system(C.System, C.pres, box(dims, noise))
        s.profile_kernel(True)
        s.step(2)
        assert s.kernel_time()[2] == "k_f3z<%d, %d>" % (dims[2], width)
        s.close()
