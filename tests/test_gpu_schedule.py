"""The tiles that a batch's size classes take without timing runs, and that no
choice of tiles changes a bit."""
import re

import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, spec_cahn_hilliard, spec_kpz
from cupss_amd.systems import spec_gray_scott

pytestmark = pytest.mark.gpu


def tiles(specs, autotune):
    """(rows, columns) a workgroup of each size class after a run."""
    b = C.Batch(autotune=autotune)
    keep = [build_system(C.System, C.pres, spec)[0] for spec in specs]
    for s in keep:
        b.add(s)
    b.step(2)
    b.synchronize()
    got = [(int(m.group(1)), int(m.group(2)))
           for m in re.finditer(r"rows/wg (\d+), cols/wg (\d+)", b.schedule())]
    b.close()
    for s in keep:
        s.close()
    return got


# lanes of a column: the points by the elements a lane holds (8; 4 for 256 and
# from 1024 on; 16 at 4096)
@pytest.mark.parametrize("ny,lanes", [(8, 1), (32, 4), (64, 8), (256, 64), (512, 64), (1024, 256), (2048, 512),
                                      (4096, 256)])
def test_default_columns_keep_256_threads(ny, lanes):
    (rows, cols), = tiles([spec_cahn_hilliard((32, ny, 1))], False)
    assert rows == 8
    assert cols == max([1] + [c for c in (1, 2, 4, 8, 16) if c * lanes <= 256])


@pytest.mark.parametrize("autotune", [True, False])
@pytest.mark.parametrize("members,rows", [(1, 4), (62, 4), (63, 8)])
def test_128_square_takes_fixed_tiles(members, rows, autotune):
    """The lean class holds the Cahn-Hilliard systems and one KPZ system."""
    mixed = [spec_kpz(128), spec_gray_scott(128)]
    assert tiles([spec_cahn_hilliard((128, 128, 1))] * members + mixed, autotune) == [(rows, 2), (4, 2)]


@pytest.mark.parametrize("spec,name", [
    (spec_kpz(64), "k_fsmall<32, 64>"), (spec_gray_scott(64), "k_fsmall<32, 64, true, true>"),
    (spec_kpz(128), "k_fcols<128, 2>"), (spec_gray_scott(128), "k_fcols<128, 2, true, true>")])
def test_timed_kernel_is_the_one_launched(spec, name):
    """Simple systems run the lean kernels, which have no template flags."""
    s, _ = build_system(C.System, C.pres, spec)
    s.profile_kernel(True)
    s.step(4)
    assert s.kernel_time()[2] == name


def rect(spec, w, h):
    rng = np.random.default_rng(12)
    init = {f: rng.uniform(0.1, 0.5, w * h).astype(np.float32) for f, dyn in spec["fields"] if dyn}
    return dict(spec, dims=(w, h, 1), init=init)


def three_fields():
    spec = spec_kpz(8)
    return dict(spec, terms=spec["terms"] + [("h", ["h", "h"], [(-0.1,)]), ("h", ["h"], [(-0.05,)])])


@pytest.mark.parametrize("kind", [lambda: spec_gray_scott(8), three_fields, lambda: spec_kpz(8)],
                         ids=["two fields", "three fields", "lean"])
@pytest.mark.parametrize("dims", [(512, 32), (1024, 32), (2048, 32), (4096, 32), (2048, 256), (32, 2048)])
def test_tuned_and_default_tiles_give_equal_bits(kind, dims):
    got = []
    for autotune in (True, False, True):
        b = C.Batch(autotune=autotune)
        s, ids = build_system(C.System, C.pres, rect(kind(), *dims))
        b.add(s)
        b.step(9)
        print(dims, autotune, b.schedule().split("\n")[0], flush=True)
        got.append({f: s.get_real(i) for f, i in ids.items()})
        b.close()
        s.close()
    for f in got[0]:
        assert np.array_equal(got[0][f], got[1][f]) and np.array_equal(got[0][f], got[2][f]), f
