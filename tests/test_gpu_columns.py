"""Transforms whose column pass takes 4 lines a workgroup (1024 points and more,
100 workgroups or more of them) and fewer lines on narrower grids, on both
sides of the line between them, forward and back.

Bars: relative L2 against numpy's 64-bit transform.  Each of the log2(n) <= 23
radix-2 levels rounds once or twice to 6e-8, the roundings are independent:
sqrt(2 * 23) * 6e-8 = 4e-7 expected, 2e-6 allowed; twice that there and back."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


# (kx, x) lines along y: 9 workgroups of 4, 33, 65, 100 (the line, in 3D), 129
@pytest.mark.parametrize("dims", [(64, 1024, 1), (64, 2048, 1), (256, 1024, 1), (512, 1024, 1), (1024, 1024, 1),
                                  (512, 2048, 1), (1024, 2048, 1), (16, 16, 1024), (32, 16, 1024), (32, 32, 1024),
                                  (64, 8, 1024), (32, 1024, 8)])
def test_long_columns(dims):
    print("columns", dims, flush=True)
    sx, sy, sz = dims
    n, nh = sx * sy * sz, (sx // 2 + 1) * sy * sz
    x = np.random.default_rng(1).standard_normal(n).astype(np.float32)
    a, b, c, d = (C.DeviceBuffer(s) for s in (4 * n, 8 * nh, 8 * nh, 4 * n))
    a.upload(x)
    C.check(C.lib().cupss_r2c(sx, sy, sz, a.ptr, b.ptr, None))
    C.check(C.lib().cupss_device_synchronize())
    got = b.download(np.float32, 2 * nh)
    want = np.fft.rfftn(x.astype(np.float64).reshape(sz, sy, sx))
    assert rel_l2(got[0::2] + 1j * got[1::2], want) <= 2e-6
    C.check(C.lib().cupss_c2r(sx, sy, sz, b.ptr, 0, 1.0 / n, d.ptr, c.ptr, None))
    C.check(C.lib().cupss_device_synchronize())
    assert rel_l2(d.download(np.float32, n), x) <= 4e-6
