"""cupss_system_device_bytes of 2D systems: what admission by memory counts
for the operator tables of the fused step is no less than what it makes."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system
from cupss_amd.systems import spec_gray_scott

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pres", [(0.1, 0, 0, 0, 2), (0.1, 1, 0, 0, 0, 1)], ids=["qz", "1/|q|"])
def test_operators_that_become_tables_are_counted(pres):
    """A table is one float per bin."""
    base = spec_gray_scott(64)
    got = []
    for extra in ([("u", ["u"], [(0.1,)])], [("u", ["u"], [pres])]):
        s, ids = build_system(C.System, C.pres, dict(base, terms=base["terms"] + extra))
        got.append(s.device_bytes())
        s.step(3)
        assert np.all(np.isfinite(s.get_real(ids["u"])))
        assert s.device_bytes() == got[-1]
    assert got[1] - got[0] == 4 * s.nh
