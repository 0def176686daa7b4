"""The row tile's transforms of two fields and two products at a time: one to
three real fields with one to three products, so with and without a last
single one, at every row length and a few column lengths, against the general
step program.

Bar: relative L2 <= 1e-5.  Both run the same equations with the operations
rounded differently: 10 steps of at most six transforms of 24 stages and
about 20 operations a bin, independent roundings of 6e-8:
sqrt(10 * 164) * 6e-8 = 2.4e-6 expected."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2

pytestmark = pytest.mark.gpu

DIMS = [(16, 32), (32, 64), (64, 64), (128, 16), (256, 128), (512, 32), (1024, 16), (2048, 16), (4096, 8)]


def system(dims, nreal, nprod):
    n = dims[0] * dims[1]
    rng = np.random.default_rng(nreal)
    last = ["phi", "psi", "gx"][nreal - 1]
    # products in groups of their own: another operator or another target
    prods = [("phi", ["phi", last], [(-0.2, 1)]), ("phi", ["phi", "phi"] + ["psi"] * (nreal > 1), [(0.1,)]),
             ("psi", ["phi"] * 2 + [last], [(-0.1,)])][:nprod]
    return {"dims": dims + (1,), "dt": 0.01, "fields": [("phi", True), ("psi", True), ("gx", False)],
            "implicit": {"phi": [(-1.0, 1)], "psi": [(-0.5, 1)]},
            "terms": prods + [("psi", ["phi"], [(0.3,)]), ("gx", ["psi"], [(1.0, 0, 1)])],
            "init": {"phi": rng.uniform(-0.2, 0.2, n).astype(np.float32),
                     "psi": rng.uniform(-0.2, 0.2, n).astype(np.float32)}}


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("nprod", [1, 2, 3])
@pytest.mark.parametrize("nreal", [1, 2, 3])
def test_fields_and_products_in_pairs(nreal, nprod, dims):
    print("row pairs", nreal, "fields", nprod, "products", dims, flush=True)
    got = []
    for path in (0, 1):
        s, ids = build_system(C.System, C.pres, system(dims, nreal, nprod))
        s.set_path(path)
        assert path == 1 or s.fused_eligible
        s.step(7)
        s.step(3)
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[0][f], got[1][f]) <= 1e-5, f
