"""Operators of the general fused 2D tiles: monomials and divisor polynomials
evaluated in the tile, and sums, 1/|q| and powers above q^6 read from tables,
each in a group, a single-field term, a derived field, a second dynamic field
and a constraint, at grids on both sides of the tiles' widths, against the
general step program; the tables follow new parameters and a new dt.

Bar: relative L2 <= 1e-5.  Both run the same equations with the operations
rounded differently: 10 steps of at most six transforms of 22 stages and
about 30 operations a bin, independent roundings of 6e-8:
sqrt(10 * 162) * 6e-8 = 2.4e-6 expected."""
import numpy as np
import pytest

import cupss_amd as C
from tests.helpers import build_system, rel_l2, spec_model_h

pytestmark = pytest.mark.gpu

# operators with and without the factor i
OPS = {"monomial": ([(-0.2, 1)], [(0.3, 1, 1)]),
       "sum": ([(-0.2, 1), (0.01, 2), (0.1,)], [(0.3, 0, 1), (-0.2, 0, 0, 1)]),
       "inverse q": ([(-0.2, 0, 1, 1, 0, 1)], [(0.3, 0, 1, 0, 0, 1)]),
       "sum with inverse q": ([(-0.2, 1, 0, 0, 0, 1), (0.1,)], [(0.3, 0, 1, 0, 0, 1), (0.1, 0, 0, 1)])}
# divisors of the constraint (the dynamic fields take the negative)
DIVS = {"polynomial": [(1.0,), (0.5, 1), (0.25, 1), (0.1, 2), (0.01, 3)],
        "q^8": [(1.0,), (0.001, 4)],
        "inverse q": [(1.0,), (0.5, 1, 0, 0, 0, 1)]}
DIMS = [(64, 32), (64, 64), (128, 128), (512, 64), (64, 256), (1024, 16), (128, 1024)]


def system(dims, ops, div):
    """dt phi + D phi = A phi^3 + A w;  dt psi + D psi = B phi + psi w;  gx = B psi;  D w = A psi + gx^2"""
    even, odd = OPS[ops]
    d = DIVS[div]
    neg = [(-p[0],) + tuple(p[1:]) for p in d]
    n = dims[0] * dims[1]
    rng = np.random.default_rng(6)
    return {"dims": dims + (1,), "dt": 0.01, "fields": [("phi", True), ("psi", True), ("gx", False), ("w", False)],
            "implicit": {"phi": neg, "psi": neg, "w": d},
            "terms": [("phi", ["phi"] * 3, even), ("phi", ["w"], even), ("psi", ["phi"], odd),
                      ("psi", ["psi", "w"], [(-0.1,)]), ("gx", ["psi"], odd), ("w", ["psi"], even),
                      ("w", ["gx", "gx"], [(0.2,)])],
            "init": {"phi": rng.uniform(-0.2, 0.2, n).astype(np.float32),
                     "psi": rng.uniform(-0.2, 0.2, n).astype(np.float32)}}


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("div", sorted(DIVS))
@pytest.mark.parametrize("ops", sorted(OPS))
def test_operators_equal_general_program(ops, div, dims):
    print("operators", ops, div, dims, flush=True)
    got = []
    for path in (0, 1):
        s, ids = build_system(C.System, C.pres, system(dims, ops, div))
        s.set_path(path)
        assert path == 1 or s.fused_eligible
        s.step(7)
        s.step(3)
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[0][f], got[1][f]) <= 1e-5, f


def test_tables_follow_parameters():
    got = []
    for path in (0, 1):
        s, ids = build_system(C.System, C.pres, system((64, 32), "sum with inverse q", "inverse q"))
        s.set_path(path)
        s.step(3)
        s.set_implicits(ids["w"], [C.pres(2.0), C.pres(0.3, q2n=1, invq=1)])
        s.step(2)
        C.check(s.L.cupss_system_set_dt(s.h, 0.005))
        s.step(3)
        s.set_implicits(ids["phi"], [C.pres(-0.5), C.pres(-0.002, q2n=4)])
        s.step(2)
        got.append({f: s.get_real(i) for f, i in ids.items()})
    for f in got[0]:
        assert rel_l2(got[0][f], got[1][f]) <= 1e-5, f


def test_fields_read_between_runs_change_nothing():
    """The fields a first run starts from are made only where it reads them."""
    spec = spec_model_h(64)
    one, ids = build_system(C.System, C.pres, spec)
    two, _ = build_system(C.System, C.pres, spec)
    gen, _ = build_system(C.System, C.pres, spec)
    gen.set_path(1)
    for k in (1, 4, 5):
        two.step(k)
        gen.step(k)
        for f, i in ids.items():
            assert rel_l2(two.get_real(i), gen.get_real(i)) <= 1e-4 or np.abs(gen.get_real(i)).max() < 1e-6, f
    one.step(10)
    for f, i in ids.items():
        assert np.array_equal(one.get_real(i), two.get_real(i)), f
