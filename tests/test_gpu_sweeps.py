"""GPU: the persistent solves against the CPU oracle, where their lists have every kind of
item: panels in parts, many more items than the device holds, a short last panel, leading
levels of narrow supernodes, right-hand sides around a group of 16."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P
import oracle_py as O
from helpers import full_csr

pytestmark = pytest.mark.gpu

CASES = [("lap3d_26", lambda: P.laplacian3d_var(26)), ("vec3d_13", lambda: P.vector3d_var(13)),
         ("lap2d_240", lambda: P.laplacian2d_var(240, 2)), ("dense_130", lambda: P.dense_spd(130))]


@pytest.fixture(scope="module", params=CASES, ids=[c[0] for c in CASES])
def case(request):
    prob = request.param[1]()
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    return prob, f, full_csr(prob)


@pytest.mark.parametrize("nrhs", [1, 2, 15, 16, 17, 40])
def test_solves_reach_oracle_backward_error(case, nrhs):
    """Each replay solves other right-hand sides: an entry left from the solve before, or
    taken before it is made, shows in the residual.  1e-14 is the solves' parity bar."""
    prob, f, (A, rp, ci, v) = case
    for rep in range(3):
        B = np.random.default_rng(100 * nrhs + rep).uniform(-1, 1, (prob.n, nrhs))
        X = f.solve(B)
        for j in range(nrhs):
            assert O.backward_error(rp, ci, v, np.ascontiguousarray(X[:, j]),
                                    np.ascontiguousarray(B[:, j])) < 1e-14


def test_solution_does_not_depend_on_timing(case):
    prob, f, _ = case
    B = np.random.default_rng(1).uniform(-1, 1, (prob.n, 20))
    x1, x20 = f.solve(B[:, 0]), f.solve(B)
    f.set_graphs(False)
    for _ in range(3):
        assert np.array_equal(f.solve(B[:, 0]), x1) and np.array_equal(f.solve(B), x20)
    f.set_graphs(True)


def test_nan_in_a_right_hand_side_comes_back_as_nan(case):
    """Entries in transit are marked by a NaN's bits; a right-hand side that holds those
    very bits (or any NaN) ends as NaN and keeps nobody waiting."""
    prob, f, _ = case
    b = np.random.default_rng(2).uniform(-1, 1, prob.n)
    clean = f.solve(b)
    for bits in (0x7ff4a5c35a3c4b21, 0x7ff8000000000000, 0x7ff0000000000000):
        bad = b.copy()
        bad[prob.n // 2] = np.array([bits], dtype=np.uint64).view(np.float64)[0]
        x = f.solve(bad)
        assert not np.isfinite(x[prob.n // 2])
    assert np.array_equal(f.solve(b), clean)
