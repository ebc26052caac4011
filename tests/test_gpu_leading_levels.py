"""GPU: the solves' launches of leading levels of narrow supernodes, on both sides of the
rule that packs four supernodes into a wave."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P

pytestmark = pytest.mark.gpu


# most rows below a supernode of the leading level: at most 16 (16 lanes a supernode) in
# the first two, 48 (a wave a supernode) in the last
@pytest.mark.parametrize("make,packed", [(lambda: P.laplacian2d_var(240, 2), True), (lambda: P.gmrf2d(210), True),
                                         (lambda: P.laplacian3d_var(40, shift=1e-2), False)],
                         ids=["lap2d_240", "gmrf2d_210", "lap3d_40"])
def test_leading_levels_solve_to_rounding(make, packed):
    prob = make()
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    plan = api.build_plan(b)
    ls, sm = plan["sweep_lvl_small"], plan["sweep_small"]
    first = sm[ls[0]:ls[1]]
    assert ((first["R"] - first["w"]).max() <= 16) == packed
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    rhs = np.random.default_rng(3).standard_normal(prob.n)
    x = f.solve(rhs)
    A = prob.scipy_full()
    eta = np.abs(A @ x - rhs).max() / (abs(A).sum(axis=1).max() * np.abs(x).max() + np.abs(rhs).max())
    # longest sums of a row: fewer than 2,000 products, each within eps of the largest
    assert eta <= 2000 * np.finfo(float).eps
    assert np.array_equal(f.solve(rhs), x)
