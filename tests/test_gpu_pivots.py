"""Pivots that are not positive, in every block of 16 columns of a panel: the sweeps that
factor a block run without a test in each column and are done again with one."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,col", [(8, 3), (16, 0), (16, 15), (40, 20), (40, 39), (64, 16), (64, 63), (90, 5), (90, 70)])
@pytest.mark.parametrize("value", [-1.0, 0.0, float("nan")])
def test_first_bad_pivot_is_reported_and_the_next_factor_is_sound(n, col, value):
    prob = P.dense_spd(n, seed=5)  # one supernode of n columns
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    f = S.Factor(b)
    cols = np.repeat(np.arange(n), np.diff(prob.colptr))
    bad = prob.values.copy()
    bad[(prob.rowidx == cols) & (cols == b.Perm[col])] = value
    assert f.factor(bad) == col + 1
    assert f.factor(prob.values) == 0
    Ap = prob.scipy_full().toarray()[np.ix_(b.Perm, b.Perm)]
    L = f.L_values()
    ref = np.linalg.cholesky(Ap)
    # both factors carry errors of about n eps |L| (the operator is well conditioned)
    err = 0.0
    for s in range(b.nsuper):
        c0, c1 = b.super[s], b.super[s + 1]
        rows = b.s[b.pi[s]:b.pi[s + 1]]
        blk = L[b.p[c0]:b.p[c0] + len(rows) * (c1 - c0)].reshape(c1 - c0, len(rows)).T
        keep = rows[:, None] >= np.arange(c0, c1)[None, :]
        err = max(err, np.abs(np.where(keep, blk - ref[np.ix_(rows, np.arange(c0, c1))], 0.0)).max())
    assert err <= 10 * n * np.finfo(float).eps * np.linalg.cond(Ap) * np.abs(ref).max()
