"""Update matrices that are not worth their size: such structures keep the left-looking plan."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
from swcholesky_amd._lib import SwcError
import oracle_py as O
from helpers import relF
from test_wide_borders import UNMERGED


def columns_below(nleaf, border):
    """Single columns, each coupled to all of a dense border."""
    n = nleaf + border
    r, c = (a.ravel() for a in np.tril_indices(border))
    rows = np.concatenate([np.arange(nleaf), np.tile(np.arange(nleaf, n), nleaf), r + nleaf])
    cols = np.concatenate([np.arange(nleaf), np.repeat(np.arange(nleaf), border), c + nleaf])
    vals = np.where(rows == cols, 2.0 * n, np.random.default_rng(1).uniform(-1, 1, rows.size))
    return P.Problem(n, *P.lower_csc_from_coo(n, rows, cols, vals), np.arange(n), f"columns_{nleaf}_{border}")


def _analysis(prob):
    return S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm, **UNMERGED)


@pytest.mark.parametrize("nleaf,border,fronts", [(300, 1000, False), (300, 600, True), (30, 1500, True)])
def test_rule(nleaf, border, fronts):
    b = _analysis(columns_below(nleaf, border))
    assert b.nsuper >= nleaf
    if fronts:
        assert api.build_fronts(b)["usize"] > 4 * b.xsize
    else:
        with pytest.raises(SwcError, match="no front tree"):
            api.build_fronts(b)


@pytest.mark.gpu
def test_factor_takes_little_memory():
    import torch
    prob = columns_below(300, 1000)
    b = _analysis(prob)
    Lo, _ = O.factor(b, b.a2_values(prob.values))
    small = columns_below(3, 3)
    S.Factor(_analysis(small)).factor(small.values)  # what the device keeps once per process
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    f = S.Factor(b)
    taken = before - torch.cuda.mem_get_info()[0]
    assert taken < 16 * 8 * b.xsize  # the update matrices are 230 times L
    for _ in range(3):  # uncaptured, captured, replayed
        assert f.factor(prob.values) == 0
        assert relF(f.L_values(), Lo) < 1e-12
    x = f.solve(np.ones(prob.n))
    A = prob.scipy_full()
    assert np.abs(A @ x - 1.0).max() <= 1e-14 * (abs(A).sum(axis=1).max() * np.abs(x).max() + 1.0)
