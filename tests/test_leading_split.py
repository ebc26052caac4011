"""Leading levels of the solves that are split: supernodes with at most 16 rows below go 16
lanes each, the others a wave each."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
from swcholesky_amd.batch import Batch


def planes_and_volumes():
    """A forest whose leading level has leaves of both kinds."""
    return [P.laplacian2d_var(100, k) for k in range(5)] + [P.laplacian3d_var(14, k, shift=1e-2) for k in range(4)]


def _split(plan):
    return np.diff(plan["sweep_lvl_small"]), plan["sweep_lvl_small16"]


def _check_order(plan):
    sm, at = plan["sweep_small"], plan["sweep_lvl_small"]
    for l, n16 in enumerate(plan["sweep_lvl_small16"]):
        below = (sm["R"] - sm["w"])[at[l]:at[l + 1]]
        if n16:
            assert (below[:n16] <= 16).all() and (below[n16:] > 16).all()
            assert n16 == len(below) or n16 >= 2048


@pytest.mark.parametrize("make,packed", [(lambda: P.laplacian2d_var(240, 2), True),
                                         (lambda: P.laplacian3d_var(40, shift=1e-2), False)], ids=["lap2d_240", "lap3d_40"])
def test_whole_levels(make, packed):
    prob = make()
    plan = api.build_plan(S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm), derive_sets=True)
    n, n16 = _split(plan)
    assert len(n) and (n16 == (n if packed else 0)).all()
    _check_order(plan)


def test_split_level():
    plan = api.build_plan(Batch(planes_and_volumes()).bcsc, derive_sets=True)
    n, n16 = _split(plan)
    assert 2048 <= n16[0] < n[0]
    _check_order(plan)


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [1, 3])
def test_split_level_solves(nrhs):
    probs = planes_and_volumes()
    bt = Batch(probs)
    f = bt.factor
    assert f.factor(bt.values(probs)) == 0
    B = np.random.default_rng(3).standard_normal((bt.n, nrhs))
    X = f.solve(B)
    for k, p in enumerate(probs):  # every instance to its own backward error
        A = p.scipy_full()
        rows = slice(bt.offsets[k], bt.offsets[k + 1])
        x, b = X[rows], B[rows]
        eta = np.abs(A @ x - b).max(axis=0) / (abs(A).sum(axis=1).max() * np.abs(x).max(axis=0) + np.abs(b).max(axis=0))
        assert eta.max() < 1e-14
    assert np.array_equal(f.solve(B), X)
