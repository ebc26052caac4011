"""Narrow supernodes with thousands of rows below, as above a wide border."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
import oracle_py as O
from helpers import relF, setup
from test_gpu_fronts import arrow
from test_sweeps import _Sweeps

UNMERGED = {"nrelax": (0, 0, 0), "zrelax": (0.0, 0.0, 0.0)}


@pytest.mark.parametrize("border", [1100, 4090])
def test_solves_take_each_whole(border):
    """One item's work each, and its entries where the other items look for them."""
    prob = arrow(6, 2, border)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm, **UNMERGED)
    plan = api.build_plan(b)
    w, R = np.diff(b.super), np.diff(b.pi)
    assert plan["sweep_small"].shape[0] == ((w <= 16) & (R - w <= 4096)).sum() >= 4
    L = np.random.default_rng(0).uniform(-1e-3, 1e-3, b.xsize)
    for s in range(b.nsuper):
        L[b.p[b.super[s]] + np.arange(w[s]) * (R[s] + 1)] = 1.0
    rhs = np.random.default_rng(1).uniform(-1, 1, b.n)
    sw = _Sweeps(b, plan, L)
    sw.forward(rhs)
    x = sw.backward()
    assert relF(x, O.ltsolve(b, L, O.lsolve(b, L, rhs.copy()))[:, 0]) < 1e-11


@pytest.mark.gpu
@pytest.mark.parametrize("border", [1025, 4093, 4100])
def test_right_hand_sides_above_a_wide_border(border):
    prob = arrow(20, 2, border)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm, **UNMERGED)
    f = S.Factor(b)
    assert ((np.diff(b.super) <= 16) & (np.diff(b.pi) > border)).sum() >= 19
    assert f.factor(prob.values) == 0
    A = prob.scipy_full()
    rng = np.random.default_rng(border)
    for nrhs in (1, 2, 5, 33, 130):
        print(f"[border] {border} nrhs={nrhs}", flush=True)
        B = rng.uniform(-1, 1, (prob.n, nrhs))
        X = f.solve(B)
        assert np.array_equal(f.solve(B), X)
        eta = np.abs(A @ X - B).max(axis=0) / (abs(A).sum(axis=1).max() * np.abs(X).max(axis=0) + np.abs(B).max(axis=0))
        assert eta.max() < 1e-14
