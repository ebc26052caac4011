"""Descendant sets that leave out supernodes whose rows hold only zeros: the numbers they
give are those of the full sets, so the solves and the selected inverse, which read by the
row lists, must take their order from the rows."""
from types import SimpleNamespace

import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
from swcholesky_amd._lib import check, lib, ptr
import oracle_py as O
from helpers import full_csr, relF
from test_sweeps import _Sweeps


def cut_off_root(prob):
    """(problem, analysis, the analysis's arrays with an empty descendant set for the last
    supernode): every stored entry that couples its columns to others is zero."""
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    c0 = int(b.super[-2])
    col = np.repeat(np.arange(b.n), np.diff(b.a2p))
    values = prob.values.copy()
    values[b.a2src[(col < c0) & (b.a2i >= c0)]] = 0.0
    assert b.prunePtr[-1] > b.prunePtr[-2]
    less = SimpleNamespace(**{k: getattr(b, k) for k in ("n", "nsuper", "xsize", "super", "p", "i_ptr", "s", "pi")})
    less.prunePtr = b.prunePtr.copy()
    less.prunePtr[-1] = less.prunePtr[-2]
    less.pruneSet = b.pruneSet[:less.prunePtr[-1]].copy()
    return P.Problem(prob.n, prob.colptr, prob.rowidx, values, prob.perm, "cut"), b, less


MAKE = [lambda: P.laplacian2d_var(20, 1), lambda: P.laplacian3d_var(9, shift=1.0)]


@pytest.mark.parametrize("make", MAKE, ids=["lap2d_20", "lap3d_9"])
def test_sweeps_are_ordered_by_the_rows(make):
    prob, b, less = cut_off_root(make())
    Lo, info = O.factor(b, b.a2_values(prob.values))
    assert info == 0
    rhs = np.random.default_rng(1).uniform(-1, 1, b.n)
    sw = _Sweeps(b, api.build_plan(less), Lo)
    sw.forward(rhs)
    assert relF(sw.Y, O.lsolve(b, Lo, rhs.copy())[:, 0]) < 1e-12
    x = sw.backward()
    assert relF(x, O.ltsolve(b, Lo, O.lsolve(b, Lo, rhs.copy()))[:, 0]) < 1e-8


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [1, 3])
@pytest.mark.parametrize("make", MAKE, ids=["lap2d_20", "lap3d_9"])
def test_solve_and_inverse_with_shorter_sets(make, nrhs):
    prob, b, less = cut_off_root(make())
    Lo, _ = O.factor(b, b.a2_values(prob.values))
    f = S.Factor(b)
    p, iptr = b.p.astype(np.uint64), b.i_ptr.astype(np.uint64)
    check(lib().swc_upload(f._h, b.n, ptr(b.super), b.nsuper, ptr(p), ptr(b.s), ptr(iptr), ptr(less.prunePtr),
                           ptr(less.pruneSet), ptr(b.a2p), ptr(b.a2i), ptr(b.a2src), b.nnz))
    assert f.factor(prob.values) == 0
    assert relF(f.L_values(), Lo) < 1e-12
    B = np.random.default_rng(2).uniform(-1, 1, (b.n, nrhs))
    X = f.solve(B)
    A, rp, ci, v = full_csr(prob)
    for k in range(nrhs):
        assert O.backward_error(rp, ci, v, np.ascontiguousarray(X[:, k]), B[:, k].copy()) < 1e-14
    Z = f.selected_inverse()
    inv = np.linalg.inv(A.toarray()[np.ix_(b.Perm, b.Perm)])
    for s in range(b.nsuper):
        c0, c1 = b.super[s], b.super[s + 1]
        rows = b.s[b.pi[s]:b.pi[s + 1]]
        blk = Z[b.p[c0]:b.p[c0] + len(rows) * (c1 - c0)].reshape(c1 - c0, len(rows)).T
        low = rows[:, None] >= np.arange(c0, c1)[None, :]
        ref = inv[np.ix_(rows, np.arange(c0, c1))]
        # n eps cond(A) bounds either inverse's error
        tol = b.n * np.finfo(float).eps * np.linalg.cond(A.toarray()) * np.abs(inv).max()
        assert np.abs(np.where(low, blk - ref, 0.0)).max() <= tol
