"""GPU: factorizations replayed from their captured sequence.  The first factorization of a
structure in a precision mode is launched kernel by kernel, the second captures and launches
the sequence, later ones replay it."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P
import oracle_py as O
from helpers import full_csr, relF, setup
from test_gpu_fronts import EDGES, arrow

pytestmark = pytest.mark.gpu


def test_replay_after_the_solve_workspace_grew():
    """A solve with 8 right-hand sides moves the solve workspace after the factor's sequence was
    captured; the replayed refactorization reports info and ||A||_inf of the new values."""
    prob = P.laplacian3d_var(20)
    b, a2x, Lo, _ = setup(prob)
    f = S.Factor(b)
    rhs = np.random.default_rng(4).uniform(-1, 1, (prob.n, 8))
    f.factor(prob.values)
    f.solve(rhs[:, 0])
    for rep in range(2):  # launched, captured
        assert f.factor(prob.values) == 0
    f.solve(rhs)
    for scale in (2.0, 0.25, 3.0):  # replayed
        v = prob.values * scale
        assert f.factor(v) == 0
        Ls, _ = O.factor(b, b.a2_values(v))
        assert relF(f.L_values(), Ls) < 1e-12
        A, rp, ci, av = full_csr(P.Problem(prob.n, prob.colptr, prob.rowidx, v, prob.perm, "scaled"))
        x, eta, _ = f.refine(rhs[:, 0], tol=1e-12)
        assert eta[0] <= 1e-12
        xp = x + 1e-6 * np.random.default_rng(5).standard_normal(prob.n)
        assert np.isclose(f.backward_error(rhs[:, 0], xp)[0], O.backward_error(rp, ci, av, xp, rhs[:, 0]), rtol=1e-10)


@pytest.mark.parametrize("nleaf,leaf,ncore", EDGES)
def test_replays_at_front_edges(nleaf, leaf, ncore):
    prob = arrow(nleaf, leaf, ncore)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm, nrelax=(0, 0, 0), zrelax=(0.0, 0.0, 0.0))
    Lo, _ = O.factor(b, b.a2_values(prob.values))
    f = S.Factor(b)
    for mode in (0, 1, 2):
        f.set_precision(mode)
        L = []
        for rep in range(4):  # launched, captured, replayed twice
            assert f.factor(prob.values) == 0
            L.append(f.L_values())
            assert np.array_equal(L[rep], L[0])
        if mode == 0:
            assert relF(L[3], Lo) < 1e-12


def test_replays_of_each_precision_mode():
    """Every mode keeps its own sequence: switching back and forth gives each mode's eager
    factor, bitwise, and replays see new values."""
    prob = P.vector3d_var(6)
    b, a2x, Lo, _ = setup(prob)
    f = S.Factor(b)
    f.set_graphs(False)
    eager = {}
    for mode in (0, 1, 2):
        f.set_precision(mode)
        assert f.factor(prob.values) == 0
        eager[mode] = f.L_values()
    assert not np.array_equal(eager[0], eager[1])
    f.set_graphs(True)
    for mode in (1, 0, 2, 1, 1, 0, 2, 1, 0, 2, 0):
        f.set_precision(mode)
        assert f.factor(4.0 * prob.values) == 0
        assert np.array_equal(f.L_values(), 2.0 * eager[mode])  # powers of two: the same rounding
        assert f.factor(prob.values) == 0
        assert np.array_equal(f.L_values(), eager[mode])
