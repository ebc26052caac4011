"""GPU: several right-hand sides, on both sides of the rule that takes them one or 16 to an
item of the sweeps, and with every share of a last group."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
from test_gpu_fronts import arrow

pytestmark = pytest.mark.gpu


def band(n, k):
    """Diagonally dominant band matrix in natural order: a chain of n / 16 supernodes."""
    r = np.concatenate([np.arange(d, n) for d in range(k + 1)])
    c = np.concatenate([np.arange(n - d) for d in range(k + 1)])
    v = np.where(r == c, 2.0 * k + 1, -1.0 / (1 + r - c))
    return P.Problem(n, *P.lower_csc_from_coo(n, r, c, v), np.arange(n), f"band_{n}_{k}")


CASES = {"lap3d_12": lambda: P.laplacian3d_var(12, 1), "vec3d_6": lambda: P.vector3d_var(6, 1),
         "dense_130": lambda: P.dense_spd(130), "band_900_7": lambda: band(900, 7),
         "diagonal_3000": lambda: band(3000, 0), "lap2d_240": lambda: P.laplacian2d_var(240, 2),
         "arrow_300_1_30": lambda: arrow(300, 1, 30)}


@pytest.mark.parametrize("name", list(CASES))
def test_right_hand_sides_on_both_sides_of_the_rule(name):
    prob = CASES[name]()
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    most = api.build_plan(b)["sweep_one_each"]
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    A = prob.scipy_full()
    rng = np.random.default_rng(1)
    past = [most + d for d in (1, 2, 5, 16, 17)] if most < 400 else []
    for nrhs in sorted({2, 3, 5, 17, max(most, 2)} | set(past)):
        if nrhs > 1200:
            continue
        print(f"[groups] {name} nrhs={nrhs} most={most}", flush=True)
        B = rng.uniform(-1, 1, (prob.n, nrhs))
        X = f.solve(B)
        assert np.array_equal(f.solve(B), X)
        eta = np.abs(A @ X - B).max(axis=0) / (abs(A).sum(axis=1).max() * np.abs(X).max(axis=0) + np.abs(B).max(axis=0))
        assert eta.max() < 1e-14
        for j in {0, nrhs // 2, nrhs - 1}:
            x = f.solve(B[:, j])
            if nrhs <= most:  # the same work, one item each
                assert np.array_equal(X[:, j], x)
            else:  # sums in another order: condition times rounding
                assert np.linalg.norm(X[:, j] - x) <= 1e-8 * np.linalg.norm(x)
