"""A supernode of many blocks whose thousands of children have rows in few of them each."""
import time

import numpy as np

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
from helpers import relF, setup
from test_fronts import _Emulation


def _numbered_tree(n):
    """A binary tree numbered from its root: its factor ends in one wide supernode."""
    i = np.arange(1, n)
    r, c = np.concatenate([i, np.arange(n)]), np.concatenate([(i - 1) // 2, np.arange(n)])
    colptr, rowidx, values = P.lower_csc_from_coo(n, r, c, np.where(r == c, 4.0, -1.0))
    return P.Problem(n, colptr, rowidx, values, np.arange(n), f"tree_{n}")


def test_emulated_fronts_match_oracle():
    prob = _numbered_tree(900)
    b, a2x, Lo, _ = setup(prob)
    plan = api.build_fronts(b)
    assert np.diff(b.super).max() > 64
    assert relF(_Emulation(b, plan, a2x, np.random.default_rng(0)).run(), Lo) < 1e-12


def test_lists_take_no_longer_than_the_plan_of_the_solves():
    prob = _numbered_tree(30000)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)

    def best(build):
        t = []
        for _ in range(4):
            t0 = time.process_time()
            build(b)
            t.append(time.process_time() - t0)
        return min(t)
    # 39 and 13 ms where every tile of the root asked every child; 7 and 13 now
    assert best(api.build_fronts) < 1.5 * best(api.build_plan)
