"""GPU: a device allocation that is refused.  The multifrontal arena is then given back and
the call goes on, where there is one to give; every refused allocation of a life of a
handle is played in turn."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P
from swcholesky_amd._lib import SwcError, lib
import oracle_py as O
from helpers import full_csr, relF, setup

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _nothing_refused_afterwards():
    yield
    lib().swc_refuse_allocation(0)


def _operator():
    return P.laplacian3d_var(9, shift=1.0)


def _check(f, prob, b, Lo, rng):
    assert f.factor(prob.values) == 0
    assert relF(f.L_values(), Lo) < 1e-12
    A, rp, ci, v = full_csr(prob)
    B = rng.uniform(-1, 1, (prob.n, 3))
    X = f.solve(B)
    for k in range(3):
        assert O.backward_error(rp, ci, v, np.ascontiguousarray(X[:, k]), B[:, k].copy()) < 1e-14


def _mixed(f, prob):
    f.set_precision(2)
    assert f.factor(prob.values) == 0
    assert f.refine(np.ones(prob.n))[1][0] <= 1e-12


def test_upload_without_room_for_the_arena():
    prob = _operator()
    b, a2x, Lo, _ = setup(prob)
    rng = np.random.default_rng(1)
    for nth in range(1, 42):
        print(f"[no room] upload, allocation {nth}", flush=True)
        lib().swc_refuse_allocation(nth)
        f = S.Factor(b)
        lib().swc_refuse_allocation(0)
        _check(f, prob, b, Lo, rng)
        _check(f, prob, b, Lo, rng)  # captured
        _mixed(f, prob)


# the call, and how many allocations it makes
@pytest.mark.parametrize("what,count", [("solve", 7), ("refine", 7), ("precision", 1), ("inverse", 8),
                                        ("gradient", 16), ("csc", 4)])
def test_call_without_room_gives_up_the_arena(what, count):
    prob = _operator()
    b, a2x, Lo, _ = setup(prob)
    rng = np.random.default_rng(2)
    rhs = rng.uniform(-1, 1, (prob.n, 3))
    calls = {"solve": lambda f: f.solve(rhs), "refine": lambda f: f.refine(rhs)[0],
             "precision": lambda f: f.set_precision(1), "inverse": lambda f: f.selected_inverse(),
             "gradient": lambda f: f.gradient(rhs[:, 0], beta=1.0), "csc": lambda f: f.L_csc().toarray()}
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    want = calls[what](f)
    for nth in range(1, count + 1):
        print(f"[no room] {what}, allocation {nth}", flush=True)
        f = S.Factor(b)
        assert f.factor(prob.values) == 0 and f.factor(prob.values) == 0
        L = f.L_values()
        lib().swc_refuse_allocation(nth)
        got = calls[what](f)
        lib().swc_refuse_allocation(0)
        if want is not None:
            np.testing.assert_array_equal(got, want)  # the factor has not moved
        np.testing.assert_array_equal(f.L_values(), L)
        f.set_precision(0)
        for _ in range(3):  # the arena gone: left-looking, captured, replayed
            _check(f, prob, b, Lo, rng)
        _mixed(f, prob)


def test_a_handle_without_an_arena_reports_it():
    prob = _operator()
    b, a2x, Lo, _ = setup(prob)
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    lib().swc_refuse_allocation(1)
    f.solve(np.ones(prob.n))  # the arena goes
    lib().swc_refuse_allocation(1)
    with pytest.raises(SwcError):
        f.solve(np.ones((prob.n, 9)))
    _check(f, prob, b, Lo, np.random.default_rng(3))
