"""GPU: handles come and go: more at once than one block of host records holds, freed in any
order, each reporting its own factorization."""
import gc

import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P

pytestmark = pytest.mark.gpu


def test_many_handles_report_their_own_results():
    prob = P.dense_spd(5)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    rng = np.random.default_rng(1)
    handles = [S.Factor(b) for _ in range(300)]
    for round_ in range(2):
        for k, f in enumerate(handles):
            assert f.factor(prob.values * (k + 1.0)) == 0
        want = handles[0].logdet()
        for k, f in enumerate(handles):
            assert np.isclose(f.logdet(), want + prob.n * np.log(k + 1.0), rtol=1e-12, atol=1e-12)
        bad = prob.values.copy()
        bad[-1] = -1.0
        assert handles[7].factor(bad) == prob.n and handles[8].info == 0
        for k in rng.permutation(300)[:200]:
            handles[k] = None
        gc.collect()
        handles = [S.Factor(b) if f is None else f for f in handles]
