"""GPU: what the reported solve time covers."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P
from swcholesky_amd._lib import check, lib, ptr

pytestmark = pytest.mark.gpu


def test_solve_time_covers_the_marks_with_an_ordering():
    """The launch that marks the work vectors belongs to the solve: with an ordering it also
    permutes B, so the reported time cannot be shorter than without one (4 of 81 us here)."""
    import torch
    prob = P.laplacian2d_const(100)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    B = torch.ones(prob.n, dtype=torch.float64, device="cuda")
    perm = np.ascontiguousarray(b.Perm, dtype=np.int32)
    times = {True: [], False: []}
    for rep in range(200):
        for ordered in (True, False):
            check(lib().swc_set_perm(f._h, ptr(perm) if ordered else None))
            f.solve_device(B)
            times[ordered].append(f.timings()["solve_ms"])
            B.fill_(1.0)
            torch.cuda.synchronize()
    assert np.median(times[True][20:]) >= 0.99 * np.median(times[False][20:])
