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


def test_upload_frees_what_the_old_structure_held():
    """A handle that formed the selected inverse of a large structure and then takes a small one
    keeps nothing of the large one's size."""
    import torch
    large, small = P.laplacian3d_var(32, 1), P.laplacian3d_var(4, 1)
    bl, bs = (S.analyze_p2(p.n, p.colptr, p.rowidx, p.perm) for p in (large, small))
    f = S.Factor(bs)
    assert f.factor(small.values) == 0
    f.selected_inverse()
    before = torch.cuda.mem_get_info()[0]
    S._lib.check(S._lib.lib().swc_upload_symbolic(f._h, bl._h))
    f.bcsc, f.n = bl, bl.n
    assert f.factor(large.values) == 0
    f.logdet()
    S._lib.check(S._lib.lib().swc_selected_inverse(f._h, None, 0))
    used = before - torch.cuda.mem_get_info()[0]
    assert used > 3 * 8 * bl.xsize  # L, Z, update matrices and [T; U]
    S._lib.check(S._lib.lib().swc_upload_symbolic(f._h, bs._h))
    f.bcsc, f.n = bs, bs.n
    assert f.factor(small.values) == 0
    assert before - torch.cuda.mem_get_info()[0] < 0.05 * used
