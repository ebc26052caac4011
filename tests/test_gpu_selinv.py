"""Selected inverse at the edges of its kernels: 16-column small supernodes, 32 x 32 product
tiles, 64 x 64 blocks of T = L11^{-1}, and a factor larger than one chunk of levels."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P

pytestmark = pytest.mark.gpu


def _factor(prob):
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    return b, f


# one supernode of n columns: around 16, 32, 64 and 128; grids give rows below around 64
@pytest.mark.parametrize("make", [lambda n=n: P.dense_spd(n, seed=3) for n in (2, 15, 16, 17, 31, 33, 63, 64, 65, 127, 130)]
                         + [lambda: P.laplacian3d_var(10), lambda: P.gmrf2d(40), lambda: P.vector3d_var(5)])
def test_selected_inverse_dense_oracle(make):
    prob = make()
    b, f = _factor(prob)
    Z = f.selected_inverse()
    Ap = prob.scipy_full().toarray()[np.ix_(b.Perm, b.Perm)]
    Ainv = np.linalg.inv(Ap)
    # both inverses carry errors of about cond(A) eps |A^-1|
    tol = max(1e-12, 20 * np.linalg.cond(Ap) * np.finfo(float).eps) * np.abs(Ainv).max()
    for s in range(b.nsuper):
        c0, c1 = b.super[s], b.super[s + 1]
        rows = b.s[b.pi[s]:b.pi[s + 1]]
        blk = Z[b.p[c0]:b.p[c0] + len(rows) * (c1 - c0)].reshape(c1 - c0, len(rows)).T
        ref = np.where(rows[:, None] >= np.arange(c0, c1)[None, :], Ainv[np.ix_(rows, np.arange(c0, c1))], 0.0)
        assert np.abs(blk - ref).max() <= tol, (s, len(rows), c1 - c0)


def test_several_chunks_and_repeats():
    """A factor of more than one chunk (8.4 M values); a second factor of the same handle."""
    prob = P.laplacian3d_var(30, shift=1.0)
    b, f = _factor(prob)
    assert b.xsize > 1 << 23
    rng = np.random.default_rng(0)
    for scale in (1.0, 4.0):
        assert f.factor(prob.values * scale) == 0
        Z = f.selected_inverse()
        for s in [b.nsuper - 1, b.nsuper - 2, 0] + list(rng.integers(0, b.nsuper, 9)):
            c = int(rng.integers(b.super[s], b.super[s + 1]))
            rows = b.s[b.pi[s]:b.pi[s + 1]]
            keep = rows >= c
            e = np.zeros(prob.n)
            e[b.Perm[c]] = 1.0
            col = f.solve(e)[b.Perm[rows[keep]]]
            z = Z[b.p[c]:b.p[c] + len(rows)][keep]
            # eigenvalues between 1 and 1200 (weights up to 100, six neighbours)
            assert np.abs(col - z).max() <= 20 * 1200 * np.finfo(float).eps * np.abs(col).max(), (s, c)
