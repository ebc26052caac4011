"""GPU: the entries of A that an upload takes: any order within a column, none outside the
structure."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import problems as P
from swcholesky_amd._lib import SwcError, check, lib, ptr

pytestmark = pytest.mark.gpu


def _upload(f, b, a2i, a2src):
    p, iptr = b.p.astype(np.uint64), b.i_ptr.astype(np.uint64)
    check(lib().swc_upload(f._h, b.n, ptr(b.super), b.nsuper, ptr(p), ptr(b.s), ptr(iptr), ptr(b.prunePtr),
                           ptr(b.pruneSet), ptr(b.a2p), ptr(a2i), ptr(a2src), b.nnz))


@pytest.mark.parametrize("make", [lambda: P.dense_spd(90), lambda: P.laplacian3d_var(8, 1), lambda: P.vector3d_var(4, 1)],
                         ids=["dense_90", "lap3d_8", "vec3d_4"])
@pytest.mark.parametrize("order", ["reversed", "shuffled"])
def test_entries_in_any_order_within_a_column(make, order):
    prob = make()
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    f = S.Factor(b)
    assert f.factor(prob.values) == 0
    L = f.L_values()
    rng = np.random.default_rng(1)
    a2i, a2src = b.a2i.copy(), b.a2src.copy()
    for j in range(b.n):
        e = np.arange(b.a2p[j], b.a2p[j + 1])
        to = e[::-1] if order == "reversed" else rng.permutation(e)
        a2i[e], a2src[e] = b.a2i[to], b.a2src[to]
    _upload(f, b, a2i, a2src)
    assert f.factor(prob.values) == 0
    assert np.array_equal(f.L_values(), L)


def test_entries_outside_the_structure_are_refused():
    prob = P.laplacian3d_var(8, 1)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    f = S.Factor(b)
    j = int(b.super[0])
    rows = set(b.s[b.pi[0]:b.pi[1]].tolist())
    outside = next(i for i in range(b.n - 1, 0, -1) if i not in rows)
    for q, row in ((b.a2p[j + 1] - 1, outside), (b.a2p[j + 1] - 1, b.n), (b.a2p[b.n // 2], 0)):
        a2i = b.a2i.copy()
        a2i[q] = row
        with pytest.raises(SwcError, match="outside the structure"):
            _upload(f, b, a2i, b.a2src)
    _upload(f, b, b.a2i, b.a2src)
    assert f.factor(prob.values) == 0
