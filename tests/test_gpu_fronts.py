"""GPU: the multifrontal factorization at the edges of its tiles and fronts, and the
left-looking path that stays behind it, against the CPU oracle."""
import os

import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
import oracle_py as O
from helpers import relF, setup

pytestmark = pytest.mark.gpu


def arrow(nleaf, leaf, ncore, seed=1):
    """nleaf dense blocks of `leaf` unknowns, each coupled to all of a dense core ordered
    last: the core's supernode, which takes in the last block, has one child for every other
    block."""
    rng = np.random.default_rng(seed)
    n = nleaf * leaf + ncore
    A = np.zeros((n, n))
    core = np.arange(n - ncore, n)
    for k in range(nleaf):
        i = np.arange(k * leaf, (k + 1) * leaf)
        A[np.ix_(i, i)] = rng.uniform(-1, 1, (leaf, leaf))
        A[np.ix_(core, i)] = rng.uniform(-1, 1, (ncore, leaf))
    A[np.ix_(core, core)] = rng.uniform(-1, 1, (ncore, ncore))
    A = np.tril(A) + np.tril(A, -1).T
    A[np.diag_indices(n)] = np.abs(A).sum(axis=1) + 1.0
    r, c = np.nonzero(np.tril(A))
    return P.Problem(n, *P.lower_csc_from_coo(n, r, c, A[r, c]), np.arange(n), f"arrow_{nleaf}_{leaf}_{ncore}")


# rows of the children's fronts around one tile (64), small fronts' widths around 16 and
# rows below around 48, parents of one, two and more panels; 70 and 130 children pass the
# 64 descriptors one load brings
EDGES = [(3, 16, 47), (3, 16, 48), (3, 16, 49), (2, 15, 20), (2, 17, 46), (2, 17, 47), (2, 17, 48),
         (3, 33, 31), (3, 64, 64), (2, 65, 63), (2, 70, 130), (70, 6, 24), (130, 6, 70), (4, 100, 17)]


@pytest.mark.parametrize("nleaf,leaf,ncore", EDGES)
def test_front_edges_match_oracle(nleaf, leaf, ncore):
    prob = arrow(nleaf, leaf, ncore)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm, nrelax=(0, 0, 0), zrelax=(0.0, 0.0, 0.0))
    plan = api.build_fronts(b)
    if nleaf > 64:
        n = [int(t["dg1"] - t["dg0"]) for t in plan["ftiles"]] + [int(f["g1"] - f["g0"]) for f in plan["small"]]
        assert max(n) == nleaf - 1
    a2x = b.a2_values(prob.values)
    Lo, info = O.factor(b, a2x)
    assert info == 0
    L32, _ = O.factor(b, a2x, fp32_updates=True)
    f = S.Factor(b)
    for mode in (0, 1, 2):
        f.set_precision(mode)
        for rep in range(2):  # captured, then replayed
            assert f.factor(prob.values) == 0
            L = f.L_values()
            if mode == 0:
                assert relF(L, Lo) < 1e-12
            else:
                assert relF(L, L32) < 10 * max(relF(L32, Lo), 1e-7)


@pytest.mark.parametrize("rlb", [1, 2, 8])
@pytest.mark.parametrize("make", [lambda: P.dense_spd(200), lambda: P.vector3d_var(9)], ids=["dense_200", "vec3d_9"])
def test_right_looking_blocks_match_oracle(make, rlb):
    prob = make()
    b, a2x, Lo, _ = setup(prob)
    f = S.Factor(b, params=(rlb,))
    assert f.factor(prob.values) == 0
    assert relF(f.L_values(), Lo) < 1e-12


@pytest.mark.parametrize("fuse", [0, 1])
@pytest.mark.parametrize("mode", [0, 1])
def test_left_looking_narrow_kernels(fuse, mode):
    """The H-level schedule keeps the left-looking path: its one-wave kernels, forced by a
    one-tile threshold, give the oracle's factor."""
    g = np.load(os.path.join(os.path.dirname(__file__), "golden", "c1_lap2d_const_100.npz"))
    prob = P.laplacian2d_const(100)
    b, a2x, Lo, _ = setup(prob)
    f = S.Factor(b, params=(8, 128, 1, 256, fuse), schedule=(g["levelptr"], g["parptr"], g["partition"]))
    f.set_precision(mode)
    assert f.factor(prob.values) == 0
    if mode == 0:
        assert relF(f.L_values(), Lo) <= 1e-12
    else:
        L32, _ = O.factor(b, a2x, fp32_updates=True)
        assert relF(f.L_values(), L32) < 10 * max(relF(L32, Lo), 1e-7)


@pytest.mark.parametrize("make", [lambda: P.dense_spd(600, seed=2), lambda: P.dense_spd(641, seed=2),
                                  lambda: P.laplacian3d_var(13, shift=1.0), lambda: P.vector3d_var(11)],
                         ids=["dense_600", "dense_641", "lap3d_13", "vec3d_11"])
@pytest.mark.parametrize("mode", [0, 2])
def test_updates_of_many_columns_match_dense_cholesky(make, mode):
    """Supernodes of 128 columns and more (operands by way of LDS), remainders in every
    dimension; FP64 updates, and FP32 ones whose products carry 2^-24 each."""
    prob = make()
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    assert np.diff(b.super).max() >= 128
    f = S.Factor(b)
    f.set_precision(mode)
    assert f.factor(prob.values) == 0
    Ap = prob.scipy_full().toarray()[np.ix_(b.Perm, b.Perm)]
    L = f.L_values()
    ref = np.linalg.cholesky(Ap)
    err = 0.0
    for s in range(b.nsuper):
        c0, c1 = b.super[s], b.super[s + 1]
        rows = b.s[b.pi[s]:b.pi[s + 1]]
        blk = L[b.p[c0]:b.p[c0] + len(rows) * (c1 - c0)].reshape(c1 - c0, len(rows)).T
        low = rows[:, None] >= np.arange(c0, c1)[None, :]
        err = max(err, np.abs(np.where(low, blk - ref[np.ix_(rows, np.arange(c0, c1))], 0.0)).max())
    eps = np.finfo(float).eps if mode == 0 else 2.0 ** -24
    # backward error n eps |A| at most, and cond(A) between it and L
    assert err <= 10 * np.sqrt(prob.n) * eps * np.linalg.cond(Ap) * np.abs(ref).max()
