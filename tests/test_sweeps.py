"""The solves' work lists and their kernels' index arithmetic, emulated on the CPU."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
import oracle_py as O
from helpers import relF, setup
from test_fronts import CASES

OWN, BELOW, SMALL = 0, 1, 2


class _Sweeps:
    """Items in list order on vectors whose pending entries are NaN.  Every read of an
    entry must find it there: the list is a topological order of the waits, which is what
    keeps the persistent launch free of deadlock."""

    def __init__(self, b, plan, L):
        self.b, self.p, self.L = b, plan, L
        n = b.n
        self.Y = np.full(n, np.nan)
        self.V = np.full(max(plan["vsize"], 1), np.nan)
        self.P = np.full(max(plan["sweep_psize"], 1), np.nan)

    def block(self, vbase, ld, r0, nr, c0, nc):
        i = vbase + (c0 + np.arange(nc))[None, :] * ld + (r0 + np.arange(nr))[:, None]
        assert i.min() >= 0 and i.max() < self.b.xsize and r0 + nr <= ld
        return self.L[i]

    def got(self, a, at):
        v = a[at]
        assert not np.isnan(v).any(), "an item waits for an entry no earlier item makes"
        return v

    def put(self, a, at, v):
        assert np.isnan(a[at]).all(), "an entry made twice"
        a[at] = v

    def gather(self, c):
        g = self.p["gidx"][self.p["gptr"][c]:self.p["gptr"][c + 1]]
        return self.got(self.V, g).sum()

    def smalls(self, lo, hi, fn):
        for s in self.p["sweep_small"][lo:hi]:
            assert s["w"] <= 16
            fn(s)

    def forward(self, x):
        self.X = x.copy()
        ls = self.p["sweep_lvl_small"]
        for k in range(len(ls) - 1):
            self.smalls(ls[k], ls[k + 1], self.small_fwd)
        for it in self.p["sweep_fwd"]:
            if it["kind"] == SMALL:
                self.smalls(it["first"], it["first"] + it["count"], self.small_fwd)
                continue
            vb, ld, w, c0 = int(it["vbase"]), int(it["ld"]), int(it["w"]), int(it["c0"])
            r0, nr, nq = int(it["row0"]), int(it["nr"]), int(it["nq"])
            ncol = min(64 * nq, w)
            sums = np.zeros(nr)
            if ncol:
                sums = self.block(vb, ld, r0, nr, 0, ncol) @ self.got(self.Y, c0 + np.arange(ncol))
            if it["kind"] == OWN:
                assert r0 == 64 * it["p"] and nq == it["p"]
                cols = c0 + r0 + np.arange(nr)
                t = self.X[cols] - sums - np.array([self.gather(c) for c in cols])
                tri = np.tril(self.block(vb, ld, r0, nr, r0, nr))
                self.put(self.Y, cols, np.linalg.solve(tri, t))
                self.X[cols] = np.nan
            else:
                assert ncol == w
                self.put(self.V, int(it["out"]) + np.arange(nr), sums)

    def small_fwd(self, s):
        R, w, c0 = int(s["R"]), int(s["w"]), int(s["c0"])
        B = self.block(int(s["vbase"]), R, 0, R, 0, w)
        cols = c0 + np.arange(w)
        t = self.X[cols] - np.array([self.gather(c) for c in cols])
        y = np.linalg.solve(np.tril(B[:w]), t)
        self.put(self.Y, cols, y)
        self.X[cols] = np.nan
        if R > w:
            self.put(self.V, int(s["voff"]) + np.arange(R - w), B[w:] @ y)

    def small_bwd(self, s):
        R, w, c0, ro = int(s["R"]), int(s["w"]), int(s["c0"]), int(s["rows_off"])
        B = self.block(int(s["vbase"]), R, 0, R, 0, w)
        t = self.got(self.Y, c0 + np.arange(w)) - B[w:].T @ self.got(self.X, self.b.s[ro + w:ro + R])
        self.put(self.X, c0 + np.arange(w), np.linalg.solve(np.tril(B[:w]).T, t))

    def backward(self):
        for it in self.p["sweep_bwd"]:
            if it["kind"] == SMALL:
                self.smalls(it["first"], it["first"] + it["count"], self.small_bwd)
                continue
            vb, ld, w, c0 = int(it["vbase"]), int(it["ld"]), int(it["w"]), int(it["c0"])
            p, nr, r0, r1 = int(it["p"]), int(it["nr"]), int(it["row0"]), int(it["row1"])
            ro, col0 = int(it["rows_off"]), 64 * int(it["p"])
            assert nr == min(64, w - col0)
            t = np.zeros(nr)
            if r1 > r0:
                t += self.block(vb, ld, r0, r1 - r0, col0, nr).T @ self.got(self.X, self.b.s[ro + r0:ro + r1])
            if it["kind"] == BELOW:
                self.put(self.P, int(it["out"]) + np.arange(nr), t)
                continue
            if col0 + 64 < w:
                q = np.arange(col0 + 64, w)
                t += self.block(vb, ld, col0 + 64, len(q), col0, nr).T @ self.got(self.X, c0 + q)
            for c in range(int(it["nq"])):
                t += self.got(self.P, int(it["out"]) + 64 * c + np.arange(nr))
            y = self.got(self.Y, c0 + col0 + np.arange(nr))
            tri = np.tril(self.block(vb, ld, col0, nr, col0, nr))
            self.put(self.X, c0 + col0 + np.arange(nr), np.linalg.solve(tri.T, y - t))
        ls = self.p["sweep_lvl_small"]
        for k in range(len(ls) - 2, -1, -1):
            self.smalls(ls[k], ls[k + 1], self.small_bwd)
        return self.X


MORE = [("gmrf_100", lambda: P.gmrf2d(100), 8), ("lap3d_20", lambda: P.laplacian3d_var(20), 8),
        # 2048 and more narrow leaves: a leading level gets launches of its own
        ("lap2d_240", lambda: P.laplacian2d_var(240, 2), 8)]


@pytest.mark.parametrize("derive", [False, True])
@pytest.mark.parametrize("name,make,_rlb", CASES + MORE, ids=[c[0] for c in CASES + MORE])
def test_emulated_sweeps_match_oracle(name, make, _rlb, derive):
    prob = make()
    b, a2x, Lo, _ = setup(prob)
    plan = api.build_plan(b, derive_sets=derive)
    assert (len(plan["sweep_lvl_small"]) > 1) == (name == "lap2d_240")
    rhs = np.random.default_rng(1).uniform(-1, 1, b.n)
    sw = _Sweeps(b, plan, Lo)
    sw.forward(rhs)
    assert relF(sw.Y, O.lsolve(b, Lo, rhs.copy())[:, 0]) < 1e-12
    x = sw.backward()
    xo = O.ltsolve(b, Lo, O.lsolve(b, Lo, rhs.copy()))[:, 0]
    assert relF(x, xo) < 1e-8  # forward error of operators of condition up to ~1e8
    assert plan["sweep_psize"] <= 128 * max(1, int(np.diff(plan["lvl_fblk"]).max()))


def test_partials_of_tall_supernodes():
    """A panel over more rows below than one item takes has its sums made in parts."""
    prob = P.laplacian3d_var(24)
    b = S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)
    plan = api.build_plan(b)
    it = plan["sweep_bwd"]
    own = it[(it["kind"] == OWN) & (it["nq"] > 0)]
    assert len(own) > 0 and (it["kind"] == BELOW).sum() == own["nq"].sum()
    L = np.random.default_rng(0).uniform(-1e-3, 1e-3, b.xsize)
    for s in range(b.nsuper):
        R = int(b.pi[s + 1] - b.pi[s])
        w = int(b.super[s + 1] - b.super[s])
        L[b.p[b.super[s]] + np.arange(w) * (R + 1)] = 1.0
    rhs = np.random.default_rng(1).uniform(-1, 1, b.n)
    sw = _Sweeps(b, plan, L)
    sw.forward(rhs)
    x = sw.backward()
    xo = O.ltsolve(b, L, O.lsolve(b, L, rhs.copy()))[:, 0]
    assert relF(x, xo) < 1e-11
