"""The multifrontal plan and its kernels' index arithmetic, emulated on the CPU."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
import oracle_py as O
from helpers import relF, setup


def _bits(mask):
    return np.array([i for i in range(64) if (int(mask) >> i) & 1], dtype=np.int64)


class _Emulation:
    """F and U launches on one array holding L and the arena.  Entries nobody has written
    are NaN, so a tile that reads a child before it is formed, after its room is used
    again, or outside its lower triangle shows up in L."""

    def __init__(self, bcsc, plan, vals, rng):
        self.b, self.p, self.vals, self.rng = bcsc, plan, vals, rng
        self.X = np.full(bcsc.xsize + plan["usize"], np.nan)
        self.X[:bcsc.xsize] = 0.0
        self.scratch = {}
        self.info = 0

    def idx(self, base, ld, nr, nc):
        i = base + np.arange(nc)[None, :] * ld + np.arange(nr)[:, None]
        assert nr <= 0 or nc <= 0 or (i.min() >= 0 and i.max() < len(self.X)), "outside the buffer"
        return i

    def assemble(self, g0, g1, a0, a1, nr, nc, diag):
        """The children's and A's part of a tile (rows nr, columns nc)."""
        t = np.zeros((64, 64))
        low = np.arange(64)[:, None] >= np.arange(64)[None, :]
        for g in self.p["gathers"][g0:g1]:
            r, c = _bits(g["rmask"]), _bits(g["cmask"])
            v = self.X[self.idx(int(g["src"]), int(g["ld"]), len(r), len(c))].copy()
            if diag:
                v[~low[np.ix_(r, c)]] = 0.0
            t[np.ix_(r, c)] += v
        for e in self.p["aents"][a0:a1]:
            t[e["pos"] & 63, e["pos"] >> 6] += self.vals[e["q"]]
        assert not t[nr:].any() and not t[:, nc:].any(), "landing outside the tile"
        return t[:nr, :nc]

    def potrf(self, a, c0):
        l = np.zeros_like(a)
        for j in range(len(a)):
            l[j, j] = np.sqrt(a[j, j])
            l[j + 1:, j] = a[j + 1:, j] / l[j, j]
            for c in range(j + 1, len(a)):
                a[c:, c] -= l[c:, j] * l[c, j]
        return l

    def small(self, f):
        R, w, m = int(f["R"]), int(f["w"]), int(f["R"] - f["w"])
        assert R <= 64 and w <= 16
        full = np.zeros((R, R))
        low = np.tril(np.ones((R, R), bool))
        for g in self.p["gathers"][f["g0"]:f["g1"]]:
            assert g["rmask"] == g["cmask"]
            r = _bits(g["rmask"])
            assert r.max() < R
            v = self.X[self.idx(int(g["src"]), int(g["ld"]), len(r), len(r))].copy()
            v[np.triu_indices(len(r), 1)] = 0.0
            full[np.ix_(r, r)] += v
        for e in self.p["aents"][f["a0"]:f["a1"]]:
            assert (e["pos"] >> 6) < w and (e["pos"] & 63) < R
            full[e["pos"] & 63, e["pos"] >> 6] += self.vals[e["q"]]
        l11 = self.potrf(np.tril(full[:w, :w]), int(f["c0"]))
        l21 = np.linalg.solve(l11, full[w:, :w].T).T
        keep = low[:, :w]
        self.X[self.idx(int(f["vbase"]), R, R, w)[keep]] = np.vstack([l11, l21])[keep]
        if m:
            u = full[w:, w:] - l21 @ l21.T
            keep = np.tril(np.ones((m, m), bool))
            self.X[self.idx(int(f["ubase"]), int(f["ldu"]), m, m)[keep]] = u[keep]

    def factor_tile(self, t):
        nc, nr, ld = int(t["ncol"]), int(t["nr"]), int(t["ld"])
        base = int(t["vbase"]) + int(t["r0"])
        first = nc if t["kind"] == 0 else 0
        if t["first"]:
            d = self.assemble(t["dg0"], t["dg1"], t["da0"], t["da1"], 64, nc, True)
            a11 = np.tril(d[:nc])
            rows = d[nc:nr] if t["kind"] == 0 else self.assemble(
                t["g0"], t["g1"], t["a0"], t["a1"], nr, nc, False)
        else:
            owner, a11 = self.scratch[int(t["slot"])]
            assert owner == int(t["vbase"])
            rows = self.X[self.idx(base + first, ld, nr - first, nc)]
        l11 = self.potrf(a11.copy(), int(t["c0"]))
        out = []
        if t["kind"] == 0:
            keep = np.tril(np.ones((nc, nc), bool))
            out.append((self.idx(base, ld, nc, nc)[keep], l11[keep]))
        out.append((self.idx(base + first, ld, nr - first, nc), np.linalg.solve(l11, rows.T).T))
        return out

    def update_tile(self, u):
        nr, nc, k = int(u["nr"]), int(u["nc"]), int(u["k"])
        at = self.idx(int(u["vbase"]), int(u["ld"]), nr, nc)
        keep = np.arange(nr)[:, None] >= np.arange(nc)[None, :] if u["diag"] else np.ones((nr, nc), bool)
        cur = self.assemble(u["g0"], u["g1"], u["a0"], u["a1"], nr, nc, bool(u["diag"])) \
            if u["first"] else self.X[at].copy()
        A = self.X[self.idx(int(u["asrc"]), int(u["sld"]), nr, k)]
        B = self.X[self.idx(int(u["bsrc"]), int(u["sld"]), nc, k)]
        cur = cur - A @ B.T
        if u["slot"] >= 0:
            assert u["slot"] + nc * nc <= self.p["diag_scratch"]
            self.scratch[int(u["slot"])] = (int(u["vbase"]), np.tril(cur[:nc, :nc]))
        self.X[at[keep]] = cur[keep]

    def run(self):
        p = self.p
        for l in range(p["nlevel"]):
            f = p["ftiles"][p["lvl_f"][l]:p["lvl_f"][l + 1]]
            assert np.all(f["ncol"][:p["lvl_fn"][l]] <= 16) and np.all(f["ncol"][p["lvl_fn"][l]:] > 16)
            # one launch: every factor tile reads before any other's stores are relied on,
            # and the tiles deferred from the level before run at any point of it
            outs = []
            for t in self.rng.permutation(len(f)):
                outs += self.factor_tile(f[t])
            d = p["lvl_ud"][l - 1] if l else 0
            if self.rng.integers(2):
                for at, v in outs:
                    self.X[at] = v
                outs = []
            for q in range(p["lvl_u"][l] - d, p["lvl_u"][l]):
                self.update_tile(p["utiles"][q])
            for at, v in outs:
                self.X[at] = v
            for s in p["small"][p["lvl_small"][l]:p["lvl_small"][l + 1]]:
                self.small(s)
            ut = p["utiles"][p["lvl_u"][l]:p["lvl_u"][l + 1] - p["lvl_ud"][l]]
            for q in self.rng.permutation(len(ut)):
                self.update_tile(ut[q])
        return self.X[:self.b.xsize]


CASES = [("lap2d_37", lambda: P.laplacian2d_var(37, 3), 8), ("lap3d_12", lambda: P.laplacian3d_var(12), 8),
         ("vec3d_6", lambda: P.vector3d_var(6), 2), ("lap3d_13_rlb1", lambda: P.laplacian3d_var(13), 1),
         ("dense_300", lambda: P.dense_spd(300), 2), ("dense_1100", lambda: P.dense_spd(1100), 8),
         ("dense_64", lambda: P.dense_spd(64), 8), ("dense_65", lambda: P.dense_spd(65), 8),
         ("dense_17", lambda: P.dense_spd(17), 8), ("dense_3", lambda: P.dense_spd(3), 8),
         ("mesh_1500", lambda: P.mesh2d_random(1500), 8)]


@pytest.mark.parametrize("name,make,rlb", CASES, ids=[c[0] for c in CASES])
def test_emulated_fronts_match_oracle(name, make, rlb):
    """relF < 1e-12 is the factor's parity bar; the emulation rounds like the kernels."""
    prob = make()
    b, a2x, Lo, info = setup(prob)
    assert info == 0
    plan = api.build_fronts(b, rlb)
    L = _Emulation(b, plan, a2x, np.random.default_rng(0)).run()
    assert relF(L, Lo) < 1e-12


def test_every_product_once():
    """Useful products of the plan: per supernode and column of it, the pairs of rows
    below the column's panel are multiplied once; counted against the structure."""
    prob = P.laplacian3d_var(12)
    b, *_ = setup(prob)
    plan = api.build_fronts(b, 2)
    got = 0
    for u in plan["utiles"]:
        nr, nc = int(u["nr"]), int(u["nc"])
        got += (nc * (nc + 1) // 2 + (nr - nc) * nc if u["diag"] else nr * nc) * int(u["k"])
    got += sum(int(f["w"]) * int(f["R"] - f["w"]) * int(f["R"] - f["w"] + 1) // 2 for f in plan["small"])
    want = 0
    for s in range(b.nsuper):
        R, w = int(b.pi[s + 1] - b.pi[s]), int(b.super[s + 1] - b.super[s])
        for p in range(0, w, 64):
            e = min(p + 64, w)
            want += (R - e) * (R - e + 1) // 2 * (e - p)
    assert got == want


def test_structures_without_a_front_tree_are_refused():
    """Descendant sets that are not those of the row lists have no front plan."""
    prob = P.laplacian2d_var(12, 1)
    b, *_ = setup(prob)
    b.pruneSet = b.pruneSet[:-1].copy()
    b.prunePtr = b.prunePtr.copy()
    b.prunePtr[-1] -= 1
    with pytest.raises(S.SwcError, match="front tree"):
        api.build_fronts(b)
