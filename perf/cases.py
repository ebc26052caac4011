"""Cases for measuring the numeric phase through its public entry points.

A case names an operator (one of the generators of ``swcholesky_amd.problems``),
its size, and what a program does with it:

* ``solve``: new values for a kept structure are factored and one or more
  right-hand sides solved (the loop of an implicit time step or a Newton
  iteration); ``where`` says whether values and vectors are host arrays or
  device tensors, ``mode`` the precision of the factorization (0 FP64, 1 and 2
  FP32 updates, both refined to a backward error of 1e-12 in FP64);
* ``reuse``: a kept factor solves new right-hand sides (a preconditioner, many
  load cases);
* ``batch``: many independent 2D instances factored and solved together;
* ``adjoint``: logdet(A) + b^T A^{-1} b and its gradients, forward and backward;
* ``oneshot``: the reference's own entry point, host arrays in and L out.

Right-hand sides are A x of uniform x, as in the benchmark.
"""
import math

import numpy as np
import torch

import swcholesky_amd as S
from swcholesky_amd import problems as P
from swcholesky_amd.autograd import logdet_quad
from swcholesky_amd.batch import Batch

TOL = 1e-12
SIDE_MAX = {"lap2d": 320, "gmrf2d": 320, "lap3d": 64, "vec3d": 40, "mesh2d": 24000, "dense": 2600}
SIDE_MIN = {"lap2d": 12, "gmrf2d": 12, "lap3d": 6, "vec3d": 4, "mesh2d": 300, "dense": 40}


def listed():
    return [
        # the smallest call: a small 3D operator, host arrays in and out, latency alone
        dict(name="solve_lap3d_12_host", what="solve", op="lap3d", size=12, nrhs=1, mode=0, where="host"),
        # an ordinary 2D operator (n = 10,000) refactored and solved on the device
        dict(name="solve_lap2d_100", what="solve", op="lap2d", size=100, nrhs=1, mode=0, where="device"),
        # an unstructured mesh with the library's own ordering
        dict(name="solve_mesh2d_20000", what="solve", op="mesh2d", size=20000, nrhs=1, mode=0, where="device"),
        # one wide supernode of an odd number of columns, several right-hand sides
        dict(name="solve_dense_1100_rhs3", what="solve", op="dense", size=1100, nrhs=3, mode=0, where="device"),
        # an ordinary 3D operator in mixed precision, refined, several right-hand sides
        dict(name="solve_lap3d_32_mixed_rhs8", what="solve", op="lap3d", size=32, nrhs=8, mode=1, where="device"),
        # the benchmark's operator: time to solution in FP64
        dict(name="solve_lap3d_64", what="solve", op="lap3d", size=64, nrhs=1, mode=0, where="device"),
        # the largest: the vector operator with every update in FP32, refined
        dict(name="solve_vec3d_48_mixed", what="solve", op="vec3d", size=48, nrhs=1, mode=2, where="device"),
        # one right-hand side after another on the benchmark operator's factor
        dict(name="reuse_lap3d_64_rhs1", what="reuse", op="lap3d", size=64, nrhs=1),
        # a block of right-hand sides on the vector operator's factor
        dict(name="reuse_vec3d_48_rhs32", what="reuse", op="vec3d", size=48, nrhs=32),
        # independent instances of uneven sizes in one launch sequence
        dict(name="batch_256", what="batch", count=256, lo=16, hi=128),
        # the gradient of a Gaussian Markov random field's likelihood
        dict(name="adjoint_gmrf2d_256", what="adjoint", op="gmrf2d", size=256),
        # the reference's call with nothing kept: plan, factor and copy of L out
        dict(name="oneshot_lap2d_100", what="oneshot", op="lap2d", size=100),
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["solve", "solve", "solve", "solve", "reuse", "reuse", "batch", "adjoint", "adjoint", "oneshot"])
    if what == "batch":
        lo = rng.randint(12, 40)
        return dict(what=what, count=_log_size(rng, 4, 256), lo=lo, hi=rng.randint(lo + 8, 128))
    if what == "adjoint":
        op = rng.choice(["gmrf2d", "gmrf2d", "lap2d", "lap3d"])
        return dict(what=what, op=op, size=_log_size(rng, SIDE_MIN[op], 24 if op == "lap3d" else SIDE_MAX[op]))
    if what == "oneshot":
        op = rng.choice(["lap2d", "lap2d", "lap3d"])
        return dict(what=what, op=op, size=_log_size(rng, SIDE_MIN[op], 20 if op == "lap3d" else 110))
    op = rng.choice(["lap2d", "lap3d", "lap3d", "lap3d", "vec3d", "gmrf2d", "mesh2d", "dense"])
    c = dict(what=what, op=op, size=_log_size(rng, SIDE_MIN[op], SIDE_MAX[op]), nrhs=rng.choice([1, 1, 1, _log_size(rng, 2, 32)]))
    if what == "solve":
        c |= dict(mode=rng.choice([0, 0, 0, 1, 2]), where=rng.choice(["device", "device", "device", "host"]))
    return c


def _problem(case, seed):
    op, size = case["op"], case["size"]
    if op == "lap2d":
        return P.laplacian2d_var(size, seed)
    if op == "lap3d":
        # shift 1e-2: an implicit step's operator, well enough conditioned for
        # solutions that are refined to TOL to be compared
        return P.laplacian3d_var(size, seed, shift=1e-2)
    if op == "vec3d":
        return P.vector3d_var(size, seed, shift=1e-2)
    if op == "gmrf2d":
        return P.gmrf2d(size, seed)
    if op == "mesh2d":
        return P.mesh2d_random(size, seed)
    return P.dense_spd(size, seed)


def _rhs(prob, nrhs, seed):
    """n x nrhs right-hand sides A x of uniform x in [-1, 1)."""
    x = np.random.default_rng(seed + 101).uniform(-1, 1, (prob.n, nrhs))
    return np.asfortranarray(prob.scipy_full() @ x)


def _instances(case, seed):
    rng = np.random.default_rng(seed)
    sides = np.random.default_rng(3).integers(case["lo"], case["hi"] + 1, size=case["count"])
    return [P.laplacian2d_var(int(s), seed=None, rng=rng) for s in sides]


def _analysis(prob):
    return S.analyze_p2(prob.n, prob.colptr, prob.rowidx, prob.perm)


def _on_device(b):
    """Host columns (n x nrhs) as the device tensor the solves take: (nrhs, n), or (n,)."""
    t = torch.from_numpy(np.ascontiguousarray(b.T)).cuda()
    return t[0] if t.shape[0] == 1 else t


def prepare(case, seed):
    what = case["what"]
    if what == "batch":
        probs = _instances(case, seed)
        bt = Batch(probs)
        f = bt.factor
        rhs = np.concatenate([_rhs(p, 1, seed + k) for k, p in enumerate(probs)])
        return dict(what=what, f=f, values=torch.from_numpy(bt.values(probs)).cuda(), b=_on_device(rhs))
    prob = _problem(case, seed)
    bcsc = _analysis(prob)
    if what == "oneshot":
        return dict(what=what, bcsc=bcsc, a2x=bcsc.a2_values(prob.values), lC=bcsc.p.astype(np.uint64),
                    iptr=bcsc.i_ptr.astype(np.uint64))
    f = S.Factor(bcsc)
    b = _rhs(prob, case.get("nrhs", 1), seed)
    s = dict(what=what, f=f)
    if what == "solve":
        f.set_precision(case["mode"])
        host = case["where"] == "host"
        s |= dict(mode=case["mode"], host=host, values=prob.values if host else torch.from_numpy(prob.values).cuda(),
                  b=(b[:, 0].copy() if case["nrhs"] == 1 else b) if host else _on_device(b))
    elif what == "reuse":
        assert f.factor(prob.values) == 0
        s |= dict(b=_on_device(b))
    else:
        s |= dict(values=torch.from_numpy(prob.values).cuda().requires_grad_(),
                  b=torch.from_numpy(b[:, 0].copy()).cuda().requires_grad_())
    return s


def _copy(b):
    """The right-hand sides in a tensor of their own, complete before the library's stream reads it."""
    x = b.clone()
    torch.cuda.current_stream().synchronize()
    return x


def run(s):
    what = s["what"]
    if what == "oneshot":
        b = s["bcsc"]
        L = np.zeros(b.xsize)
        timing = np.zeros(8)
        ok = S.sw_cholesky_left_par_05(b.n, b.a2p, b.a2i, s["a2x"], s["lC"], b.s, s["iptr"], L, b.super,
                                       b.nsuper, timing, b.prunePtr, b.pruneSet)
        return dict(L=L, ok=ok)
    f = s["f"]
    if what == "adjoint":
        s["values"].grad = s["b"].grad = None
        out = logdet_quad(s["values"], s["b"], f)
        out.backward()
        return dict(value=out.detach(), dvalues=s["values"].grad, db=s["b"].grad)
    if what == "reuse":
        return dict(x=f.solve_device(_copy(s["b"])))
    if what == "batch":
        info = f.factor(s["values"])
        x, _, _ = f.refine(_copy(s["b"]), tol=TOL)
        return dict(x=x, info=info)
    info = f.factor(s["values"])
    if s["mode"]:
        x = f.refine(s["b"] if s["host"] else _copy(s["b"]), tol=TOL)[0]
    elif s["host"]:
        x = f.solve(s["b"])
    else:
        x = f.solve_device(_copy(s["b"]))
    return dict(x=x, info=info)


def work(case):
    """Bytes: the values and vectors, L written by a factorization and read by
    each sweep of a solve.  Flops: sum ColCount^2 for a factorization (twice
    that more for the selected inverse), 4 per entry of L and right-hand side."""
    if case["what"] == "batch":
        probs = _instances(case, 0)
        b = S.api.analyze_batch([(p.n, p.colptr, p.rowidx, p.perm) for p in probs])
    else:
        b = _analysis(_problem(case, 1))
    nnzL = float(b.ColCount.astype(np.int64).sum())
    nrhs = case.get("nrhs", 1)
    factor = {"bytes": 8.0 * (b.nnz + nnzL), "flops": b.flops}
    solve = {"bytes": 16.0 * nnzL + 16.0 * b.n * nrhs, "flops": 4.0 * nnzL * nrhs}
    parts = {"solve": [factor, solve], "batch": [factor, solve], "reuse": [solve], "oneshot": [factor],
             "adjoint": [factor, solve, {"bytes": 8.0 * (2 * nnzL + b.nnz), "flops": 2.0 * b.flops}]}[case["what"]]
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


# ---- the same answers from dense blocks in 64 bits --------------------------

class _Blocks:
    """Block tridiagonal Cholesky of an operator whose unknowns come plane by
    plane (grids: every plane of the first axis; otherwise one dense block)."""

    def __init__(self, prob, device):
        n = prob.n
        planes = prob.shape[0] if prob.shape else 1
        m = self.m = n // planes
        col = np.repeat(np.arange(n, dtype=np.int64), np.diff(prob.colptr))
        row = prob.rowidx.astype(np.int64)
        order = np.argsort(col // m, kind="stable")
        cut = np.searchsorted((col // m)[order], np.arange(planes + 1))
        dev = dict(dtype=torch.float64, device=device)
        self.chol, self.E = [], []
        schur = None
        for p in range(planes):
            e = order[cut[p]:cut[p + 1]]
            r, c, v = (torch.from_numpy(np.ascontiguousarray(a)).to(device)
                       for a in (row[e] - p * m, col[e] - p * m, prob.values[e]))
            here = r < m
            D = torch.zeros(m, m, **dev)
            D[r[here], c[here]] = v[here]
            D = D + torch.tril(D, -1).T
            if schur is not None:
                D -= schur
            C = torch.linalg.cholesky(D)
            self.chol.append(C)
            if p + 1 < planes:
                E = torch.zeros(m, m, **dev)  # rows of the next plane, columns of this one
                E[r[~here] - m, c[~here]] = v[~here]
                G = torch.linalg.solve_triangular(C, E.T.contiguous(), upper=False)
                schur = G.T.contiguous() @ G
                self.E.append(E)

    def solve(self, b):
        b = torch.as_tensor(b, dtype=torch.float64, device=self.chol[0].device).reshape(len(self.chol), self.m, -1)
        y = []
        for p, C in enumerate(self.chol):
            t = b[p] if p == 0 else b[p] - self.E[p - 1] @ torch.cholesky_solve(y[-1], self.chol[p - 1])
            y.append(t)
        x = [torch.cholesky_solve(y[-1], self.chol[-1])]
        for p in range(len(self.chol) - 2, -1, -1):
            x.append(torch.cholesky_solve(y[p] - self.E[p].T @ x[-1], self.chol[p]))
        return torch.cat(x[::-1])

    def logdet(self):
        return sum(2.0 * torch.log(torch.diagonal(C)).sum() for C in self.chol)

    def inverse_at(self, row, col):
        """Entries (row, col), row >= col, of the inverse, within a plane or a plane apart."""
        m, dev = self.m, self.chol[0].device
        row, col = (torch.as_tensor(a, dtype=torch.int64, device=dev) for a in (row, col))
        out = torch.zeros(row.shape, dtype=torch.float64, device=dev)
        Z = None
        for p in range(len(self.chol) - 1, -1, -1):
            inv = torch.cholesky_inverse(self.chol[p])
            if Z is None:
                Z = inv
            else:
                ES = self.E[p] @ inv
                below = -(Z @ ES)  # Z(p + 1, p)
                at = (col // m == p) & (row // m == p + 1)
                out[at] = below[row[at] % m, col[at] % m]
                Z = inv - ES.T @ below
            at = (col // m == p) & (row // m == p)
            out[at] = Z[row[at] % m, col[at] % m]
        return out


def _block_solution(prob, b, device):
    return _Blocks(prob, device).solve(b)


def exact(case, seed):
    what = case["what"]
    if what == "batch":
        probs = _instances(case, seed)
        return dict(x=torch.cat([_block_solution(p, _rhs(p, 1, seed + k), "cpu")[:, 0] for k, p in enumerate(probs)]),
                    info=0)
    prob = _problem(case, seed)
    b = _rhs(prob, case.get("nrhs", 1), seed)
    if what == "oneshot":
        bcsc = _analysis(prob)  # for the ordering and layout of L alone
        A = torch.from_numpy(prob.scipy_full()[bcsc.Perm][:, bcsc.Perm].toarray()).cuda()
        C = torch.linalg.cholesky(A).cpu().numpy()
        L = np.zeros(bcsc.xsize)
        for s in range(bcsc.nsuper):
            c0, c1 = bcsc.super[s], bcsc.super[s + 1]
            rows = bcsc.s[bcsc.i_ptr[c0]:bcsc.i_ptr[c1]]
            L[bcsc.p[c0]:bcsc.p[c0] + rows.size * (c1 - c0)] = np.tril(C[rows, c0:c1]).ravel(order="F")
        return dict(L=L, ok=1)
    blocks = _Blocks(prob, "cuda")
    x = blocks.solve(b)
    if what == "adjoint":
        col = np.repeat(np.arange(prob.n), np.diff(prob.colptr))
        x = x[:, 0]
        w = torch.from_numpy(np.where(prob.rowidx == col, 1.0, 2.0)).cuda()
        r, c = (torch.from_numpy(a.astype(np.int64)).cuda() for a in (prob.rowidx, col))
        dv = w * (blocks.inverse_at(prob.rowidx, col) - x[r] * x[c])
        return dict(value=blocks.logdet() + torch.dot(x, torch.from_numpy(b[:, 0].copy()).cuda()), dvalues=dv, db=2.0 * x)
    if case.get("where") == "host":
        x = x.cpu().numpy()
        return dict(x=x[:, 0].copy() if case["nrhs"] == 1 else x, info=0)
    x = x.T.contiguous()
    x = x[0] if x.shape[0] == 1 else x
    return dict(x=x) if what == "reuse" else dict(x=x, info=0)
