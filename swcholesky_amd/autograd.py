"""torch.autograd wrappers of the GPU factorization (thin: the work is in the C ABI).

``logdet_quad(values, b, factor)`` returns logdet(A) + b^T A^{-1} b for the SPD
matrix whose stored lower-triangle values (input order of the analysed pattern)
are ``values``; its backward gives d/dvalues through the supernodal selected
inverse (swc_gradient) and d/db = 2 A^{-1} b.  Each stored off-diagonal value
a_ij stands for both a_ij and a_ji, so its gradient counts both.
"""
from __future__ import annotations

import torch

from .api import Factor


def _sync(*tensors):
    """Waits until the tensors hold their values: the factor works on a stream of its own, and
    a tensor's work is on its own device's stream, whichever device is current (a host
    tensor's, say a copy under way, on the current one's)."""
    if torch.cuda.is_available():
        for device in {t.device if t.is_cuda else None for t in tensors}:
            torch.cuda.current_stream(device).synchronize()


class _LogdetQuad(torch.autograd.Function):
    @staticmethod
    def forward(ctx, values, b, factor: Factor, alpha: float, beta: float):
        vals = values.detach().to(torch.float64).contiguous()
        rhs = b.detach().to(torch.float64).contiguous()
        dev = vals.device
        _sync(vals, rhs)
        info = factor.factor(vals if vals.is_cuda else vals.numpy())
        if info:
            raise RuntimeError(f"matrix is not positive definite (column {info - 1})")
        if rhs.is_cuda and rhs.device == dev and rhs.shape == (factor.n,):
            # solved where it is: the vectors do not travel to the host and back
            x = rhs.clone()
            _sync(x)
            quad = float(torch.dot(rhs, factor.solve_device(x)))
        else:
            x = torch.from_numpy(factor.solve(rhs.cpu().numpy())).to(dev)
            quad = float(torch.dot(rhs.cpu(), x.cpu()))
        out = alpha * factor.logdet() + beta * quad
        ctx.factor, ctx.alpha, ctx.beta = factor, alpha, beta
        ctx.save_for_backward(x)
        return torch.tensor(out, dtype=torch.float64, device=dev)

    @staticmethod
    def backward(ctx, g):
        (x,) = ctx.saved_tensors
        f = ctx.factor
        if x.is_cuda:
            gv = torch.empty(f.bcsc.nnz, dtype=torch.float64, device=x.device)
            _sync(x)  # what used gv's memory before has run too
            f.gradient(x, alpha=ctx.alpha, beta=ctx.beta, out=gv)
        else:
            _sync(x)
            gv = torch.from_numpy(f.gradient(x.numpy(), alpha=ctx.alpha, beta=ctx.beta))
        return g * gv, g * 2.0 * ctx.beta * x, None, None, None


def logdet_quad(values, b, factor: Factor, alpha=1.0, beta=1.0):
    """alpha logdet(A) + beta b^T A^{-1} b, differentiable in values and b."""
    return _LogdetQuad.apply(values, b, factor, float(alpha), float(beta))
