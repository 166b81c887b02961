"""The DD projector as a differentiable torch operator.

``DDProjectorFunction`` computes y = A x with the HIP forward projector; its backward is the
hand-written matched backprojector A^T (``ctr_dd_backproject`` in adjoint mode,
``ctr_dd_adjoint_batch`` for a batch), so gradients of any loss of A x flow through the project's
own kernels.  ``DDBackprojectorFunction`` is the transpose pair (y -> A^T y, backward A).  Both
accept one volume [nz, ny, nx] or a batch [B, nz, ny, nx] (projections [nView, nv, nu] or
[B, nView, nv, nu]); the items of a batch share launches on the current stream.
"""
from __future__ import annotations

import torch

from . import projector as P
from .geometry import ScanGeometry


def _apply(one, many, x: torch.Tensor, item_shape, geom: ScanGeometry) -> torch.Tensor:
    x = x.contiguous()
    if tuple(x.shape) == tuple(item_shape):
        return one(x, geom)
    if x.dim() == 4 and tuple(x.shape[1:]) == tuple(item_shape):
        return many(x, geom)
    raise ValueError(f"expected shape {tuple(item_shape)} or [B, *{tuple(item_shape)}], got {tuple(x.shape)}")


def forward_batch(vol: torch.Tensor, geom: ScanGeometry) -> torch.Tensor:
    """A x of one volume or of every volume of a batch."""
    return _apply(P.dd_forward, P.dd_forward_batch, vol, geom.vol_shape, geom)


def adjoint_batch(proj: torch.Tensor, geom: ScanGeometry) -> torch.Tensor:
    """A^T y of one scan or of every scan of a batch."""
    return _apply(P.dd_adjoint, P.dd_adjoint_batch, proj, geom.proj_shape, geom)


class DDProjectorFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, vol, geom):
        ctx.geom = geom
        return forward_batch(vol.detach().to(torch.float32), geom)

    @staticmethod
    def backward(ctx, grad):
        return adjoint_batch(grad.to(torch.float32), ctx.geom), None


class DDBackprojectorFunction(torch.autograd.Function):
    @staticmethod
    def forward(ctx, proj, geom):
        ctx.geom = geom
        return adjoint_batch(proj.detach().to(torch.float32), geom)

    @staticmethod
    def backward(ctx, grad):
        return forward_batch(grad.to(torch.float32), ctx.geom), None


class DDProjector(torch.nn.Module):
    """``y = A x`` as a module; ``.T(y)`` is the matched backprojector ``A^T y``."""

    def __init__(self, geom: ScanGeometry | dict):
        super().__init__()
        self.geom = geom if isinstance(geom, ScanGeometry) else ScanGeometry(geom)
        self.geom.check_supported()

    def forward(self, vol: torch.Tensor) -> torch.Tensor:
        return DDProjectorFunction.apply(vol, self.geom)

    def T(self, proj: torch.Tensor) -> torch.Tensor:
        return DDBackprojectorFunction.apply(proj, self.geom)
