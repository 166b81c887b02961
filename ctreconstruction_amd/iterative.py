"""Iterative reconstruction on the DD projector pair: SART and ASD-POCS.

Two backprojectors are available:

* ``"ref"`` — the reference's own loop semantics (python/SART.py:29-59,
  python/ASD_POCS.py:130-202): the FDK-weighted DD backprojector (``backward()``, which scales by
  dtheta and by SAD^2/(SAD - y_c)^2), normalisations ``norm1 = BP(1)`` and ``norm2 = FP(1)``,
  and the reference's placement of eps.
* ``"matched"`` — the update is the gradient of the weighted least-squares data term
  ``0.5 * sum W (A x - p)^2`` with W = 1/(A 1 + eps), taken by torch autograd through
  :class:`DDProjectorFunction`, whose backward applies the matched backprojector A^T to
  W (A x - p); it is scaled by 1/(A^T 1 + eps) (the SART normalisation).

``tv_gradient`` is the normalised total-variation gradient of python/ASD_POCS.py:55-77;
``tv_gradient_autograd`` obtains the same vector by differentiating the TV functional.
All functions accept one volume [nz, ny, nx] (projections [nView, nv, nu]) or a batch.
"""
from __future__ import annotations

import ctypes
import weakref

import torch

from . import _native as N
from . import projector as P
from .autograd import DDProjectorFunction, adjoint_batch, forward_batch
from .geometry import ScanGeometry


def _bp_ref(proj: torch.Tensor, geom: ScanGeometry, mode: str = "ref") -> torch.Tensor:
    """Reference ``backward()``: FDK-weighted DD backprojection times dtheta (no filter)."""
    def one(p, g, out=None):
        return P.dd_backproject(p, g, mode=mode, out=out)
    if proj.dim() == 3:
        return one(proj.contiguous(), geom)
    out = torch.empty((proj.shape[0],) + geom.vol_shape, dtype=torch.float32, device=proj.device)
    for b in range(proj.shape[0]):
        one(proj[b].contiguous(), geom, out=out[b])
    return out


# per geometry object: {(backprojector, device): (contents, A 1, B 1)}, freed with the geometry
_NORM_CACHE: "weakref.WeakKeyDictionary[ScanGeometry, dict]" = weakref.WeakKeyDictionary()


def normalisers(geom: ScanGeometry, backprojector: str, device, eps: float):
    """(row sums A 1, column sums B 1) for the chosen backprojector B; cached per geometry object
    (held weakly: the cache goes when the geometry does) for the scan it describes at the time.

    The sums are finished when they enter the cache (one wait per scan), so that any stream, thread or
    graph capture may read them; each stream that does is noted, so that their memory outlives its
    reads.  Sums worked out inside a graph capture exist only when the graph runs and are not kept."""
    per_geom = _NORM_CACHE.setdefault(geom, {})
    key, contents = (backprojector, str(device)), geom.contents()
    hit = per_geom.get(key)
    if hit is not None and hit[0] == contents:
        stream = torch.cuda.current_stream(device)
        for t in hit[1:]:
            t.record_stream(stream)
        return hit[1:]
    ones_v = torch.ones(geom.vol_shape, device=device)
    ones_p = torch.ones(geom.proj_shape, device=device)
    a1 = P.dd_forward(ones_v, geom)
    if backprojector == "matched":
        b1 = P.dd_adjoint(ones_p, geom)
    elif backprojector == "edge":
        b1 = P.dd_backproject(ones_p, geom, mode="edge")
    else:
        b1 = _bp_ref(ones_p, geom)
    if not torch.cuda.is_current_stream_capturing():
        torch.cuda.current_stream(device).synchronize()
        per_geom[key] = (contents, a1, b1)
    return a1, b1


def sart_reference(proj0: torch.Tensor, geom: ScanGeometry, n_iter: int, alpha: float = 1.0,
                   eps: float = 1e-5, x0: torch.Tensor | None = None, callback=None) -> torch.Tensor:
    """The reference's SART loop (python/SART.py:29-59), including its update
    ``x <- x - alpha * (BP((FP x - p)/(FP 1 + eps)) / BP 1 + eps)`` (eps outside the division)."""
    geom.check_supported()
    a1, b1 = normalisers(geom, "ref", proj0.device, eps)
    shape = (proj0.shape[0],) + geom.vol_shape if proj0.dim() == 4 else geom.vol_shape
    x = torch.zeros(shape, device=proj0.device) if x0 is None else x0.clone()
    for it in range(n_iter):
        resid = (forward_batch(x, geom) - proj0) / (a1 + eps)
        x = x - alpha * (_bp_ref(resid, geom) / b1 + eps)
        if callback is not None:
            callback(it, x)
    return x


def sart(proj0: torch.Tensor, geom: ScanGeometry, n_iter: int, relaxation: float = 0.5,
         x0: torch.Tensor | None = None, nonneg: bool = False, eps: float = 1e-6,
         backprojector: str = "matched", callback=None) -> torch.Tensor:
    """SART with relaxation lambda: x <- x + lambda * B((p - A x) / (A 1 + eps)) / (B 1 + eps).

    With ``backprojector="matched"`` the step direction comes from torch autograd of the
    weighted data term (the backward pass runs the matched backprojector A^T); with ``"ref"``
    B is the reference's FDK-weighted backprojector.
    """
    geom.check_supported()
    a1, b1 = normalisers(geom, backprojector, proj0.device, eps)
    # rays that miss the volume carry no information (their measured value is noise); they are
    # left out as in python/ASD_POCS.py:175, instead of being amplified by 1 / eps
    w = torch.where(a1 > 0, 1.0 / (a1 + eps), torch.zeros_like(a1))
    x = (torch.zeros((proj0.shape[0],) + geom.vol_shape if proj0.dim() == 4 else geom.vol_shape,
                     device=proj0.device) if x0 is None else x0.detach().clone())
    for it in range(n_iter):
        if backprojector == "matched":
            # the gradient of 0.5 sum w (A x - p)^2: the projector's backward of w (A x - p)
            xv = x.detach().requires_grad_(True)
            ax = DDProjectorFunction.apply(xv, geom)
            r = _residual(proj0, ax.detach(), w, weighted=True).sum_to_size(ax.shape).to(ax.dtype)
            (grad,) = torch.autograd.grad(ax, xv, r)
            x = _update(x.detach(), grad, b1, -relaxation, eps, False, nonneg)
        else:
            step = _bp_ref((proj0 - forward_batch(x, geom)) * w, geom, "edge" if backprojector == "edge" else "ref")
            x = _update(x.detach(), step, b1, relaxation, eps, False, nonneg)
        if callback is not None:
            callback(it, x)
    return x.detach()


def _backward_differences(x: torch.Tensor):
    """Backward differences along the last three axes, at every voxel that has a predecessor
    along all three (the voxel (i, j, k) of ``x`` with i, j, k >= 1 sits at (i-1, j-1, k-1))."""
    core = x[..., 1:, 1:, 1:]
    return (core - x[..., :-1, 1:, 1:], core - x[..., 1:, :-1, 1:], core - x[..., 1:, 1:, :-1])


def _tv_terms(img: torch.Tensor, eps: float):
    """Gradient of TV(x) = sum_v sqrt(eps + |D x(v)|^2) (D: backward differences) at the interior
    voxels c, before normalisation: the voxel's own term sum_k D_k x(c) / |D x(c)|_eps minus,
    for each axis k, D_k x(c + e_k) / |D x(c + e_k)|_eps from its successor along k.  This is the
    vector of python/ASD_POCS.py:55-72."""
    d = _backward_differences(img)
    norm = torch.sqrt(eps + d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
    own = ((d[0] + d[1] + d[2]) / norm)[..., :-1, :-1, :-1]
    ratio = [dk / norm for dk in d]
    succ = ratio[0][..., 1:, :-1, :-1] + ratio[1][..., :-1, 1:, :-1] + ratio[2][..., :-1, :-1, 1:]
    return own - succ


def _normalise_pad(dtv: torch.Tensor, eps: float) -> torch.Tensor:
    dims = tuple(range(dtv.dim() - 3, dtv.dim()))
    norm = torch.sqrt(torch.sum(dtv ** 2, dim=dims, keepdim=True))
    norm = torch.where(norm.abs() < eps, torch.ones_like(norm), norm)
    return torch.nn.functional.pad(dtv / norm, (1, 1, 1, 1, 1, 1))


def _observed(*tensors: torch.Tensor) -> bool:
    """Whether something maps, differentiates forward, traces or intercepts torch's work on one of ``tensors``,
    which a kernel called by address would pass by.  A default device (``torch.set_default_device``) does not
    count.  torch has no public form for some of these questions: where it cannot answer one, the answer is yes."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing():
        return True
    try:
        modes = torch.overrides._get_current_function_mode_stack()
        if any(type(m).__module__ != "torch.utils._device" for m in modes):
            return True
        if torch.utils._python_dispatch._get_current_dispatch_mode() is not None:
            return True
        if any(map(torch._C._functorch.is_functorch_wrapped_tensor, tensors)):
            return True
        return any(torch.autograd.forward_ad.unpack_dual(t).tangent is not None for t in tensors)
    except (AttributeError, ImportError):
        return True


def _plain(*tensors: torch.Tensor) -> bool:
    """Whether a kernel may take ``tensors``: contiguous float32 batches of volumes (or projections) on the
    current GPU that nothing differentiates or observes (the torch expressions serve everything else,
    other GPUs among it: a default stream's handle does not name its device)."""
    gpu = torch.cuda.current_device() if torch.cuda.is_initialized() else None
    for t in tensors:
        if type(t) is not torch.Tensor or not t.is_cuda or t.dtype is not torch.float32 or t.get_device() != gpu:
            return False
        if t.dim() < 3 or not t.is_contiguous() or t.numel() == 0 or t.shape[:-3].numel() > 65535:
            return False
        if t.requires_grad and torch.is_grad_enabled():
            return False
    return not _observed(*tensors)


def _on_tv_kernels(img: torch.Tensor, eps: float) -> bool:
    """Whether the TV kernels take ``img`` and ``eps``: a plain number that is a normal float32 (the
    kernels' reciprocal root flushes smaller ones, which torch computes with)."""
    return (_plain(img) and min(img.shape[-3:]) >= 3 and img.shape[-3:].numel() < 2 ** 31 - 1
            and isinstance(eps, (int, float)) and ctypes.c_float(eps).value >= 2.0 ** -126)


def _elementwise(x: torch.Tensor, y: torch.Tensor, per_geom: torch.Tensor, *scalars) -> bool:
    """Whether the residual and update kernels take (x, y) with ``per_geom`` for every item: no
    broadcasting but that, and plain numbers as scalars."""
    return (all(isinstance(s, (int, float)) for s in scalars) and per_geom.numel() <= 0xffffff00
            and x.shape == y.shape and x.shape[-3:] == per_geom.shape and x.device == y.device == per_geom.device
            and _plain(x, y, per_geom))


def _residual(p, ax, a, weighted: bool, eps: float = 0.0):
    """weighted: a (ax - p); else (p - ax) / (a + eps), 0 where a is 0."""
    if _elementwise(p, ax, a, eps):
        out = torch.empty_like(ax)
        N.check(N.lib().ctr_residual(P._ptr(p), P._ptr(ax), P._ptr(a), P._ptr(out), a.numel(), p.numel() // a.numel(),
                                     int(weighted), float(eps), P._stream(p.device)), "ctr_residual")
        return out
    if weighted:
        return a * (ax - p)
    r = (p - ax) / (a + eps)
    return torch.where(a == 0, torch.zeros_like(r), r)


def _update(x, u, b, relax: float, eps: float, masked: bool, nonneg: bool):
    """x + relax u / (b + eps); masked: u counts as 0 where b is 0; nonneg: clamped at 0."""
    if _elementwise(x, u, b, relax, eps):
        out = torch.empty_like(x)
        N.check(N.lib().ctr_update(P._ptr(x), P._ptr(u), P._ptr(b), P._ptr(out), b.numel(), x.numel() // b.numel(),
                                   float(relax), float(eps), int(masked), int(nonneg), P._stream(x.device)), "ctr_update")
        return out
    if masked:
        u = torch.where(b == 0, torch.zeros_like(u), u)
    x = x + relax * u / (b + eps)
    return torch.clamp_min(x, 0.0) if nonneg else x


def _tv_call(fn, img, out, eps, steps, *args):
    lib = N.lib()
    nz, ny, nx = img.shape[-3:]
    batch = img.shape[:-3].numel()
    nbytes = lib.ctr_tv_workspace_bytes(batch, nx, ny, nz, steps)
    ws = P._workspace(nbytes, img.device)
    ptrs = [P._ptr(t) for t in args]
    tail = (steps,) if ptrs else ()
    N.check(getattr(lib, fn)(P._ptr(img), P._ptr(out), *ptrs, batch, nx, ny, nz, float(eps), *tail, P._ptr(ws), nbytes,
                             P._stream(img.device)), fn)
    return out


def tv_gradient(img: torch.Tensor, eps: float = 1e-7) -> torch.Tensor:
    """Normalised TV gradient with zero border (python/ASD_POCS.py:55-77)."""
    if _on_tv_kernels(img, eps):
        return _tv_call("ctr_tv_gradient", img, torch.empty_like(img), eps, 1)
    return _normalise_pad(_tv_terms(img, eps), eps)


def _tv_descent(x: torch.Tensor, step: torch.Tensor, n_steps: int, eps: float) -> torch.Tensor:
    """``n_steps`` of x <- x - step * tv_gradient(x, eps), one ``step`` per volume."""
    if n_steps > 0 and _on_tv_kernels(x, eps) and step.dtype == torch.float32 and not step.requires_grad:
        flat = step.reshape(-1).expand(x.shape[:-3].numel()).contiguous()
        return _tv_call("ctr_tv_descent", x, torch.empty_like(x), eps, n_steps, flat)
    for _ in range(n_steps):
        x = x - step * tv_gradient(x, eps)
    return x


def tv_gradient_autograd(img: torch.Tensor, eps: float = 1e-7) -> torch.Tensor:
    """The same vector as :func:`tv_gradient`, from autograd of
    TV(x) = sum over voxels v with all backward neighbours of sqrt(eps + |grad_b x(v)|^2),
    restricted to interior voxels and normalised as the reference does."""
    x = img.detach().requires_grad_(True)
    d = _backward_differences(x)
    tv = torch.sqrt(eps + d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
    # the reference's sum covers the interior voxels and their +1 neighbours in one axis
    (grad,) = torch.autograd.grad(tv.sum(), x)
    inner = grad[..., 1:-1, 1:-1, 1:-1]
    return _normalise_pad(inner, eps)


def asd_pocs(proj0: torch.Tensor, geom: ScanGeometry, n_outer: int = 20, na: int = 5, ng: int = 20,
             x0: torch.Tensor | None = None, alpha: float = 0.007, beta: float = 1.0,
             beta_red: float = 0.999, r_max: float = 0.99, alpha_red: float = 0.95, eps: float = 1e-7,
             backprojector: str = "ref", tv: str = "reference", callback=None) -> torch.Tensor:
    """ASD-POCS (python/ASD_POCS.py:130-202): ``na`` non-negative SART steps, then ``ng``
    normalised TV steepest-descent steps of size alpha * |dx_POCS|, with the reference's
    adaptive rules for alpha and beta.  ``tv="autograd"`` takes the TV gradient by autograd.
    ``x0=None`` starts from the FDK reconstruction, as the reference script does.  As in the
    reference, the TV steps are not followed by a non-negativity projection."""
    geom.check_supported()
    a1, b1 = normalisers(geom, "matched" if backprojector == "matched" else "ref", proj0.device, eps)
    bp = (lambda r: adjoint_batch(r, geom)) if backprojector == "matched" else (lambda r: _bp_ref(r, geom))
    if x0 is None:
        # the reference starts from the FDK reconstruction (python/ASD_POCS.py:142-143)
        x = (torch.stack([P.fdk(p.contiguous(), geom) for p in proj0]) if proj0.dim() == 4
             else P.fdk(proj0.contiguous(), geom))
    else:
        x = x0.detach().clone()
    # a batch holds independent reconstructions: distances and alpha are per volume
    dims = tuple(range(x.dim() - 3, x.dim()))
    dist = lambda a, b: torch.sqrt(torch.sum((a - b) ** 2, dim=dims, keepdim=True))  # noqa: E731
    alpha = torch.full_like(x[..., :1, :1, :1], alpha)
    for it in range(n_outer):
        f0 = x.clone()
        for _ in range(na):
            upd = bp(_residual(proj0, forward_batch(x, geom), a1, weighted=False, eps=eps))
            x = _update(x, upd, b1, beta, eps, True, True)
        dp = dist(x, f0)
        dtvg = alpha * dp
        f0 = x.clone()
        if tv == "autograd":
            for _ in range(ng):
                x = x - dtvg * tv_gradient_autograd(x, eps)
        else:
            x = _tv_descent(x, dtvg, ng, eps)
        dg = dist(x, f0)
        alpha = torch.where(dg > r_max * dp, alpha * alpha_red, alpha)
        beta *= beta_red
        if callback is not None:
            callback(it, x)
    return x
