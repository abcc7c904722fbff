"""Mip-Splatting's 3D smoothing filter (metal_gauss/mipfilter.py).

Same two functions, same arguments and results:

* ``compute_3d_filter(means, views, near=0.2, margin=0.15)`` - per-Gaussian
  low-pass size, min seen depth / max focal * sqrt(0.2) (mipfilter.py:29-73).
  Here one HIP kernel pass over all views (mg_compute_3d_filter) instead of a
  torch loop with one projection per view.
* ``apply_3d_filter(scales, opacities, filter_3d)`` - the reparameterisation
  scales' = sqrt(scales^2 + f^2), opacity * sqrt(prod s^2 / prod s'^2)
  (mipfilter.py:76-93), kept as the reference's torch expression for callers
  that want the filtered tensors themselves (a ply export bakes them in).

For training, pass ``filter_3d`` to ``render`` instead: the projection kernel
applies the filter and its adjoint itself, with no extra passes over the
scales and opacities.
"""

from __future__ import annotations

import numpy as np
import torch

from . import _lib


def _host_f64(tensors, rows: int, cols: int) -> np.ndarray:
    """The views' leading (rows, cols) blocks as one float64 host array: one
    stack and one transfer where they share a device and shape, per view
    otherwise."""
    try:
        t = torch.stack(tensors)
    except RuntimeError:
        t = torch.stack([x[:rows, :cols].to("cpu", torch.float64) for x in tensors])
    return t.detach().to("cpu", torch.float64).numpy()[:, :rows, :cols]


def _view_records(views, near: float, margin: float):
    """(V, 20) float32 per-view records and the largest focal length.

    Formed for all views at once in float64: element by element, with a
    transfer per matrix, 100 views took over a millisecond of host time, many
    times the kernels' own."""
    views = list(views)
    if not views:
        return torch.zeros(0, 20), 0.0
    vm = _host_f64([v.viewmat for v in views], 3, 4)
    K = _host_f64([v.K for v in views], 2, 3)
    shapes = [v.image.shape for v in views]
    H = np.array([s[0] for s in shapes], dtype=np.float64)
    W = np.array([s[1] for s in shapes], dtype=np.float64)
    rec = np.empty((len(views), 20))
    rec[:, :9] = vm[:, :, :3].reshape(-1, 9)
    rec[:, 9:12] = vm[:, :, 3]
    rec[:, 12], rec[:, 13], rec[:, 14], rec[:, 15] = K[:, 0, 0], K[:, 1, 1], K[:, 0, 2], K[:, 1, 2]
    rec[:, 16], rec[:, 17] = -margin * W, (1.0 + margin) * W
    rec[:, 18], rec[:, 19] = -margin * H, (1.0 + margin) * H
    return torch.from_numpy(rec.astype(np.float32)), max([0.0, *rec[:, 12:14].ravel().tolist()])


@torch.no_grad()
def compute_3d_filter(means: torch.Tensor, views, near: float = 0.2,
                      margin: float = 0.15) -> torch.Tensor:
    """Per-Gaussian low-pass scale, one value per Gaussian (mipfilter.py:29-73).

    ``views`` need ``.K``, ``.viewmat`` and an ``.image`` for the frame size.
    A Gaussian seen by no camera gets the largest distance any Gaussian got;
    with none seen at all every distance is 1.
    """
    if means.device.type != "cuda":
        raise RuntimeError(
            f"hip backend requires ROCm (cuda) tensors, got device '{means.device}'. "
            "Refusing to silently move data or fall back to another backend.")
    lib = _lib.load()
    means = means.detach().to(torch.float32).contiguous()
    N = means.shape[0]
    rec, focal = _view_records(views, near, margin)
    rec = rec.to(means.device)
    out = torch.empty(N, device=means.device)
    scratch = torch.empty(1, dtype=torch.int32, device=means.device)
    _lib.check(lib.mg_compute_3d_filter(
        N, _lib.dev_tensor(means, "means"), rec.shape[0],
        rec.data_ptr() if rec.numel() else None, float(focal), float(near), out.data_ptr(),
        scratch.data_ptr(), _lib.stream(means)))
    return out


def apply_3d_filter(scales: torch.Tensor, opacities: torch.Tensor,
                    filter_3d: torch.Tensor):
    """Widen the Gaussians and dim them to match (mipfilter.py:76-93).

    Returns (scales, opacities); differentiable in both, with ``filter_3d`` a
    constant.
    """
    f2 = (filter_3d ** 2).unsqueeze(-1)
    s2 = scales ** 2
    s2f = s2 + f2
    coef = torch.sqrt((s2.prod(dim=-1) / s2f.prod(dim=-1)).clamp(0.0, 1.0))
    return torch.sqrt(s2f), opacities * coef
