"""The rays of a scene on the device (optk_scene_rays): one ray per
(wavelength, field, pupil) cell, as ``_rayfunction_from_vertices``
(``optika/systems/_sequential.py:1002-1083``) places and weights them."""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import _lib, _trace

__all__ = ["rays"]


def rays(wavelength, axes, radiance, u, field_is_angle: bool):
    """``wavelength``: [W + 1] vertices (host); ``axes``: field x, field y,
    pupil x, pupil y vertices, each [W + 1][n + 1] (host); ``radiance``:
    W X Y values (host array or tensor); ``u``: uniform weights [5][W][X][Y]
    [PX][PY] (device float64).  Returns (wavelength, [field x, field y, pupil
    x, pupil y], flux), flat device tensors of the rays."""
    dev = u.device
    on_device = isinstance(radiance, torch.Tensor)
    parts = [wavelength, *axes] + ([] if on_device else [radiance])
    # every host array in one copy
    packed = torch.as_tensor(np.concatenate([np.asarray(p, np.float64).reshape(-1) for p in parts])).to(dev)
    starts = np.cumsum([0] + [int(np.size(p)) for p in parts])
    at = lambda k: packed.data_ptr() + 8 * int(starts[k])  # noqa: E731
    keep = None
    if on_device:
        keep = radiance.detach().to(device=dev, dtype=torch.float64).contiguous()
    n = u[0].numel()
    W = len(wavelength) - 1
    cells = [int(a.shape[-1]) - 1 for a in axes]
    out = torch.empty((6, n), dtype=torch.float64, device=dev)
    field = W * cells[0] * cells[1]
    work = torch.empty(field + W * cells[2] * cells[3], dtype=torch.float64, device=dev)
    a = _lib.SceneArgs()
    a.wavelength = at(0)
    a.radiance = keep.data_ptr() if on_device else at(5)
    a.out_wavelength, a.flux = out[4].data_ptr(), out[5].data_ptr()
    for k in range(4):
        a.axis[k] = at(1 + k)
        a.out[k] = out[k].data_ptr()
        a.n[k] = cells[k]
    for k in range(5):
        a.u[k] = u[k].data_ptr()
    a.measure_field, a.measure_pupil = work.data_ptr(), work.data_ptr() + 8 * field
    a.nw = W
    a.field_is_angle = 1 if field_is_angle else 0
    _lib.check(_lib.lib().optk_scene_rays(ctypes.byref(a), _trace.stream_handle()))
    return out[4], [out[0], out[1], out[2], out[3]], out[5]
