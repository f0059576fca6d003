"""The forward model's ray kernels (optk_scene_rays) against the same
expressions in numpy: coordinates bit for bit, fluxes against the solid
angles in extended precision.

The solid angle's triple product is formed of the differences of unit
vectors, each within 2 ulp (4e-16): relative to a cell of side d that is an
error of a few 1e-16 / d, squared differences included, 1e-11 for the
smallest cell here (0.001 deg = 1.7e-5 rad); 1e-10 leaves a factor of ten."""

import numpy as np
import pytest
import torch

from optika_amd import _scene, workloads
from optika_amd.pupil import solid_angle_cells
from optika_amd.vectors import Cartesian2dVectorArray

pytestmark = pytest.mark.gpu


def _solid(ax, ay):
    """solid_angle_cells in extended precision."""
    ax, ay = np.deg2rad(np.asarray(ax, np.longdouble)), np.deg2rad(np.asarray(ay, np.longdouble))
    x, y = ax[..., :, None], ay[..., None, :]
    x, y = np.broadcast_arrays(x, y)
    d = np.stack([-np.cos(y) * np.sin(x), -np.sin(y), np.cos(y) * np.cos(x)], axis=-1)

    def tri(a, b, c):
        den = 1 + (a * b).sum(-1) + (b * c).sum(-1) + (c * a).sum(-1)
        return 2 * np.arctan2((a * np.cross(b - a, c - a)).sum(-1), den)

    v00, v10, v11, v01 = d[..., :-1, :-1, :], d[..., 1:, :-1, :], d[..., 1:, 1:, :], d[..., :-1, 1:, :]
    return np.abs(tri(v00, v10, v11) + tri(v00, v11, v01))


@pytest.mark.parametrize("field_is_angle", [True, False])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1, 1), (2, 3, 5, 1, 2), (3, 17, 1, 2, 3), (1, 40, 33, 3, 1)])
def test_scene_rays_against_numpy(shape, field_is_angle):
    print(f"case: scene rays {shape} {field_is_angle}", flush=True)
    W, X, Y, PX, PY = shape
    rng = np.random.default_rng(5)
    wv = np.sort(rng.uniform(400.0, 700.0, W + 1))[::-1].copy()  # descending vertices count too
    angle = lambda n: np.sort(rng.uniform(-0.02, 0.02, (W + 1, 1)) + 0.001 * np.arange(n + 1)) + 3.0  # noqa: E731
    place = lambda n: np.cumsum(rng.uniform(0.1, 2.0, (W + 1, n + 1)), axis=1) - 4.0  # noqa: E731
    f, p = (angle, place) if field_is_angle else (place, angle)
    axes = [f(X), f(Y), p(PX), p(PY)]
    R = rng.uniform(0.5, 2.0, (W, X, Y))
    u = torch.rand((5,) + shape, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    lam, coords, flux = _scene.rays(wv, axes, R, u, field_is_angle)
    v = u.cpu().numpy()
    np.testing.assert_array_equal(
        lam.cpu().numpy(), (wv[:-1, None, None, None, None]
                            + (wv[1:] - wv[:-1])[:, None, None, None, None] * v[0]).reshape(-1))
    for k, lead in enumerate([(W, X, 1, 1, 1), (W, 1, Y, 1, 1), (W, 1, 1, PX, 1), (W, 1, 1, 1, PY)]):
        a = axes[k]
        lo, hi = a[:-1, :-1].reshape(lead), a[:-1, 1:].reshape(lead)
        lo2, hi2 = a[1:, :-1].reshape(lead), a[1:, 1:].reshape(lead)
        q, r = lo + (lo2 - lo) * v[0], hi + (hi2 - hi) * v[0]
        np.testing.assert_array_equal(coords[k].cpu().numpy(), (q + (r - q) * v[k + 1]).reshape(-1))
    area = lambda x, y: np.abs(np.diff(x)[..., :, None] * np.diff(y)[..., None, :])  # noqa: E731
    mf, mp = (_solid, area) if field_is_angle else (area, _solid)
    mf, mp = mf(axes[0], axes[1]), mp(axes[2], axes[3])
    mf, mp = (mf[:-1] + mf[1:]) / 2, (mp[:-1] + mp[1:]) / 2
    want = (R * np.abs(np.diff(wv))[:, None, None] * mf)[:, :, :, None, None] * mp[:, None, None]
    np.testing.assert_allclose(flux.cpu().numpy(), want.reshape(-1).astype(float), rtol=1e-10)
    # the host's solid angles are the same measure
    np.testing.assert_allclose(solid_angle_cells(axes[0 if field_is_angle else 2], axes[1 if field_is_angle else 3]),
                               _solid(axes[0 if field_is_angle else 2], axes[1 if field_is_angle else 3]).astype(float),
                               rtol=1e-5)


def test_image_takes_a_device_radiance_and_rejects_another_shape():
    system = workloads.stop_newtonian()
    f, w = np.linspace(-0.03, 0.03, 7), np.array([500.0, 520.0, 540.0])
    v = np.linspace(-1, 1, 4)
    R = np.random.default_rng(1).uniform(1e6, 2e6, (2, 6, 6))
    kw = dict(pupil=Cartesian2dVectorArray(v, v), noise=False, seed=4)
    a = system.image(w, f, f, R, **kw)
    b = system.image(w, f, f, torch.as_tensor(R, device="cuda"), **kw)
    np.testing.assert_allclose(a.cpu().numpy(), b.cpu().numpy(), rtol=1e-12)
    with pytest.raises(ValueError):
        system.image(w, f, f, R[:1], **kw)
