"""The work that is timed, as data: cases over the framework's public entry points.

A case is a dict of plain values.  ``prepare`` makes what a user's program has
in hand before the call (inputs on the GPU, plans, trained weights), ``run``
is one pass through the public entry points, ``exact`` the same result from
plain torch in float64 without this package's code, ``work`` the bytes and
operations a pass cannot do without, ``tolerance`` how far another correct
implementation of the same precision may be off.

The families (``path``) and what each stands for:

* ``normalized``  ``SequentialSystem.rayfunction`` with normalized field and
  pupil (the API's default): a stop solve, then the trace.  The smallest
  calls, made while a system is being designed.
* ``rayfunction`` the same entry point in physical coordinates, from a
  spot-diagram's thousand rays to 2^24; ``api`` "plan" is a prepared
  ``GridTracePlan``, as a loop over many batches keeps one.  Systems: the
  Newtonian telescope and the EUV spectrograph (two diffraction orders,
  multilayer coatings) of ``optika_amd.workloads``, and a glass singlet.
* ``rays``        ``propagators.propagate_rays`` / ``accumulate_rays``: rays
  that the program already has, through a list of surfaces.
* ``image``       ``SequentialSystem.image``: the forward model of a scene,
  from radiance to noisy electrons (stop solve, ray generation, trace,
  binning, exposure).
* ``collect``     ``ImagingSensor.collect``: binning of traced rays.
* ``tolerance``   ``BatchedSystem.trace``: perturbed spectrographs, each with
  its own number of rays.
* ``infer``       ``Surrogate.infer_traced``: the learned surrogate with its
  flagged rays traced.
* ``train``       one optimiser step of the surrogate's network: loss, all
  gradients, Adam.
"""

from __future__ import annotations

import math
import pathlib

import numpy as np
import torch

from optika_amd import (BatchedSystem, apertures, materials, propagators, sags, sensors, surfaces,
                        surrogate, systems, workloads)
from optika_amd._trace import GridTracePlan
from optika_amd.batch import STAT_FIELDS
from optika_amd.rays import RayVectorArray
from optika_amd.transformations import Cartesian3dTranslation
from optika_amd.vectors import Cartesian2dVectorArray, Cartesian3dVectorArray

DEV = "cuda"

# field half width (deg), pupil radius (mm) and wavelengths (nm) of the ray
# grids, as the repository's workloads draw them
GRIDS = {
    "newtonian": (0.25, 100.0, 400.0, 700.0),
    "spectrograph": (0.05, 40.0, 58.0, 63.0),
    "singlet": (0.5, 12.0, 400.0, 700.0),
}
SURROGATE_LO = [-0.05, -0.05, -40.0, -40.0, 58.0]
SURROGATE_HI = [0.05, 0.05, 40.0, 40.0, 63.0]
SURROGATE_FIT_RAYS = 1 << 18
# residual scales (mm, mm, log intensity) of the network's outputs: a system
# whose cubic fit leaves a few pixels, so that the network's part of the
# outputs stands well above float32 rounding
SURROGATE_SCALE = (0.05, 0.05, 0.05)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # interactive design: normalized coordinates, one wavelength
        {"name": "normalized_1k", "path": "normalized", "rays": 1024},
        # the headline workload, float64 drop-in form, a loop over batches
        {"name": "newtonian_f64_16m", "path": "rayfunction", "system": "newtonian",
         "precision": "f64", "rays": 1 << 24, "api": "plan"},
        # the float32 form, a ragged count through the system's own method
        {"name": "newtonian_f32_5m", "path": "rayfunction", "system": "newtonian",
         "precision": "f32", "rays": 5_000_011, "api": "system"},
        # coated optics, two diffraction orders, both forms
        {"name": "spectrograph_f64_2m", "path": "rayfunction", "system": "spectrograph",
         "precision": "f64", "rays": 2_000_003, "api": "system"},
        {"name": "spectrograph_f32_8m", "path": "rayfunction", "system": "spectrograph",
         "precision": "f32", "rays": 1 << 23, "api": "plan"},
        # a refracting system of a user's own
        {"name": "singlet_f64_1m", "path": "rayfunction", "system": "singlet",
         "precision": "f64", "rays": 1_048_583, "api": "system"},
        # rays in hand through a list of surfaces, every field in and out
        {"name": "propagate_f64_3m", "path": "rays", "precision": "f64", "rays": 3_000_001,
         "accumulate": False},
        # the forward model of a small field with a sampled pupil
        {"name": "image_1m", "path": "image", "bands": 4, "field": 128, "pupil": 4},
        # the binning of the headline workload's float32 rays
        {"name": "collect_f32_16m", "path": "collect", "precision": "f32", "rays": 1 << 24,
         "pixels": 2048, "bands": 1},
        # tolerance analysis
        {"name": "tolerance_f32_256", "path": "tolerance", "precision": "f32", "instances": 256},
        # the surrogate, used and trained
        {"name": "infer_4m", "path": "infer", "rays": 1 << 22},
        {"name": "train_64k", "path": "train", "rows": 65536},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["normalized", "rayfunction", "rayfunction", "rayfunction", "rays", "image",
                       "collect", "tolerance", "infer", "train"])
    precision = rng.choice(["f64", "f32"])
    if path == "normalized":
        return {"path": path, "rays": _log_int(rng, 64, 1 << 20)}
    if path == "rayfunction":
        system = rng.choice(["newtonian", "spectrograph", "singlet"])
        most = {"newtonian": 1 << 24, "spectrograph": 1 << 21, "singlet": 1 << 23}[system]
        return {"path": path, "system": system, "precision": precision,
                "rays": _log_int(rng, 64, most), "api": rng.choice(["system", "plan"])}
    if path == "rays":
        acc = rng.random() < 0.4
        return {"path": path, "precision": precision, "rays": _log_int(rng, 64, 1 << (21 if acc else 23)),
                "accumulate": acc}
    if path == "image":
        return {"path": path, "bands": rng.randint(1, 5), "field": _log_int(rng, 8, 128),
                "pupil": rng.randint(1, 4)}
    if path == "collect":
        return {"path": path, "precision": precision, "rays": _log_int(rng, 1000, 1 << 23),
                "pixels": rng.choice([128, 500, 1024, 2048]), "bands": rng.randint(1, 3)}
    if path == "tolerance":
        return {"path": path, "precision": precision, "instances": _log_int(rng, 8, 200)}
    if path == "infer":
        return {"path": path, "rays": _log_int(rng, 100, 1 << 22)}
    return {"path": path, "rows": 128 * _log_int(rng, 4, 512)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _uniform(g, n, lo, hi, dtype=torch.float64):
    return torch.rand(n, generator=g, device=DEV, dtype=dtype) * (hi - lo) + lo


def _grid(kind, n, seed, dtype):
    """Field x, y (deg), pupil x, y (mm; uniform on a disc), wavelength (nm):
    float32-representable values, so that both precisions trace the same
    rays."""
    half, radius, w0, w1 = GRIDS[kind]
    g = _generator(seed)
    r = radius * torch.sqrt(_uniform(g, n, 0.0, 1.0))
    th = _uniform(g, n, 0.0, 2 * math.pi)
    cols = [_uniform(g, n, -half, half), _uniform(g, n, -half, half),
            r * torch.cos(th), r * torch.sin(th), _uniform(g, n, w0, w1)]
    return [c.float().to(dtype).contiguous() for c in cols]


def _dtype(case):
    return torch.float64 if case["precision"] == "f64" else torch.float32


def _singlet():
    """A biconvex N-BK7 lens of about 100 mm focal length, stopped at its
    first surface."""
    lens = dict(aperture=apertures.CircularAperture(12.7))
    return systems.SequentialSystem(
        surfaces=[
            surfaces.Surface(name="front", sag=sags.SphericalSag(radius=103.0),
                             material=materials.Glass.n_bk7(), is_pupil_stop=True,
                             transformation=Cartesian3dTranslation(z=20.0), **lens),
            surfaces.Surface(name="back", sag=sags.SphericalSag(radius=-103.0),
                             transformation=Cartesian3dTranslation(z=24.0), **lens),
        ],
        sensor=sensors.ImagingSensor(
            name="sensor", width_pixel=5e-3, num_pixel=Cartesian2dVectorArray(1024, 1024),
            is_field_stop=True, transformation=Cartesian3dTranslation(z=121.5)),
    )


def _system(kind):
    return {"newtonian": workloads.newtonian, "spectrograph": workloads.spectrograph,
            "singlet": _singlet}[kind]()


def _normalized_inputs(case, seed):
    g = _generator(seed)
    return [_uniform(g, case["rays"], -1.0, 1.0) for _ in range(4)]


def _ray_inputs(case, seed):
    """Rays in the Newtonian's system frame with every field set, as another
    program hands them over: collimated within the field, on the pupil."""
    fx, fy, px, py, wl = _grid("newtonian", case["rays"], seed, torch.float64)
    ax, ay = torch.deg2rad(fx), torch.deg2rad(fy)
    d = [-torch.cos(ay) * torch.sin(ax), -torch.sin(ay), torch.cos(ay) * torch.cos(ax)]
    g = _generator(seed + 7)
    n = case["rays"]
    return {"position": [px, py, torch.zeros_like(px)], "direction": d, "wavelength": wl,
            "intensity": _uniform(g, n, 0.5, 1.5), "attenuation": torch.zeros_like(px),
            "index": torch.ones_like(px), "unvignetted": _uniform(g, n, 0.0, 1.0) < 0.98}


def _image_inputs(case, seed):
    """A scene of bright lognormal structure over the Newtonian's field."""
    rng = np.random.default_rng(int(seed))
    f = np.linspace(-0.05, 0.05, case["field"] + 1)
    w = np.linspace(480.0, 560.0, case["bands"] + 1)
    radiance = 1e10 * rng.lognormal(0.0, 0.7, (case["bands"], case["field"], case["field"]))
    v = np.linspace(-1.0, 1.0, case["pupil"] + 1)
    return w, f, radiance, v


def _collect_inputs(case, seed):
    """Rays at the sensor as the headline workload leaves them: field angles
    of +-0.25 deg on a 1 m focal length, a blur of under a pixel, a few per
    cent vignetted."""
    n, dt = case["rays"], _dtype(case)
    half = 0.015 * case["pixels"] / 2
    reach = min(4.4, 1.02 * half)
    g = _generator(seed)
    blur = lambda: torch.randn(n, generator=g, device=DEV, dtype=torch.float64) * 0.008  # noqa: E731
    x = _uniform(g, n, -reach, reach) + blur()
    y = _uniform(g, n, -reach, reach) + blur()
    dx, dy = _uniform(g, n, -0.1, 0.1), _uniform(g, n, -0.1, 0.1)
    dz = torch.sqrt(1 - dx * dx - dy * dy)
    wl = _uniform(g, n, 400.0, 700.0)
    inten = _uniform(g, n, 0.5, 1.0)
    ok = _uniform(g, n, 0.0, 1.0) < 0.97
    c = [t.to(dt) for t in (x, y, dx, dy, dz, wl, inten)]
    return c, ok, np.linspace(400.0, 700.0, case["bands"] + 1)


def _tolerance_inputs(case, seed):
    systems_, counts, grid = workloads.tolerance_batch(case["instances"], seed=int(seed))
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a, np.float32), device=DEV)  # noqa: E731
    cols = [t(a) for a in (grid.field_x, grid.field_y, grid.pupil_x, grid.pupil_y, grid.wavelength)]
    return systems_, counts, [c.to(_dtype(case)) for c in cols]


def _fit_columns(seed):
    return lambda count, chunk_seed: _grid("spectrograph", count, int(seed) * 4096 + chunk_seed,
                                           torch.float32)


def _mlp_params(seed):
    """Weights of the surrogate's network (flat, float32, host): uniform
    within 1/sqrt(fan in) times sqrt(3), small biases."""
    g = torch.Generator().manual_seed(int(seed))
    parts = []
    for a, b in zip(surrogate.WIDTHS[:-1], surrogate.WIDTHS[1:]):
        s = math.sqrt(3.0 / a)
        parts += [(torch.rand(a * b, generator=g) * 2 - 1) * s, (torch.rand(b, generator=g) * 2 - 1) * 0.1]
    return torch.cat(parts)


def _train_inputs(case, seed):
    """Normalised inputs and standardised residual targets (a smooth map with
    some structure, as a polynomial's residual has)."""
    g = _generator(seed)
    n = case["rows"]
    x = torch.rand(n, 5, generator=g, device=DEV) * 2 - 1
    a = torch.randn(5, 3, generator=g, device=DEV) * 2
    t = torch.sin(x[:, :1] * a[0] + x[:, 1:2] * a[1] + x[:, 2:3] * a[2]) \
        + torch.cos(x[:, 3:4] * a[3] + x[:, 4:] * a[4]) * 0.5
    return x.contiguous(), t.contiguous()


def prepare(case, seed):
    path = case["path"]
    if path == "normalized":
        return {"case": case, "system": workloads.stop_newtonian(), "cols": _normalized_inputs(case, seed)}
    if path == "rayfunction":
        state = {"case": case, "system": _system(case["system"]),
                 "cols": _grid(case["system"], case["rays"], seed, _dtype(case))}
        if case["api"] == "plan":
            state["plan"] = GridTracePlan(state["system"], case["rays"], precision=case["precision"])
        return state
    if path == "rays":
        r, dt = _ray_inputs(case, seed), _dtype(case)
        rays = RayVectorArray(
            wavelength=r["wavelength"].to(dt),
            position=Cartesian3dVectorArray(*(t.to(dt) for t in r["position"])),
            direction=Cartesian3dVectorArray(*(t.to(dt) for t in r["direction"])),
            intensity=r["intensity"].to(dt), attenuation=r["attenuation"].to(dt),
            index_refraction=r["index"].to(dt), unvignetted=r["unvignetted"])
        return {"case": case, "surfaces": workloads.newtonian().surfaces_all, "rays": rays}
    if path == "image":
        return {"case": case, "system": workloads.stop_newtonian(), "scene": _image_inputs(case, seed),
                "seed": int(seed)}
    if path == "collect":
        (x, y, dx, dy, dz, wl, inten), ok, edges = _collect_inputs(case, seed)
        rays = RayVectorArray(wavelength=wl, position=Cartesian3dVectorArray(x, y, torch.zeros_like(x)),
                              direction=Cartesian3dVectorArray(dx, dy, dz), intensity=inten,
                              unvignetted=ok)
        p = case["pixels"]
        return {"case": case, "rays": rays, "edges": edges,
                "sensor": sensors.ImagingSensor(num_pixel=Cartesian2dVectorArray(p, p))}
    if path == "tolerance":
        systems_, counts, cols = _tolerance_inputs(case, seed)
        return {"case": case, "batch": BatchedSystem(systems_), "counts": counts, "cols": cols}
    if path == "infer":
        sg = surrogate.Surrogate(workloads.spectrograph(), SURROGATE_LO, SURROGATE_HI)
        sg.prepare(_fit_columns(seed), SURROGATE_FIT_RAYS)
        sg.mlp.set_params(_mlp_params(seed).to(DEV))
        sg.scale = torch.tensor(SURROGATE_SCALE, dtype=torch.float64, device=DEV)
        # the map of a calibration that flags no cell
        sg.err_map = torch.zeros(16 * 8 * 8, dtype=torch.bool, device=DEV)
        return {"case": case, "surrogate": sg,
                "cols": _grid("spectrograph", case["rays"], seed + 1, torch.float32)}
    x, t = _train_inputs(case, seed)
    mlp = surrogate.MLP(torch.device(DEV))
    mlp.set_params(_mlp_params(seed).to(DEV))
    return {"case": case, "mlp": mlp, "x": x, "t": t,
            "weight": torch.tensor([1.0, 1.0, 0.25], device=DEV)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _vec(v):
    return [v.x, v.y] + ([v.z] if hasattr(v, "z") else [])


def _rays_out(r, full, on_sensor=True):
    # on_sensor: z is the sensor's plane, zero but for rounding, of which no
    # relative error can be stated
    out = {"position": _vec(r.position)[:2 if on_sensor else 3], "direction": _vec(r.direction),
           "intensity": r.intensity, "unvignetted": r.unvignetted}
    if full:
        out.update(wavelength=r.wavelength, attenuation=r.attenuation, index=r.index_refraction)
    return out


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "normalized":
        fx, fy, px, py = state["cols"]
        r = state["system"].rayfunction(wavelength=500.0, field=Cartesian2dVectorArray(fx, fy),
                                        pupil=Cartesian2dVectorArray(px, py)).outputs
        return _rays_out(r, False)
    if path == "rayfunction":
        full = case["system"] == "singlet"  # glass: the wavelength and the index change on the way
        if case["api"] == "plan":
            return _rays_out(state["plan"](*state["cols"]), full)
        fx, fy, px, py, wl = state["cols"]
        r = state["system"].rayfunction(
            wavelength=wl, field=Cartesian2dVectorArray(fx, fy), pupil=Cartesian2dVectorArray(px, py),
            normalized_field=False, normalized_pupil=False, precision=case["precision"]).outputs
        return _rays_out(r, full)
    if path == "rays":
        f = propagators.accumulate_rays if case["accumulate"] else propagators.propagate_rays
        return _rays_out(f(state["surfaces"], state["rays"], precision=case["precision"]), True, False)
    if path == "image":
        w, f, radiance, v = state["scene"]
        return state["system"].image(w, f, f, radiance, pupil=Cartesian2dVectorArray(v, v),
                                     seed=state["seed"])
    if path == "collect":
        image, cosine = state["sensor"].collect(state["rays"], wavelength=state["edges"])
        return {"image": image, "cosine": cosine}
    if path == "tolerance":
        stats = state["batch"].trace(*state["cols"], counts=state["counts"], precision=case["precision"])
        return {k: stats[..., i] for i, k in enumerate(STAT_FIELDS)}
    if path == "infer":
        out = state["surrogate"].infer_traced(*state["cols"])
        # "list" is the kernel's work list: the same rays as "fallback", in
        # the order in which the blocks found them
        return {k: out[k] for k in ("x", "y", "intensity", "unvignetted", "fallback", "count")}
    mlp = state["mlp"]
    loss = mlp.loss_grad(state["x"], state["t"], state["weight"])
    mlp.adam_step(2e-3)
    return {"loss": loss, "y": mlp.y, "gradient": mlp.g, "parameters": mlp.p}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

# float64 operations of one ray (both orders of the spectrograph): the
# surfaces' geometry, and for a coated mirror the 2 x 2 transfer matrices of
# both polarizations
FLOPS = {"newtonian": 400, "singlet": 300, "spectrograph": 3 * 2500 + 1500}
MLP_FLOPS = 2 * sum(a * b for a, b in zip(surrogate.WIDTHS[:-1], surrogate.WIDTHS[1:]))


def _tolerance_counts(case):
    # mean of a log-uniform count in [1000, 64000)
    return int(case["instances"] * (64000 - 1000) / math.log(64.0))


def work(case):
    path = case["path"]
    w = 4 if case.get("precision") == "f32" else 8
    if path == "normalized":
        n = case["rays"]
        return {"bytes": n * (4 * 8 + 7 * 8 + 1), "flops": n * 400 + 441 * 2000}
    if path == "rayfunction":
        n, s = case["rays"], case["system"]
        paths = 2 if s == "spectrograph" else 1
        ins = 4 if s == "newtonian" else 5  # an all-mirror trace does not read the wavelength
        outs = 10 if s == "singlet" else 7
        return {"bytes": n * (ins * w + paths * (outs * w + 1)), "flops": n * FLOPS[s]}
    if path == "rays":
        n = case["rays"]
        return {"bytes": n * (10 * w + 1) * (1 + (4 if case["accumulate"] else 1)), "flops": n * 400}
    if path == "image":
        rays = case["bands"] * case["field"] ** 2 * case["pupil"] ** 2
        # one ray per cell, binned where it lands: the scene in, the electrons out
        return {"bytes": case["bands"] * (case["field"] ** 2 + 128 * 128) * 8, "flops": rays * 450}
    if path == "collect":
        return {"bytes": case["rays"] * (5 * w + 1) + 2 * 8 * case["bands"] * case["pixels"] ** 2,
                "flops": case["rays"] * 10}
    if path == "tolerance":
        n = _tolerance_counts(case)
        return {"bytes": n * 5 * w, "flops": n * FLOPS["spectrograph"]}
    if path == "infer":
        return {"bytes": case["rays"] * (5 * 4 + 3 * 4 + 2), "flops": case["rays"] * MLP_FLOPS}
    return {"bytes": case["rows"] * 8 * 4 + 7 * 4 * surrogate.NUM_PARAMS,
            "flops": 3 * case["rows"] * MLP_FLOPS}


def tolerance(case):
    """About four times what the path is off ``exact``."""
    path = case["path"]
    if path == "normalized":
        return {"rel": 1e-11, "max": 1e-9, "differ": 1e-4}
    if path in ("rayfunction", "rays"):
        # float64: the conic intercept's quadratic cancels on the Newtonian,
        # which leaves it 1e-8 off a stable evaluation
        if case["precision"] == "f64":
            return {"rel": 5e-8, "max": 1e-5, "differ": 1e-4}
        return {"rel": 2e-6, "max": 1e-4, "differ": 1e-4}
    if path == "image":
        # electrons are Poisson draws around sums whose order is not fixed
        return {"rel": 1e-4, "max": 1e-2}
    if path == "collect":
        return {"rel": 1e-12, "max": 1e-10}
    if path == "tolerance":
        if case["precision"] == "f64":
            return {"rel": 1e-9, "max": 1e-7}
        return {"rel": 2e-6, "max": 1e-4}
    if path == "infer":
        # "max": a ray at the margin that one side traces and the other
        # predicts is off by the network's whole part
        return {"rel": 4e-5, "max": 0.2, "differ": 1e-4}
    return {"rel": 1e-2, "max": 0.4}


# ---------------------------------------------------------------------------
# the same in float64 without this package's code
# ---------------------------------------------------------------------------

def _affine(t):
    """(matrix, vector) of a transformation, its elements applied in order."""
    m, v = np.eye(3), np.zeros(3)
    for e in ([] if t is None else getattr(t, "transformations", [t])):
        if hasattr(e, "angle"):
            c, s = math.cos(math.radians(e.angle)), math.sin(math.radians(e.angle))
            axis = type(e).__name__[-1]
            k = {"X": [[1, 0, 0], [0, c, -s], [0, s, c]], "Y": [[c, 0, s], [0, 1, 0], [-s, 0, c]],
                 "Z": [[c, -s, 0], [s, c, 0], [0, 0, 1]]}[axis]
            m, v = np.array(k) @ m, np.array(k) @ v
        else:
            v = v + np.array([e.x, e.y, e.z], float)
    return m, v


def _mat(m, p):
    return [sum(float(m[i][j]) * p[j] for j in range(3)) for i in range(3)]


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _sag_gradient(sag, p):
    """A function that vanishes on the sag, and its gradient (z part < 0)."""
    x, y, z = p
    kind = type(sag).__name__
    if kind == "NoSag":
        return -z, [torch.zeros_like(x), torch.zeros_like(x), -torch.ones_like(x)]
    c = 1.0 / sag.radius
    if kind == "ToroidalSag":
        r = sag.radius_of_rotation
        g = torch.sqrt(1 - (c * y) ** 2)
        zy = c * y * y / (1 + g)
        f = torch.sqrt((r - zy) ** 2 - x * x)
        return ((zy * (2 * r - zy) + x * x) / (r + f) - z,
                [x / f, (r - zy) * (c * y / g) / f, -torch.ones_like(x)])
    kp1 = 1.0 + (sag.conic if kind == "ConicSag" else 0.0)
    return (0.5 * c * (x * x + y * y + kp1 * z * z) - z,
            [c * x, c * y, c * kp1 * z - 1])


def _chemical(name, wl):
    path = pathlib.Path(surrogate.__file__).parent / "data" / "nk" / f"{name}.nk"
    t = np.array([[float(v) for v in line.split()[:3]] for line in path.read_text().splitlines()
                  if line.strip() and not line.strip().startswith(";")])
    w, n, k = (torch.as_tensor(np.ascontiguousarray(c), device=DEV) for c in t.T)
    x = wl * 10.0
    j = (torch.searchsorted(w, x, right=True) - 1).clamp(0, len(w) - 2)
    f = (x - w[j]) / (w[j + 1] - w[j])
    return torch.complex(n[j] + f * (n[j + 1] - n[j]), k[j] + f * (k[j + 1] - k[j]))


def _multilayer(material, wl, cos):
    """Reflectance of a periodic multilayer on a substrate, both
    polarizations averaged: characteristic matrices, in complex128."""
    layers = [(la.chemical, float(la.thickness)) for la in material.layers.layers]
    stack = [(None, 0.0), *layers, (material.substrate.chemical, 0.0)]
    amb = (torch.ones_like(wl) + 0j, cos + 0j, None)
    media = [amb]
    for name, h in stack[1:]:
        n = _chemical(name, wl)
        c = torch.sqrt(1 - (1 - cos * cos) / (n * n))
        media.append((n, c, torch.exp(4j * math.pi * h * n * c / wl)))

    def crossing(i, j):
        """The interface i -> j and the way through j, as the matrix of the
        map from the amplitude ratio behind j to the one before i, both
        polarizations: r -> (rho + r f) / (1 + rho r f), f = exp(2 i beta)."""
        (ni, ci, _), (nj, cj, f) = i, j
        rho = torch.stack([(ni * ci - nj * cj) / (ni * ci + nj * cj),
                           (ci.conj() / ni - cj.conj() / nj) / (ci.conj() / ni + cj.conj() / nj)])
        return f.expand_as(rho), rho, rho * f, torch.ones_like(rho)

    def times(x, y):
        return (x[0] * y[0] + x[1] * y[2], x[0] * y[1] + x[1] * y[3],
                x[2] * y[0] + x[3] * y[2], x[2] * y[1] + x[3] * y[3])

    # first period from the ambient medium, the others from the last layer
    first, again = crossing(media[0], media[1]), crossing(media[-2], media[1])
    for i, j in zip(media[1:-2], media[2:-1]):
        first, again = times(first, crossing(i, j)), times(again, crossing(i, j))
    total, e = first, material.layers.num_periods - 1
    while e:
        if e & 1:
            total = times(total, again)
        again, e = times(again, again), e >> 1
    _, rho, _, one = times(total, crossing(media[-2], media[-1]))
    return ((rho / one).abs() ** 2).mean(0)


def _inside(aperture, p):
    x, y = p[0], p[1]
    kind = type(aperture).__name__
    if kind == "CircularAperture":
        return x * x + y * y <= aperture.radius ** 2
    if kind == "RectangularAperture":
        return (x.abs() <= aperture.half_width.x) & (y.abs() <= aperture.half_width.y)
    inside = torch.zeros_like(x, dtype=torch.bool)
    for (xi, yi), (xj, yj) in _sides(aperture):
        if yi != yj:
            inside ^= ((yi > y) != (yj > y)) & (x < (xj - xi) * (y - yi) / (yj - yi) + xi)
    return inside


def _sides(aperture):
    n = aperture.num_vertices
    v = [(aperture.radius * math.cos(2 * math.pi * k / n), aperture.radius * math.sin(2 * math.pi * k / n))
         for k in range(n)]
    return [(v[k], v[k - 1]) for k in range(n)]


def _half_width(surface):
    w, p = surface.width_pixel, surface.num_pixel
    return apertures.RectangularAperture(half_width=(w * p.x / 2, w * p.y / 2))


def _step(s, r, order):
    """Rays through one surface, in and out in the system frame; ``local``:
    the position and direction in the surface's own frame."""
    m, v = _affine(s.transformation)
    p = _mat(m.T, [r["p"][k] - float(v[k]) for k in range(3)])
    d = _mat(m.T, r["d"])
    sensor = hasattr(s, "num_pixel")
    sag = s.sag
    o = _affine(getattr(sag, "transformation", None))[1]
    q = [p[k] - float(o[k]) for k in range(3)]
    t = -q[2] / d[2]
    for _ in range(0 if type(sag).__name__ == "NoSag" else 8):
        f, g = _sag_gradient(sag, [q[k] + t * d[k] for k in range(3)])
        t = t - f / _dot(g, d)
    q = [q[k] + t * d[k] for k in range(3)]
    _, g = _sag_gradient(sag, q)
    length = torch.sqrt(_dot(g, g))
    u = [c / length for c in g]
    p = [q[k] + float(o[k]) for k in range(3)]
    wl, n1, a = r["wl"], r["index"], d
    if s.rulings is not None:
        c = s.rulings.spacing.coefficients
        spacing = sum(c[k] * p[0] ** k for k in c)
        sign = torch.sign(_dot(a, u))
        a = [a[0] + sign * order * wl * 1e-6 / (n1 * spacing), a[1], a[2]]
    mat = s.material
    kind = type(mat).__name__
    mirror = kind in ("Mirror", "MultilayerMirror")
    n2 = n1 if mirror else torch.ones_like(wl)
    if kind == "Glass":
        w2 = (wl * 1e-3) ** 2
        n2 = torch.sqrt(1 + sum(b * w2 / (w2 - cc) for b, cc in
                                ((mat.b1, mat.c1), (mat.b2, mat.c2), (mat.b3, mat.c3))))
    ratio = n1 / n2
    au = _dot(a, u)
    root = torch.sqrt(1 / ratio ** 2 + au * au - _dot(a, a))
    k = -au - torch.sign(au) * (1.0 if mirror else -1.0) * root
    b = [ratio * (a[i] + k * u[i]) for i in range(3)]
    inten = r["inten"]
    if kind == "MultilayerMirror":
        inten = inten * _multilayer(mat, wl, -au)
    ap = _half_width(s) if sensor else s.aperture
    ok = r["ok"]
    if ap is not None:
        ok = ok & _inside(ap, b if ap.unit == "direction" else p)
    out = {"p": [c + float(v[i]) for i, c in enumerate(_mat(m, p))], "d": _mat(m, b),
           "wl": wl / ratio, "inten": inten, "index": n2, "ok": ok}
    return out, {**out, "p": p, "d": b}


def _grid_rays(cols):
    fx, fy, px, py, wl = [c.double() for c in cols]
    ax, ay = torch.deg2rad(fx), torch.deg2rad(fy)
    one = torch.ones_like(px)
    return {"p": [px, py, torch.zeros_like(px)],
            "d": [-torch.cos(ay) * torch.sin(ax), -torch.sin(ay), torch.cos(ay) * torch.cos(ax)],
            "wl": wl, "inten": one, "index": one, "ok": torch.ones_like(px, dtype=torch.bool)}


def _all_surfaces(system):
    return [system.object, *system.surfaces, system.sensor]


def _trace_exact(surfaces_, r, order=0):
    """After every surface, in the system frame and in the surface's own."""
    world, local = [], []
    for s in surfaces_:
        r, loc = _step(s, r, order)
        world.append(r)
        local.append(loc)
    return world, local


def _exact_out(rs, full, stack, on_sensor=True):
    cat = (lambda f: torch.stack([f(r) for r in rs])) if stack else (lambda f: f(rs[0]))
    out = {"position": [cat(lambda r, k=k: r["p"][k]) for k in range(2 if on_sensor else 3)],
           "direction": [cat(lambda r, k=k: r["d"][k]) for k in range(3)],
           "intensity": cat(lambda r: r["inten"]), "unvignetted": None}
    if full:
        out.update(wavelength=cat(lambda r: r["wl"]), attenuation=None, index=cat(lambda r: r["index"]))
    return out


def _stop_pupil(system):
    """Half extents (field in degrees, pupil in mm, per axis: low, high) of
    the stop-solve Newtonian: rays along the field outline that meet the
    pupil stop's outline, by Newton's method on their start position."""
    az = torch.deg2rad(torch.linspace(0.0, 360.0, 21, device=DEV, dtype=torch.float64))
    f, a = torch.meshgrid(az, az, indexing="ij")
    f, a = f.reshape(-1), a.reshape(-1)
    sin_r, radius = system.object.aperture.radius, system.surfaces[1].aperture.radius
    d = [sin_r * torch.cos(f), sin_r * torch.sin(f)]
    d.append(torch.sqrt(1 - d[0] ** 2 - d[1] ** 2))
    goal = [radius * torch.cos(a), radius * torch.sin(a)]

    def end(x, y):
        one = torch.ones_like(x)
        r = {"p": [x, y, 0 * x], "d": d, "wl": 500.0 * one, "inten": one, "index": one, "ok": one > 0}
        world, _ = _trace_exact(list(system.surfaces), r)
        return world[-1]["p"]

    x, y = goal[0].clone(), goal[1].clone()
    h = 1e-5
    for _ in range(12):
        e = end(x, y)
        ex, ey = end(x + h, y), end(x, y + h)
        j = [(ex[0] - e[0]) / h, (ey[0] - e[0]) / h, (ex[1] - e[1]) / h, (ey[1] - e[1]) / h]
        det = j[0] * j[3] - j[1] * j[2]
        rx, ry = e[0] - goal[0], e[1] - goal[1]
        x, y = x - (j[3] * rx - j[1] * ry) / det, y - (j[0] * ry - j[2] * rx) / det
    ang = [-torch.rad2deg(torch.atan2(d[0], d[2])), -torch.rad2deg(torch.asin(d[1]))]
    return [(float(t.min()), float(t.max())) for t in (*ang, x, y)]


def _exact_normalized(case, seed):
    system = workloads.stop_newtonian()
    cols = [(hi - lo) * (u + 1) / 2 + lo
            for u, (lo, hi) in zip(_normalized_inputs(case, seed), _stop_pupil(system))]
    _, local = _trace_exact(_all_surfaces(system), _grid_rays(cols + [torch.full_like(cols[0], 500.0)]))
    return _exact_out([local[-1]], False, False)


def _exact_rayfunction(case, seed):
    system = _system(case["system"])
    r = _grid_rays(_grid(case["system"], case["rays"], seed, _dtype(case)))
    orders = (-1, 1) if case["system"] == "spectrograph" else (0,)
    ends = [_trace_exact(_all_surfaces(system), r, o)[1][-1] for o in orders]
    return _exact_out(ends, case["system"] == "singlet", len(orders) > 1)


def _exact_rays(case, seed):
    r, dt = _ray_inputs(case, seed), _dtype(case)
    c = lambda t: t.to(dt).double()  # noqa: E731
    world, _ = _trace_exact(workloads.newtonian().surfaces_all, {
        "p": [c(t) for t in r["position"]], "d": [c(t) for t in r["direction"]], "wl": c(r["wavelength"]),
        "inten": c(r["intensity"]), "index": c(r["index"]), "ok": r["unvignetted"]})
    return _exact_out(world if case["accumulate"] else world[-1:], True, case["accumulate"], False)


def _exact_collect(case, seed):
    (x, y, _, _, dz, wl, inten), ok, edges = _collect_inputs(case, seed)
    p = case["pixels"]
    half = 0.015 * p / 2

    def bins(v, e):
        e = torch.as_tensor(e, device=DEV)
        j = torch.searchsorted(e, v, right=True) - 1
        j = torch.where(v == e[-1], len(e) - 2, j)
        return j, (j >= 0) & (j < len(e) - 1)

    e = np.linspace(-half, half, p + 1)
    jx, ox = bins(x.double(), e)
    jy, oy = bins(y.double(), e)
    jw, ow = bins(wl.double(), edges)
    w = torch.where(ok & ox & oy & ow, inten.double(), 0.0)
    at = torch.where(ox & oy & ow, (jw * p + jx) * p + jy, 0)
    size = case["bands"] * p * p
    image = torch.zeros(size, dtype=torch.float64, device=DEV).index_add_(0, at, w)
    moment = torch.zeros(size, dtype=torch.float64, device=DEV).index_add_(0, at, w * dz.double())
    cosine = torch.where(image > 0, moment / torch.where(image > 0, image, 1.0), 1.0)
    shape = (case["bands"], p, p)
    return {"image": image.reshape(shape), "cosine": cosine.reshape(shape)}


def _exact_tolerance(case, seed):
    systems_, counts, cols = _tolerance_inputs(case, seed)
    rows, start = [], 0
    for system, n in zip(systems_, counts):
        r = _grid_rays([c[start:start + int(n)] for c in cols])
        start += int(n)
        for order in (-1, 1):
            end = _trace_exact(_all_surfaces(system), r, order)[1][-1]
            w = end["ok"].double()
            i, x, y = end["inten"], end["p"][0], end["p"][1]
            s = [w.sum()] + [torch.where(end["ok"], v, 0.0).sum() for v in (i, x, y, x * x, y * y)]
            c = s[0].clamp(min=1)
            var = s[4] / c - (s[2] / c) ** 2 + s[5] / c - (s[3] / c) ** 2
            rms = torch.where(s[0] > 0, torch.sqrt(var.clamp(min=0)), float("nan"))
            rows.append(torch.stack(s + [rms, s[1] / n]))
    t = torch.stack(rows).reshape(len(systems_), 2, 8)
    return {k: t[..., i] for i, k in enumerate(STAT_FIELDS)}


def _monomials(u):
    cols = []
    for e in surrogate.EXPONENTS:
        c = torch.ones_like(u[:, 0])
        for k, n in enumerate(e):
            for _ in range(n):
                c = c * u[:, k]
        cols.append(c)
    return torch.stack(cols, 1)


def _edge_distance(aperture, x, y):
    if type(aperture).__name__ == "CircularAperture":
        return aperture.radius - torch.sqrt(x * x + y * y)
    if type(aperture).__name__ == "RectangularAperture":
        return torch.minimum(aperture.half_width.x - x.abs(), aperture.half_width.y - y.abs())
    best = None
    for (x1, y1), (x0, y0) in _sides(aperture):
        ex, ey = x1 - x0, y1 - y0
        s = (((x - x0) * ex + (y - y0) * ey) / (ex * ex + ey * ey)).clamp(0, 1)
        d = torch.sqrt((x - x0 - s * ex) ** 2 + (y - y0 - s * ey) ** 2)
        best = d if best is None else torch.minimum(best, d)
    return torch.where(_inside(aperture, [x, y]), best, -best)


def _network(params, x):
    at = 0
    for k, (a, b) in enumerate(zip(surrogate.WIDTHS[:-1], surrogate.WIDTHS[1:])):
        w, bias = params[at:at + a * b].reshape(b, a), params[at + a * b:at + a * b + b]
        at += a * b + b
        x = x @ w.T.contiguous() + bias
        if k < len(surrogate.WIDTHS) - 2:
            x = x * torch.sigmoid(x)
    return x


def _exact_infer(case, seed):
    system = workloads.spectrograph()
    params = _mlp_params(seed).to(DEV).double()
    lo, hi = np.array(SURROGATE_LO), np.array(SURROGATE_HI)
    clips = [(k, _half_width(s) if hasattr(s, "num_pixel") else s.aperture)
             for k, s in enumerate(_all_surfaces(system))]
    clips = [(k, a) for k, a in clips if a is not None]

    def unit(cols):
        return torch.stack([(c.double() - (hi[k] + lo[k]) / 2) / ((hi[k] - lo[k]) / 2)
                            for k, c in enumerate(cols)], 1)

    def targets(cols):
        _, local = _trace_exact(_all_surfaces(system), _grid_rays(cols), -1)
        t = [local[-1]["p"][0], local[-1]["p"][1], torch.log(local[-1]["inten"])]
        for k, _ in clips:
            t += local[k]["p"][:2]
        return torch.stack(t, 1)

    fit = _fit_columns(seed)(SURROGATE_FIT_RAYS, 1000)
    t = targets(fit)
    f = _monomials(unit(fit))
    coef = torch.as_tensor(np.linalg.solve((f.T @ f).cpu().numpy(), (f.T @ t).cpu().numpy()), device=DEV)
    near = [i for i, (_, a) in enumerate(clips)
            if float(_edge_distance(a, t[:, 3 + 2 * i], t[:, 4 + 2 * i]).abs().min()) < 4 * 0.5]
    scale = torch.tensor(SURROGATE_SCALE, dtype=torch.float64, device=DEV)
    parts = []
    cols = _grid("spectrograph", case["rays"], seed + 1, torch.float32)
    for at in range(0, case["rays"], 1 << 18):
        c = [v[at:at + (1 << 18)] for v in cols]
        u = unit(c)
        fitted = _monomials(u) @ coef
        y = fitted[:, :3] + _network(params, u) * scale
        traced = torch.zeros(len(y), dtype=torch.bool, device=DEV)
        for i in near:
            traced |= _edge_distance(clips[i][1], fitted[:, 3 + 2 * i], fitted[:, 4 + 2 * i]).abs() < 0.5
        parts.append(torch.where(traced[:, None], targets(c)[:, :3], y))
    y = torch.cat(parts)
    return {"x": y[:, 0].contiguous(), "y": y[:, 1].contiguous(), "intensity": torch.exp(y[:, 2]),
            "unvignetted": None, "fallback": None, "count": None}


def _exact_train(case, seed):
    x, t = _train_inputs(case, seed)
    p = _mlp_params(seed).to(DEV).double().requires_grad_(True)
    y = _network(p, x.double())
    weight = torch.tensor([1.0, 1.0, 0.25], device=DEV, dtype=torch.float64)
    loss = (weight * (y - t.double()) ** 2).sum() / len(y)
    g, = torch.autograd.grad(loss, p)
    step = 2e-3 * g / (g.abs() + 1e-8)  # Adam's first step
    return {"loss": loss.detach(), "y": y.detach(), "gradient": g, "parameters": (p - step).detach()}


def exact(case, seed):
    path = case["path"]
    if path == "image":
        return None  # electrons are random draws
    return {"normalized": _exact_normalized, "rayfunction": _exact_rayfunction, "rays": _exact_rays,
            "collect": _exact_collect, "tolerance": _exact_tolerance, "infer": _exact_infer,
            "train": _exact_train}[path](case, seed)
