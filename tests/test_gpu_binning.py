"""The tiled binning where its blocks, chunks and workspace change: ray counts
at the edges of a block's share, images of one to many tiles, rays sorted into
few tiles, every workspace a caller may offer, and the cosine of empty pixels."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rays(n, f32, seed, clustered):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    u = lambda lo, hi: torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * (hi - lo) + lo  # noqa: E731
    x, y = u(-1.1, 1.1), u(-1.1, 1.1)
    if clustered:  # sorted, within a few pixels
        x, y = torch.sort(0.01 * x).values, 0.01 * y
    dt = torch.float32 if f32 else torch.float64
    cols = [t.to(dt) for t in (x, y, u(0.5, 1.0), u(395.0, 705.0), u(0.1, 1.0))]
    return cols, (u(0.0, 1.0) < 0.9).view(torch.uint8)


def _bin(cols, mask, edges, nx, ny, nbytes):
    import torch

    from optika_amd import _lib

    L = _lib.lib()
    n, nw = mask.numel(), len(edges) - 1
    image = torch.zeros((nw, nx, ny), dtype=torch.float64, device="cuda")
    moment = torch.zeros_like(image)
    e = torch.as_tensor(np.asarray(edges, np.float64), device="cuda")
    a = _lib.CollectArgs()
    a.position[0], a.position[1], a.direction_z, a.wavelength, a.intensity = (
        c.data_ptr() for c in cols)
    a.unvignetted, a.wavelength_edges = mask.data_ptr(), e.data_ptr()
    a.n_wavelength, a.nx, a.ny = nw, nx, ny
    a.precision = _lib.F32 if cols[0].dtype == torch.float32 else _lib.F64
    a.x_lo, a.x_hi, a.y_lo, a.y_hi = -1.0, 1.0, -1.0, 1.0
    a.image, a.moment = image.data_ptr(), moment.data_ptr()
    want = int(L.optk_collect_workspace(ctypes.byref(a), n))
    size = want if nbytes is None else min(nbytes(n, nw, nx, ny, a.precision == _lib.F32), want)
    ws = torch.empty(max(size, 1), dtype=torch.uint8, device="cuda")
    if size:
        a.workspace, a.workspace_bytes = ws.data_ptr(), size
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(L.optk_collect(ctypes.byref(a), n, stream))
    torch.cuda.synchronize()
    return image.cpu().numpy(), moment.cpu().numpy()


def _least(n, nw, nx, ny, f32):
    """bytes of the layout with 32768 rays a block, the least that is taken"""
    up = lambda b: (b + 255) // 256 * 256  # noqa: E731
    tiles = nw * -(-nx // 32) * -(-ny // 32)
    return (up(-(-n // 32768) * tiles * 4) + up((tiles + 1) * 4) + up(4 * n)
            + (0 if f32 else up(2 * n)) + up(16 * n))


@pytest.mark.parametrize("f32", [True, False], ids=["f32", "f64"])
@pytest.mark.parametrize("n,nx,ny,bands", [
    (1, 32, 32, 1), (4095, 33, 31, 1), (4097, 128, 65, 2), (12 * 1024 + 1, 2048, 2048, 1),
    (2_097_153, 700, 2048, 1), (300_001, 2048, 2048, 3), (3_500_000, 64, 64, 4)])
def test_tiled_binning_matches_histogramdd(n, nx, ny, bands, f32):
    edges = np.linspace(400.0, 700.0, bands + 1)
    for clustered in (False, True):
        cols, mask = _rays(n, f32, 5 + clustered, clustered)
        x, y, dz, w, a = (c.cpu().numpy().astype(np.float64) for c in cols)
        m = mask.cpu().numpy() != 0
        pts = np.stack([w, x, y], -1)[m]
        rule = [edges, np.linspace(-1.0, 1.0, nx + 1), np.linspace(-1.0, 1.0, ny + 1)]
        ref = np.histogramdd(pts, rule, weights=a[m])[0]
        mom = np.histogramdd(pts, rule, weights=(a * dz)[m])[0]
        num = np.histogramdd(pts, rule)[0]
        # a sum of k positive numbers in any order: k - 1 roundings each way
        bound = 2 * np.maximum(num - 1, 1) * 2.0 ** -53
        for nbytes in (None, _least, lambda *_: 0):
            print(f"case: binning n={n} {nx}x{ny}x{bands} f32={f32} clustered={clustered}", flush=True)
            img, got = _bin(cols, mask, edges, nx, ny, nbytes)
            assert np.array_equal(img > 0, ref > 0)
            assert np.all(np.abs(img - ref) <= bound * ref)
            # its terms carry one rounding more, of the product, on each side
            assert np.all(np.abs(got - mom) <= (bound + 2.0 ** -52) * mom)


def test_cosine_of_empty_and_odd_pixels():
    import torch

    from optika_amd import _lib

    image = torch.tensor([2.0, 0.0, -1.0, float("nan"), float("inf"), 5e-324, 3.0],
                         dtype=torch.float64, device="cuda")
    moment = torch.tensor([1.0, 4.0, 1.0, 1.0, 1.0, 0.0, 1.0], dtype=torch.float64, device="cuda")
    want = torch.where(image > 0, moment / torch.where(image > 0, image, 1.0),
                       torch.ones_like(image)).cpu().numpy()
    print("case: cosine", flush=True)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib().optk_collect_cosine(image.data_ptr(), moment.data_ptr(),
                                              moment.data_ptr(), image.numel(), stream))
    torch.cuda.synchronize()
    assert np.array_equal(moment.cpu().numpy(), want)
