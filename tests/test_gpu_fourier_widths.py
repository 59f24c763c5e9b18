"""Every specialised Fourier kernel with several fields at each number of fields a workgroup, against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

A = 6.3712e6
GRIDS = [(64, 32, 21), (96, 48, 31), (128, 64, 42), (192, 94, 62), (256, 128, 84), (288, 144, 95), (384, 190, 126),
         (512, 256, 170), (576, 288, 190), (768, 384, 254), (72, 36, 23)]


# five fields: a full workgroup of four and one of a single field, or one of eight with three missing; the pairs of a
# vector transform change buffers within a workgroup
@pytest.mark.parametrize("width", ["default", "4", "8"])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: f"{g[0]}x{g[1]}")
def test_fields_per_workgroup(grid, width, monkeypatch):
    """Scalar and vector transforms in both directions at the bounds of test_gpu_transforms (FP64 1e-11; FP32 2e-6
    scalar, 2e-5 vector)."""
    import gfsdc
    monkeypatch.delenv("GFSDC_FFT_NF", raising=False)
    if width != "default":
        monkeypatch.setenv("GFSDC_FFT_NF", width)
    nlon, nlat, T = grid
    nf = 5
    o = O.Sht(nlon, nlat, T)
    rng = np.random.default_rng(nlon)
    q = np.maximum(o.degree, 1.0) ** -1.5 * np.exp(2j * np.pi * rng.random((2, nf, o.nlm)))
    q[..., o.order == 0] = q[..., o.order == 0].real
    vrt, div = 1e-5 * q[0], 1e-6 * q[1]
    grid_o, (u0, v0) = o.spectogrd(q[0]), o.getuv(vrt, div, A)
    z0, d0 = o.getvrtdivspec(u0, v0, A)
    for prec, dt, ts, tv in ((gfsdc.FP64, 0, 1e-11, 1e-11), (gfsdc.FP32, 1, 2e-6, 2e-5)):
        g = gfsdc.Context(nlon, nlat, T, prec)
        u, v = g.getuv(vrt, div, A, dt)
        z, d = g.getvrtdivspec(u0, v0, A, dt)
        s = max(np.abs(z0).max(), np.abs(d0).max())
        for name, x, ref, scale, tol in (("spectogrd", g.spectogrd(q[0], dt), grid_o, None, ts),
                                         ("grdtospec", g.grdtospec(grid_o, dt), o.grdtospec(grid_o), None, ts),
                                         ("u", u, u0, None, tv), ("v", v, v0, None, tv), ("vrt", z, z0, s, tv),
                                         ("div", d, d0, s, tv)):
            e = np.abs(x - ref).max() / (scale or np.abs(ref).max())
            assert e < tol, (name, prec, e)
