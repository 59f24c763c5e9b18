"""Kernels at the sizes where their tiling can go wrong: partial tiles,
remainders, the smallest and the largest of their range."""
import ctypes as C

import numpy as np
import pytest

import levels
import oracle as O

pytestmark = pytest.mark.gpu


# hidden and output widths on and off the 32-wide layout tiles; batches of one, three and 16 split slices
@pytest.mark.parametrize("nlev,hidden,nlay,batch", [(20, 64, 2, 100), (21, 32, 1, 700), (33, 96, 3, 4096)])
def test_mlp_layout_and_gradient(nlev, hidden, nlay, batch):
    """Parameters come back bit for bit as they went in, and the gradient
    equals the bf16-storage oracle's (FP32 sums and neighbouring bf16
    roundings: 6e-3 relative L2, as for the tile-sized networks)."""
    import gfsdc
    ak, bk = levels.hybrid_levels(nlev)
    g = gfsdc.Context(64, 32, 21, gfsdc.FP32, nlev=nlev, ak=ak, bk=bk, dt=1200.0, ntrac=1,
                      physics=gfsdc.PHYS_SIMPLE)
    g.mlp_init(hidden, nlay, maxbatch=batch, capacity=16, seed=2)
    rng = np.random.default_rng(nlev)
    p = (0.1 * rng.standard_normal(g.mlp_params().size)).astype(np.float32)
    g.mlp_params(set=p)
    assert np.array_equal(g.mlp_params(), p)
    x = rng.standard_normal((batch, g.mlp_nin)).astype(np.float32)
    t = rng.standard_normal((batch, g.mlp_nout)).astype(np.float32)
    grad, loss = g.mlp_grad(x, t)
    lo, go, _ = O.Mlp(g.mlp_nin, g.mlp_nout, hidden, nlay).loss_grad(p, x, t, grad=True, bf16=True)
    assert abs(loss - lo) < 1e-3 * lo
    assert np.linalg.norm(grad - go) < 6e-3 * np.linalg.norm(go)


# every transform length with kernels of its own but the three of test_gpu_transforms, and two without (72, 162)
GRIDS = [(64, 32, 21), (96, 48, 31), (192, 94, 62), (256, 128, 84), (288, 144, 95), (512, 256, 170), (576, 288, 190),
         (72, 36, 23), (162, 82, 53)]
A = 6.3712e6


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def device_call(g, fn, ins, outs, nf, *extra, shift=0):
    """fn of the C ABI on device buffers of the context's own type, from the HIP runtime that libgfsdc links; each
    output, of the shapes and types in outs, starts shift bytes past an allocation's start"""
    import gfsdc
    L, H = gfsdc.load(), C.CDLL("libamdhip64.so.7")
    H.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    H.hipFree.argtypes = [C.c_void_p]
    H.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    ins = [np.ascontiguousarray(x) for x in ins]
    res = [np.full(s, np.nan, t) for s, t in outs]
    buf = []
    try:
        for x, off in [(x, 0) for x in ins] + [(x, shift) for x in res]:
            p = C.c_void_p()
            assert H.hipMalloc(C.byref(p), x.nbytes + off) == 0
            buf.append((p, C.c_void_p(p.value + off)))
            assert H.hipMemcpy(buf[-1][1], x.ctypes.data, x.nbytes, 1) == 0
        dt = gfsdc.DT_F64 if g.precision == gfsdc.FP64 else gfsdc.DT_F32
        assert getattr(L, fn)(g.h, *[q for _, q in buf], nf, *extra, dt, gfsdc.DEVICE) == 0
        g.sync()
        for x, (_, q) in zip(res, buf[len(ins):]):
            assert H.hipMemcpy(x.ctypes.data, q, x.nbytes, 2) == 0
    finally:
        for p, _ in buf:
            H.hipFree(p)
    return res


# the transposing gather and scatter hold 32 (FP64: 16) fields a tile and 64 coefficients
@pytest.mark.parametrize("nf", [1, 33, 64])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: f"{g[0]}x{g[1]}")
def test_transforms_every_length(grid, nf, monkeypatch):
    """Scalar and vector transforms, both directions, against the oracle at the bounds of test_gpu_transforms
    (FP64 1e-11; FP32 2e-6 scalar, 2e-5 vector), and the same call on device buffers, aligned and off a 16-byte
    boundary, bit for bit. One batch each with the default, 8 and 2 fields per Fourier workgroup."""
    import gfsdc
    if nf > 1:
        monkeypatch.setenv("GFSDC_FFT_NF", "8" if nf == 33 else "2")
    nlon, nlat, T = grid
    o = O.Sht(nlon, nlat, T)
    rng = np.random.default_rng(nf)
    n = np.maximum(o.degree, 1).astype(float)
    q = n ** -1.5 * np.exp(2j * np.pi * rng.random((2, nf, o.nlm)))
    q[..., o.order == 0] = q[..., o.order == 0].real
    vrt, div = 1e-5 * q[0], 1e-6 * q[1]
    grid_o, (u0, v0), (gx0, gy0) = o.spectogrd(q[0]), o.getuv(vrt, div, A), o.getgrad(q[0], A)
    z0, d0 = o.getvrtdivspec(u0, v0, A)
    for prec, ts, tv in ((gfsdc.FP64, 1e-11, 1e-11), (gfsdc.FP32, 2e-6, 2e-5)):
        g, dt = gfsdc.Context(nlon, nlat, T, prec), 0 if prec == gfsdc.FP64 else 1
        ct, rt = (np.complex64, np.float32) if dt else (np.complex128, np.float64)
        S, G = ((nf, o.nlm), ct), ((nf, nlat, nlon), rt)
        a, b, w, g0, uu, vv = (x.astype(t) for x, t in ((q[0], ct), (vrt, ct), (div, ct), (grid_o, rt), (u0, rt), (v0, rt)))
        scale = max(np.abs(z0).max(), np.abs(d0).max())
        for fn, ins, outs, ref, host, tol in (
                ("gfsdc_spectogrd", [a], [G], [grid_o], [g.spectogrd(a, dt)], ts),
                ("gfsdc_grdtospec", [g0], [S], [o.grdtospec(grid_o)], [g.grdtospec(g0, dt)], ts),
                ("gfsdc_getuv", [b, w], [G, G], [u0, v0], g.getuv(b, w, A, dt), tv),
                ("gfsdc_getgrad", [a], [G, G], [gx0, gy0], g.getgrad(a, A, dt), tv),
                ("gfsdc_getvrtdivspec", [uu, vv], [S, S], [z0, d0], g.getvrtdivspec(uu, vv, A, dt), tv)):
            for r, h in zip(ref, host):
                s = scale if fn == "gfsdc_getvrtdivspec" else np.abs(r).max()
                assert np.abs(h - r).max() < tol * s, (fn, prec, np.abs(h - r).max() / s)
            extra = () if fn in ("gfsdc_spectogrd", "gfsdc_grdtospec") else (C.c_double(A),)
            for shift in (0, rt().itemsize):
                for x, h in zip(device_call(g, fn, ins, outs, nf, *extra, shift=shift), host):
                    assert np.array_equal(x, h), (fn, prec, shift)


# chunks of layers: one per thread, most empty, partial, full and half full ones; a member's columns on and off the
# 64 (FP64: 32) of a workgroup; T170 has the columns for which a getdyntend call takes one thread per column in FP32,
# T84 those (of two members) for which a pass without tracers does in FP64
@pytest.mark.parametrize("grid,nlev,ntrac", [((64, 32, 21), 2, 1), ((64, 32, 21), 7, 0), ((72, 36, 23), 17, 2),
                                             ((72, 36, 23), 32, 1), ((64, 32, 21), 33, 1), ((72, 36, 23), 63, 0),
                                             ((64, 32, 21), 64, 2), ((512, 256, 170), 5, 1),
                                             ((256, 128, 84), 5, 0), ((256, 128, 84), 18, 0)])
def test_columns_every_chunk(grid, nlev, ntrac):
    """Tendencies, omega/p and etadot grids of getdyntend and of its inverse-only form, two members, against the
    oracle at the bounds of test_gpu_dycore (FP64 1e-9, FP32 2e-4)."""
    import cases
    import gfsdc
    nlon, nlat, T = grid
    ak, bk = levels.hybrid_levels(nlev)
    o = O.Model(nlon, nlat, T, nlev, ak, bk, 600.0, ntrac=ntrac)
    st = []
    for mem in range(2):
        vrt, div, tv, lnps = cases.perturbed_state(o.sht.degree, o.sht.order, nlev, seed=3 + mem, amp=0.3)
        q = np.zeros((ntrac, nlev, o.sht.nlm), complex)
        for t in range(ntrac):
            q[t] = 1e-4 * cases.perturbed_state(o.sht.degree, o.sht.order, nlev, seed=9 + t + mem, amp=1.0)[2][0]
            q[t, :, 0] = 0.01 * np.linspace(1.0, 0.2, nlev) * np.sqrt(4 * np.pi)
        st.append((vrt[0], div[0], tv[0], lnps[0], q))
    for prec, tol in ((gfsdc.FP64, 1e-9), (gfsdc.FP32, 2e-4)):
        g = gfsdc.Context(nlon, nlat, T, prec, nlev=nlev, ak=ak, bk=bk, dt=600.0, ntrac=ntrac, nmem=2)
        a = [np.stack(x) for x in zip(*st)]
        g.set_state(a[0], a[1], a[2], a[3], trac=a[4] if ntrac else None)
        for inverse in (False, True):
            tg = g.getdyntend(1, inverse_only=inverse)
            grids = {k: g.grid(k) for k in ("dlnpdtg", "etadot", "psg", "dlnpsdt")}
            for mem in range(2):
                o.set_state(st[mem][0], st[mem][1], st[mem][2], st[mem][3], *([st[mem][4]] if ntrac else []))
                to = o.getdyntend(1)
                for k in () if inverse else ("dvrt", "ddiv", "dtv", "dlnps") + (("dtrac",) if ntrac else ()):
                    assert rel(tg[k][mem], to[k]) < tol, (prec, k, mem, rel(tg[k][mem], to[k]))
                for k, x in grids.items():
                    assert rel(x[mem], o.grid(k)) < tol, (prec, inverse, k, mem, rel(x[mem], o.grid(k)))


# coefficients and state fields on and off the 64 x 32 (FP64: 64 x 16) tiles of the packing kernel
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid,nlev,ntrac,nmem", [((64, 32, 21), 5, 2, 3), ((96, 48, 30), 21, 0, 1), ((72, 36, 23), 20, 1, 2)])
def test_state_packing(grid, nlev, ntrac, nmem, prec):
    """A state comes back bit for bit through host and through device buffers, whole and with field runs left out."""
    import gfsdc
    nlon, nlat, T = grid
    ak, bk = levels.hybrid_levels(nlev)
    p = gfsdc.FP64 if prec == "fp64" else gfsdc.FP32
    ct = np.complex128 if prec == "fp64" else np.complex64
    dt = gfsdc.DT_F64 if prec == "fp64" else gfsdc.DT_F32
    g = gfsdc.Context(nlon, nlat, T, p, nlev=nlev, ak=ak, bk=bk, dt=600.0, ntrac=ntrac, nmem=nmem)
    rng = np.random.default_rng(1)
    shapes = [(nmem, nlev, g.nlm)] * 3 + [(nmem, ntrac, nlev, g.nlm), (nmem, g.nlm)]
    x = [(rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64).astype(ct) for s in shapes]
    g.set_state(x[0], x[1], x[2], x[4], trac=x[3] if ntrac else None)
    st = g.get_state()
    for k, v in zip(("vrt", "div", "tv", "trac", "lnps"), x):
        assert np.array_equal(st[k], v), k
    # device buffers: the second state without its div and lnps, then everything back but tv
    L, H = gfsdc.load(), C.CDLL("libamdhip64.so.7")
    H.hipMalloc.argtypes, H.hipFree.argtypes = [C.POINTER(C.c_void_p), C.c_size_t], [C.c_void_p]
    H.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    y = [np.ascontiguousarray(2 * v) for v in x]
    d = [C.c_void_p() for _ in y]
    try:
        for q, v in zip(d, y):
            assert H.hipMalloc(C.byref(q), max(v.nbytes, 16)) == 0 and H.hipMemcpy(q, v.ctypes.data, v.nbytes, 1) == 0
        assert L.gfsdc_set_state(g.h, d[0], None, d[2], d[3], None, dt, gfsdc.DEVICE) == 0
        for q, v in zip(d, y):
            assert H.hipMemcpy(q, np.zeros_like(v).ctypes.data, v.nbytes, 1) == 0
        assert L.gfsdc_get_state(g.h, d[0], d[1], None, d[3], d[4], dt, gfsdc.DEVICE) == 0
        g.sync()
        for i, want in enumerate((y[0], x[1], None, y[3], x[4])):
            got = np.empty_like(y[i])
            assert H.hipMemcpy(got.ctypes.data, d[i], got.nbytes, 2) == 0
            assert np.array_equal(got, want if want is not None else np.zeros_like(got)), i
    finally:
        for q in d:
            H.hipFree(q)


# partial latitude, degree and column tiles (64 x 64 x 128 values), partial k chunks of 32, several column tiles
@pytest.mark.parametrize("grid,nf", [((64, 32, 21), 1), ((72, 36, 23), 65), ((192, 94, 62), 33), ((288, 144, 95), 64),
                                     ((384, 190, 126), 5)])
def test_bf16x3_tiles(grid, nf):
    """BF16X3 transforms against the oracle at the bounds of test_gpu_transforms (3e-5)."""
    import gfsdc
    nlon, nlat, T = grid
    o, g = O.Sht(nlon, nlat, T), gfsdc.Context(nlon, nlat, T, gfsdc.BF16X3)
    rng = np.random.default_rng(nf)
    q = np.maximum(o.degree, 1) ** -1.5 * np.exp(2j * np.pi * rng.random((nf, o.nlm)))
    q[:, o.order == 0] = q[:, o.order == 0].real
    ref = o.spectogrd(q)
    assert rel(g.spectogrd(q.astype(np.complex64), dtype=1), ref) < 3e-5
    assert rel(g.grdtospec(ref.astype(np.float32), dtype=1), o.grdtospec(ref)) < 3e-5


# levels below, on and past the 16 of a round; a member's columns on and off the 16 of a workgroup
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid,nlev,turb", [((64, 32, 21), 2, 1), ((36, 18, 11), 15, 1), ((72, 36, 23), 16, 0),
                                            ((36, 18, 11), 17, 1), ((64, 32, 21), 33, 1), ((36, 18, 11), 64, 1),
                                            ((64, 32, 21), 64, 0)])
def test_simple_columns_every_round(grid, nlev, turb, prec):
    """Simple physics of two members against the oracle at the bounds of test_gpu_moist (FP64 1e-9 of the largest
    value, FP32 2e-3 in the 2-norm: a point at saturation may condense on one side alone)."""
    import cases
    import gfsdc
    nlon, nlat, T = grid
    ak, bk = levels.hybrid_levels(nlev)
    kw = dict(ntrac=1, physics=2, simple_test=2, turbflux=turb)
    o = O.Model(nlon, nlat, T, nlev, ak, bk, 600.0, **kw)
    p = gfsdc.FP64 if prec == "fp64" else gfsdc.FP32
    g = gfsdc.Context(nlon, nlat, T, p, nlev=nlev, ak=ak, bk=bk, dt=600.0, nmem=2, **kw)
    st = []
    for mem in range(2):
        vrt, div, tv, lnps = cases.perturbed_state(o.sht.degree, o.sht.order, nlev, seed=3 + mem, amp=0.5)
        q = o.sht.grdtospec(cases.moist_grid(o.sht.lats, nlon, ak, bk, seed=5 + mem))
        st.append((vrt[0], div[0], tv[0], lnps[0], q[None]))
    a = [np.stack(x) for x in zip(*st)]
    g.set_state(a[0], a[1], a[2], a[3], trac=a[4])
    g.getdyntend(3, inverse_only=True)
    tg = g.simple_phytend()
    far, tol = (rel, 1e-9) if prec == "fp64" else (lambda x, y: np.linalg.norm(x - y) / max(np.linalg.norm(y), 1e-300), 2e-3)
    for mem in range(2):
        o.set_state(st[mem][0], st[mem][1], st[mem][2], st[mem][3], st[mem][4])
        o.getdyntend(3, inverse_only=True)
        to = o.simple_phytend()
        pairs = {k: (tg[k][mem], to[k]) for k in ("dvrt", "ddiv", "dtv", "dtrac")}
        pairs |= {k: (g.grid(k)[mem].ravel(), o.grid(k).ravel()) for k in ("precip", "pwat")}
        for k, (x, y) in pairs.items():
            if np.abs(y).max() > 0:
                assert far(x, y) < tol, (k, mem, far(x, y))
            else:  # two layers do not condense; without the boundary layer the wind is untouched
                assert np.abs(x).max() == 0, (k, mem)


# columns of a member: fewer than a round of the 128 workgroups, a little over one, over four; one member to seven
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid,nlev,nmem", [((36, 18, 11), 5, 7), ((256, 130, 84), 20, 2), ((576, 288, 190), 3, 1),
                                            ((64, 32, 21), 64, 3)])
def test_area_sums(grid, nlev, nmem, prec):
    """Dry mass of each member against the oracle at the bounds of test_gpu_moist (FP64 1e-9, FP32 2e-6), again after
    the next state, and lean steps (ps, its range and its mean in one launch) equal to full ones bit for bit."""
    import cases
    import gfsdc
    nlon, nlat, T = grid
    ak, bk = levels.hybrid_levels(nlev)
    o = O.Model(nlon, nlat, T, nlev, ak, bk, 300.0, physics=1, massfix=1)
    p = gfsdc.FP64 if prec == "fp64" else gfsdc.FP32
    a, b = (gfsdc.Context(nlon, nlat, T, p, nlev=nlev, ak=ak, bk=bk, dt=300.0, nmem=nmem, physics=1, massfix=1)
            for _ in range(2))
    for turn in range(2):
        st = [cases.perturbed_state(o.sht.degree, o.sht.order, nlev, seed=3 + m + nmem * turn, amp=0.2)
              for m in range(nmem)]
        x = [np.concatenate(v) for v in zip(*st)]
        for g in (a, b):
            g.set_state(*x)
            g.pdryini = np.zeros(nmem)
        a.advance(3, use_graph=turn == 0)
        for _ in range(3):
            b.advance(1, use_graph=turn == 0)
        sa, sb = a.get_state(), b.get_state()
        for k in ("vrt", "div", "tv", "lnps"):
            assert np.isfinite(sa[k]).all() and np.array_equal(sa[k], sb[k]), (turn, k)
        for m in range(nmem):
            o.pdryini = 0.0
            o.set_state(*(v[m] for v in x))
            o.getdyntend(1)
            for g in (a, b):
                assert abs(g.pdryini[m] - o.pdryini) < (1e-9 if prec == "fp64" else 2e-6) * o.pdryini, (turn, m)


# fields in host memory below, at and past the megabyte that goes through pinned memory: the grids alone past it, both
@pytest.mark.parametrize("prec,nf", [("fp64", 1), ("fp64", 64), ("fp64", 65), ("fp64", 270), ("fp32", 128), ("fp32", 129)])
def test_small_host_fields(prec, nf):
    """Host calls equal the calls on device buffers bit for bit, two after each other with different fields, and with
    the other element type they stay within its rounding of them."""
    import gfsdc
    nlon, nlat, T = 64, 32, 21
    g = gfsdc.Context(nlon, nlat, T, gfsdc.FP64 if prec == "fp64" else gfsdc.FP32)
    dt, ct, rt = (0, np.complex128, np.float64) if prec == "fp64" else (1, np.complex64, np.float32)
    S, G = ((nf, g.nlm), ct), ((nf, nlat, nlon), rt)
    rng = np.random.default_rng(nf)
    x = rng.standard_normal((4, nf, g.nlm)) + 1j * rng.standard_normal((4, nf, g.nlm))
    x[..., g.order == 0] = x[..., g.order == 0].real
    y = rng.standard_normal((4, nf, nlat, nlon)).astype(rt)
    a = x.astype(ct)
    for i in (0, 1):
        host = [[g.spectogrd(a[i], dt)], [g.grdtospec(y[i], dt)], g.getuv(a[i], a[i + 2], A, dt),
                g.getvrtdivspec(y[i], y[i + 2], A, dt)]
        dev = [device_call(g, "gfsdc_spectogrd", [a[i]], [G], nf), device_call(g, "gfsdc_grdtospec", [y[i]], [S], nf),
               device_call(g, "gfsdc_getuv", [a[i], a[i + 2]], [G, G], nf, C.c_double(A)),
               device_call(g, "gfsdc_getvrtdivspec", [y[i], y[i + 2]], [S, S], nf, C.c_double(A))]
        for p, q in zip(host, dev):
            for u, v in zip(p, q):
                assert np.array_equal(u, v), i
        other = g.spectogrd(a[i].astype(np.complex64 if dt == 0 else np.complex128), 1 - dt)
        assert np.abs(other - host[0][0]).max() < 2e-6 * np.abs(host[0][0]).max()


# levels on both sides of the solve's 32 and 64 rows and of its blocks of 16; coefficients of a degree off the 8 of a tile
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nlev,ntrac,nmem", [(2, 0, 3), (16, 1, 1), (31, 0, 2), (32, 2, 1), (33, 0, 2), (47, 0, 1), (64, 1, 2)])
def test_solve_every_size(nlev, ntrac, nmem, prec):
    """One semi-implicit step of each member against the oracle at the bounds of test_gpu_moist (2-norm, FP64 1e-9,
    FP32 1e-4)."""
    import cases
    import gfsdc
    ak, bk = levels.hybrid_levels(nlev)
    o = O.Model(64, 32, 21, nlev, ak, bk, 600.0, ntrac=ntrac)
    p, tol = (gfsdc.FP64, 1e-9) if prec == "fp64" else (gfsdc.FP32, 1e-4)
    g = gfsdc.Context(64, 32, 21, p, nlev=nlev, ak=ak, bk=bk, dt=600.0, ntrac=ntrac, nmem=nmem)
    x = [np.concatenate(v) for v in zip(*(cases.perturbed_state(o.sht.degree, o.sht.order, nlev, seed=3 + m, amp=0.2)
                                          for m in range(nmem)))]
    q = np.zeros((nmem, ntrac, nlev, o.sht.nlm), complex)
    for t in range(ntrac):
        q[:, t] = 1e-4 * x[2]
        q[:, t, :, 0] = 0.01 * np.linspace(1.0, 0.2, nlev) * np.sqrt(4 * np.pi)
    g.set_state(*x, trac=q if ntrac else None)
    g.advance(1)
    sg = g.get_state()
    for m in range(nmem):
        o.pdryini = 0.0  # each member keeps its own dry mass
        o.set_state(*(v[m] for v in x), *([q[m]] if ntrac else []))
        o.advance(1)
        so = o.get_state()
        for k in ("vrt", "div", "tv", "lnps") + (("trac",) if ntrac else ()):
            e = np.linalg.norm(sg[k][m] - so[k]) / np.linalg.norm(so[k])
            assert e < tol, (k, m, e)
