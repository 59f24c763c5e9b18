"""The work whose speed counts, case by case.

A case is a dict of plain values. kind says which public entry point it calls:

  host       Context.spectogrd and grdtospec on host arrays, one field at a time:
             what a host model that keeps its fields in its own memory does
  synth      gfsdc_spectogrd on device buffers
  anal       gfsdc_grdtospec on device buffers
  roundtrip  gfsdc_spectogrd, then gfsdc_grdtospec of its grids
  getuv      gfsdc_getuv: vorticity and divergence to winds
  vrtdiv     gfsdc_getvrtdivspec: winds to vorticity and divergence
  grad       gfsdc_getgrad
  tend       gfsdc_set_state and gfsdc_getdyntend (stage 1) on device buffers
  advance    gfsdc_set_state, gfsdc_advance, gfsdc_get_state: a forecast of nsteps
             steps from a given state, replayed from a HIP graph
  mlp        gfsdc_mlp_grad: one gradient of the column network on host rows

Grids are the Gauss grids of spectral models (nlon x nlat, triangular
truncation T); prec is the context's precision.
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gfs-dycore_amd"))

import gfsdc  # noqa: E402
import levels  # noqa: E402

PREC = {"f64": gfsdc.FP64, "f32": gfsdc.FP32, "bf16x3": gfsdc.BF16X3}
RERTH = float(np.float32(6.3712e6))
# truncation -> (nlon, nlat)
GRID = {21: (64, 32), 30: (96, 48), 42: (128, 64), 62: (192, 94), 84: (256, 128), 126: (384, 190), 170: (512, 256),
        190: (576, 288), 254: (768, 384)}


def listed():
    return [
        # one field through host memory and back: a host model's smallest call, latency bound
        dict(name="host_t42_f64", kind="host", T=42, prec="f64", nf=1),
        # a handful of surface fields on a grid with no kernel of its own length
        dict(name="synth_t62_f32", kind="synth", T=62, prec="f32", nf=5),
        # one 3-D field of a reference-precision run to spectral space
        dict(name="anal_t126_f64", kind="anal", T=126, prec="f64", nf=64),
        # winds of an odd number of levels, another grid
        dict(name="vrtdiv_t170_f32", kind="vrtdiv", T=170, prec="f32", nf=33),
        # winds of a full model state in the split-precision option
        dict(name="getuv_t254_bf16x3", kind="getuv", T=254, prec="bf16x3", nf=64),
        # the transform microbenchmark's batch: 64 levels x 4 fields there and back
        dict(name="roundtrip_t254_f32", kind="roundtrip", T=254, prec="f32", nf=256),
        # one tendency evaluation for a host that does its own time stepping
        dict(name="tend_t126l64_f32", kind="tend", T=126, prec="f32", nlev=64, ntrac=0, nmem=1),
        # the small reference configuration, FP64, many cheap steps
        dict(name="run_t42l20_f64", kind="advance", T=42, prec="f64", nlev=20, ntrac=0, nmem=1, phys="hs", nsteps=12),
        # the headline: T254L64 dry run
        dict(name="run_t254l64_f32", kind="advance", T=254, prec="f32", nlev=64, ntrac=0, nmem=1, phys="hs", nsteps=6),
        # an ensemble in one launch, each member with its own stochastic pattern
        dict(name="ens16_t126l64_f32", kind="advance", T=126, prec="f32", nlev=64, ntrac=0, nmem=16, phys="hs_pattern",
             nsteps=3),
        # moist run: simple physics, one tracer
        dict(name="moist_t126l64_f32", kind="advance", T=126, prec="f32", nlev=64, ntrac=1, nmem=1, phys="simple",
             nsteps=4),
        # training the column network: the gradient of one batch
        dict(name="mlp_grad_4096", kind="mlp", nlev=64, hidden=512, layers=3, batch=4096),
    ]


def draw(rng):
    """A case of the ranges that the listed ones stand for."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["host", "synth", "anal", "roundtrip", "getuv", "vrtdiv", "grad", "tend", "advance", "advance",
                       "mlp"])
    if kind == "mlp":
        return dict(kind=kind, nlev=rng.randint(20, 64), hidden=32 * log_int(4, 16), layers=rng.randint(2, 3),
                    batch=log_int(64, 4096))
    T = rng.choice(sorted(GRID))
    if kind == "host":
        return dict(kind=kind, T=min(T, 126), prec=rng.choice(["f64", "f32"]), nf=rng.randint(1, 4))
    prec = rng.choice(["f64", "f32", "f32", "bf16x3"])
    if kind in ("synth", "anal", "roundtrip", "getuv", "vrtdiv", "grad"):
        most = 128 if kind in ("synth", "anal", "roundtrip") else 64
        return dict(kind=kind, T=T, prec=prec, nf=log_int(1, most if prec != "f64" else most // 2))
    prec = rng.choice(["f64", "f32"])
    phys = rng.choice(["hs", "hs", "hs_pattern", "simple"]) if kind == "advance" else "hs"
    ntrac = 1 if phys == "simple" else 0
    nmem = log_int(1, max(1, min(16, (190 // T) ** 2)))
    c = dict(kind=kind, T=T, prec=prec, nlev=rng.randint(20, 64), ntrac=ntrac, nmem=nmem)
    if kind == "advance":
        c.update(phys=phys, nsteps=rng.randint(1, 2) if T > 126 else rng.randint(2, 6))
    return c


# ---------------------------------------------------------------------------
# what a program has in hand before the call

def _sizes(case):
    T = case["T"]
    nlon, nlat = GRID[T]
    return T, nlon, nlat, (T + 1) * (T + 2) // 2


def _types(case):
    """(real, complex, element-type code) of the context's own precision"""
    if case["prec"] == "f64":
        return torch.float64, torch.complex128, gfsdc.DT_F64
    return torch.float32, torch.complex64, gfsdc.DT_F32


@functools.lru_cache(maxsize=1)
def _plan(T, prec):
    """The transform plan, made once as a program makes it."""
    nlon, nlat = GRID[T]
    return gfsdc.Context(nlon, nlat, T, PREC[prec])


@functools.lru_cache(maxsize=4)
def _mn(T):
    """degree and order of each coefficient, on the device"""
    m = np.concatenate([np.full(T + 1 - k, k) for k in range(T + 1)])
    n = np.concatenate([np.arange(k, T + 1) for k in range(T + 1)])
    return torch.from_numpy(n).cuda().double(), torch.from_numpy(m).cuda().double()


def _random_spec(gen, T, lead, slope, zero_mean=True):
    """Random coefficients (lead, nlm), amplitude n^slope, real at order 0, unit variance at degree 1."""
    n, m = _mn(T)
    x = torch.randn(tuple(lead) + (n.numel(), 2), generator=gen, device="cuda", dtype=torch.float64)
    x = torch.view_as_complex(x) * n.clamp(min=1.0) ** slope
    x = torch.where(m == 0, x.real.to(x.dtype), x)
    if zero_mean:
        x[..., 0] = 0
    return x


def _random_grid(gen, nf, nlat, nlon):
    """Grid fields: large waves of every field's own, and small-scale noise, as products of model fields have."""
    lon = torch.arange(nlon, device="cuda", dtype=torch.float64) * (2 * math.pi / nlon)
    col = (torch.arange(nlat, device="cuda", dtype=torch.float64) + 0.5) * (math.pi / nlat)
    g = 0.1 * torch.randn(nf, nlat, nlon, generator=gen, device="cuda", dtype=torch.float64)
    a = torch.randn(nf, 6, 2, generator=gen, device="cuda", dtype=torch.float64)
    for k in range(6):
        w = torch.sin(col)[:, None] ** k * torch.cos((k + 1) * col)[:, None]
        g += a[:, k, 0, None, None] * w * torch.cos(k * lon) + a[:, k, 1, None, None] * w * torch.sin(k * lon)
    return g


def _vert(nlev):
    """(ak, bk) of nlev layers: sigma for the shallow set, hybrid for the deep ones"""
    return levels.sigma_levels(nlev) if nlev <= 20 else levels.hybrid_levels(nlev)


def _column_spec(gen, T, lead, nl):
    """Random coefficients (lead, nl, nlm) of slowly varying levels: four vertical modes, flat to degree 8 and falling as
    n^-1.5 beyond it."""
    n, _ = _mn(T)
    z = (torch.arange(nl, device="cuda", dtype=torch.float64) + 0.5) / nl
    x = 0
    for k in range(4):
        x = x + torch.cos(math.pi * k * z)[:, None] / (1 + k) * _random_spec(gen, T, lead, 0.0)[..., None, :]
    return x * (n / 8).clamp(min=1.0) ** -1.5


def _state(case, seed):
    """A model state in 64 bits: solid-body westerlies, random vorticity, divergence a twentieth of it, a temperature that
    falls with height and towards the poles, a gentle surface pressure, and humidity that dries upward."""
    T, nlon, nlat, nlm = _sizes(case)
    nl, nm, ntr = case["nlev"], case["nmem"], case["ntrac"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ak, bk = _vert(nl)
    p = torch.from_numpy(np.ascontiguousarray(((ak + 1e5 * bk)[:-1] + (ak + 1e5 * bk)[1:])[::-1] / 2e5)).cuda()
    root = math.sqrt(4 * math.pi)
    vrt = _column_spec(gen, T, (nm,), nl) * 2e-6
    vrt[..., 1] += 2 * 10.0 / RERTH * root / math.sqrt(3.0)  # (m, n) = (0, 1)
    div = _column_spec(gen, T, (nm,), nl) * 1e-7
    tv = _column_spec(gen, T, (nm,), nl) * 0.3
    tv[..., 0] += torch.clamp(288.0 * p ** 0.19, min=215.0) * root
    tv[..., 2] -= 8.0 * p  # (0, 2): warm equator
    lnps = _random_spec(gen, T, (nm,), -1.5) * 1e-3
    lnps[..., 0] = math.log(1e5) * root
    q = None
    if ntr:
        q = _column_spec(gen, T, (nm, ntr), nl) * 2e-4 * (p ** 3)[:, None]
        q[..., 0] += 9e-3 * p ** 3 * root
        q[..., 2] -= 4e-3 * p ** 3
    return dict(vrt=vrt, div=div, tv=tv, lnps=lnps, trac=q)


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _ok(rc):
    if rc:
        raise gfsdc.GfsdcError(gfsdc.load().gfsdc_last_error().decode())


def _mlp_data(case, seed):
    """Normalised rows, targets and He-scaled parameters."""
    nin, nout, h, nh, b = 4 * case["nlev"] + 3, 4 * case["nlev"], case["hidden"], case["layers"], case["batch"]
    rng = np.random.default_rng(seed)
    dims = [nin] + [h] * nh + [nout]
    parts = []
    for i, o in zip(dims[:-1], dims[1:]):
        parts += [rng.standard_normal(i * o) * math.sqrt(2.0 / i), 0.05 * rng.standard_normal(o)]
    x = rng.standard_normal((b, nin)).astype(np.float32)
    t = (rng.standard_normal((b, nout)) + x[:, :nout]).astype(np.float32)
    return dims, x, t, np.concatenate(parts).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "mlp":
        ak, bk = _vert(case["nlev"])
        s["ctx"] = gfsdc.Context(128, 64, 42, gfsdc.FP32, nlev=case["nlev"], ak=ak, bk=bk, dt=1200.0, ntrac=1,
                                 physics=gfsdc.PHYS_SIMPLE)
        s["ctx"].mlp_init(case["hidden"], case["layers"], maxbatch=case["batch"], capacity=1024, seed=1)
        _, s["x"], s["t"], w = _mlp_data(case, seed)
        s["ctx"].mlp_params(set=w)
        return s
    T, nlon, nlat, nlm = _sizes(case)
    real, cplx, _ = _types(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind == "host":
        s["ctx"] = _plan(T, case["prec"])
        s["spec"] = _random_spec(gen, T, (case["nf"],), -1.5, False).cpu().numpy()
    elif kind in ("tend", "advance"):
        ak, bk = _vert(case["nlev"])
        kw = dict(physics=gfsdc.PHYS_HS)
        if case.get("phys") == "hs_pattern":
            kw.update(tpat_amp=0.5, tpat_tau=6 * 3600.0, tpat_lscale=500.0e3, tpat_seed=1 + seed % 1000)
        elif case.get("phys") == "simple":
            kw.update(physics=gfsdc.PHYS_SIMPLE, simple_test=2, turbflux=1)
        ctx = gfsdc.Context(nlon, nlat, T, PREC[case["prec"]], nlev=case["nlev"], ak=ak, bk=bk,
                            dt=1200.0 if T <= 62 else 600.0, ntrac=case["ntrac"], nmem=case["nmem"], **kw)
        st = {k: None if v is None else v.to(cplx).contiguous() for k, v in _state(case, seed).items()}
        s.update(ctx=ctx, st=st, out={k: None if v is None else torch.empty_like(v) for k, v in st.items()})
    else:
        s["ctx"] = _plan(T, case["prec"])
        nf = case["nf"]
        pair = kind in ("getuv", "vrtdiv")
        if kind in ("anal", "vrtdiv"):
            s["in"] = [_random_grid(gen, nf, nlat, nlon).to(real) for _ in range(2 if pair else 1)]
        else:
            amp, slope = (1e-5, -0.5) if kind == "getuv" else (1.0, -1.5)
            s["in"] = [(amp * _random_spec(gen, T, (nf,), slope, kind == "getuv")).to(cplx) for _ in range(2 if pair else 1)]
        spec = [torch.empty(nf, nlm, dtype=cplx, device="cuda") for _ in range(2)]
        grid = [torch.empty(nf, nlat, nlon, dtype=real, device="cuda") for _ in range(2)]
        s["out"] = {"synth": grid[:1], "anal": spec[:1], "roundtrip": [grid[0], spec[0]], "getuv": grid,
                    "vrtdiv": spec, "grad": grid}[kind]
    torch.cuda.synchronize()
    return s


def run(s):
    case, ctx, L = s["case"], s["ctx"], gfsdc.load()
    kind = case["kind"]
    if kind == "host":
        t = gfsdc.DT_F64 if case["prec"] == "f64" else gfsdc.DT_F32
        grid = ctx.spectogrd(s["spec"], t)
        return [grid, ctx.grdtospec(grid, t)]
    if kind == "mlp":
        return list(ctx.mlp_grad(s["x"], s["t"]))
    dt, dev, o = _types(case)[2], gfsdc.DEVICE, s["out"]
    if kind in ("tend", "advance"):
        st = s["st"]
        _ok(L.gfsdc_set_state(ctx.h, _ptr(st["vrt"]), _ptr(st["div"]), _ptr(st["tv"]), _ptr(st["trac"]), _ptr(st["lnps"]),
                              dt, dev))
        if kind == "advance":
            _ok(L.gfsdc_advance(ctx.h, case["nsteps"], 1))
            _ok(L.gfsdc_get_state(ctx.h, _ptr(o["vrt"]), _ptr(o["div"]), _ptr(o["tv"]), _ptr(o["trac"]), _ptr(o["lnps"]),
                                  dt, dev))
        else:
            _ok(L.gfsdc_getdyntend(ctx.h, 1, 0, _ptr(o["vrt"]), _ptr(o["div"]), _ptr(o["tv"]), _ptr(o["trac"]),
                                   _ptr(o["lnps"]), dt, dev))
        return [o[k] for k in ("vrt", "div", "tv", "lnps", "trac") if o[k] is not None]
    i, nf = s["in"], case["nf"]
    if kind == "synth":
        _ok(L.gfsdc_spectogrd(ctx.h, _ptr(i[0]), _ptr(o[0]), nf, dt, dev))
    elif kind == "anal":
        _ok(L.gfsdc_grdtospec(ctx.h, _ptr(i[0]), _ptr(o[0]), nf, dt, dev))
    elif kind == "roundtrip":
        _ok(L.gfsdc_spectogrd(ctx.h, _ptr(i[0]), _ptr(o[0]), nf, dt, dev))
        _ok(L.gfsdc_grdtospec(ctx.h, _ptr(o[0]), _ptr(o[1]), nf, dt, dev))
    elif kind == "getuv":
        _ok(L.gfsdc_getuv(ctx.h, _ptr(i[0]), _ptr(i[1]), _ptr(o[0]), _ptr(o[1]), nf, RERTH, dt, dev))
    elif kind == "vrtdiv":
        _ok(L.gfsdc_getvrtdivspec(ctx.h, _ptr(i[0]), _ptr(i[1]), _ptr(o[0]), _ptr(o[1]), nf, RERTH, dt, dev))
    else:
        _ok(L.gfsdc_getgrad(ctx.h, _ptr(i[0]), _ptr(o[0]), _ptr(o[1]), nf, RERTH, dt, dev))
    return o


def work(case):
    """Bytes: inputs, outputs and the Legendre functions, each once. Flops: the Legendre contractions (2 nlat nlm a field
    and direction), the Fourier transforms and, where it has them, the level operators or the network's products."""
    if case["kind"] == "mlp":
        nin, nout, h, nh, b = 4 * case["nlev"] + 3, 4 * case["nlev"], case["hidden"], case["layers"], case["batch"]
        w = nin * h + (nh - 1) * h * h + h * nout
        return {"bytes": 4.0 * (b * (nin + nout) + 2 * w), "flops": 6.0 * b * w - 2.0 * b * nin * h}
    T, nlon, nlat, nlm = _sizes(case)
    e = 8 if case["prec"] == "f64" else 4
    table = e * (nlat // 2) * (nlm + T + 1)
    spec, grid = 2 * e * nlm, e * nlat * nlon
    one = 2.0 * nlat * nlm + 2.5 * nlon * math.log2(nlon) * nlat  # one scalar field, one direction
    kind = case["kind"]
    if kind in ("tend", "advance"):
        nl, nm, ntr = case["nlev"], case["nmem"], case["ntrac"]
        state = nm * spec * ((3 + ntr) * nl + 1)
        tend = nm * one * ((7 + 3 * ntr) * nl + 3 + (4 + ntr) * nl + 1)
        if kind == "tend":
            return {"bytes": 2.0 * state + table, "flops": tend}
        phys = nm * one * (2 * (nl + 1) if ntr == 0 else (5 + ntr) * nl + 3 + 4 * nl + 1)
        return {"bytes": 2.0 * state + table,
                "flops": case["nsteps"] * (3 * tend + phys + 3 * 20.0 * nl * nl * nlm * nm)}
    nf = case["nf"] * {"getuv": 2, "vrtdiv": 2, "grad": 2}.get(kind, 1)
    if kind in ("host", "roundtrip"):
        return {"bytes": 2.0 * nf * (spec + grid) + table, "flops": 2 * nf * one}
    nin = case["nf"] if kind == "grad" else nf
    return {"bytes": float(nin * (grid if kind in ("anal", "vrtdiv") else spec) +
                           nf * (spec if kind in ("anal", "vrtdiv") else grid) + table), "flops": nf * one}


# ---------------------------------------------------------------------------
# the same results in 64 bits, from the mathematics alone

class _Sphere:
    """Gauss grid, orthonormal associated Legendre functions P and H = cos(lat) dP/dlat, and dense Fourier sums."""

    def __init__(self, T):
        self.T = T
        self.nlon, self.nlat = nlon, nlat = GRID[T]
        th = np.pi * (np.arange(nlat) + 0.75) / (nlat + 0.5)
        for _ in range(6):
            x = np.cos(th)
            p0, p1 = np.ones(nlat), x
            for k in range(2, nlat + 1):
                p0, p1 = p1, ((2 * k - 1) * x * p1 - (k - 1) * p0) / k
            th = th + p1 * np.sin(th) / (nlat * (p0 - x * p1))
        w = 2 * (np.sin(th) / (nlat * p0)) ** 2
        mu, cs = torch.from_numpy(np.cos(th)).cuda(), torch.from_numpy(np.sin(th)).cuda()
        self.mu, self.cos, self.w = mu, cs, torch.from_numpy(w).cuda()
        m = torch.arange(T + 1, device="cuda", dtype=torch.float64)

        def eps(n):  # by order, at degree n
            return torch.where(n > m, torch.sqrt(((n * n - m * m) / (4 * n * n - 1)).clamp(min=0.0)), torch.zeros_like(m))

        fac = torch.cumsum(torch.cat([m.new_zeros(1), 0.5 * torch.log((2 * m[1:] + 1) / (2 * m[1:]))]), 0)
        pmm = torch.exp(fac[:, None] + m[:, None] * torch.log(cs)) * math.sqrt(1 / (4 * math.pi))
        P = torch.zeros(T + 1, T + 3, nlat, device="cuda", dtype=torch.float64)
        for n in range(T + 2):  # every order m <= n at once
            if n:
                r = mu * P[:, n - 1] - (eps(float(n - 1))[:, None] * P[:, n - 2] if n > 1 else 0.0)
                e = eps(float(n))
                P[:, n] = torch.where((m < n)[:, None], r / torch.where(e > 0, e, torch.ones_like(e))[:, None], P[:, n])
            if n <= T:
                P[n, n] = pmm[n]
        H = torch.zeros(T + 1, T + 1, nlat, device="cuda", dtype=torch.float64)
        for n in range(T + 1):
            H[:, n] = -n * eps(float(n + 1))[:, None] * P[:, n + 1]
            if n:
                H[:, n] += (n + 1) * eps(float(n))[:, None] * P[:, n - 1]
        self.P, self.H = P[:, :T + 1].contiguous(), H
        ang = (torch.arange(nlon, device="cuda")[None, :] * torch.arange(T + 1, device="cuda")[:, None] % nlon).double()
        ang = ang * (2 * math.pi / nlon)
        self.c, self.s = torch.cos(ang), torch.sin(ang)  # (m, lon)
        self.n, self.m = _mn(T)
        self.im = 1j * m
        self.at = (self.m.long() * (T + 1) + self.n.long())

    def dense(self, q):  # (f, nlm) -> (m, f, n)
        d = torch.zeros(q.shape[0], (self.T + 1) ** 2, device="cuda", dtype=torch.complex128)
        d[:, self.at] = q
        return d.reshape(-1, self.T + 1, self.T + 1).permute(1, 0, 2).contiguous()

    @staticmethod
    def mul(a, b):  # complex (m, f, k) by real (m, k, j)
        return torch.complex(torch.bmm(a.real.contiguous(), b), torch.bmm(a.imag.contiguous(), b))

    def to_grid(self, F):  # (m, f, lat) -> (f, lat, lon)
        a, b = 2 * F.real, -2 * F.imag
        a[0] *= 0.5
        b[0] = 0
        return (torch.einsum("mfj,mi->fji", a, self.c) + torch.einsum("mfj,mi->fji", b, self.s))

    def synth(self, q):
        return self.to_grid(self.mul(self.dense(q), self.P))

    def gradient(self, q, a):
        d = self.dense(q)
        k = 1 / (a * self.cos)
        return (self.to_grid(self.im[:, None, None] * self.mul(d, self.P) * k), self.to_grid(self.mul(d, self.H) * k))

    def winds(self, vrt, div, a):
        lap = -self.n * (self.n + 1) / a ** 2
        inv = torch.where(self.n > 0, 1 / torch.where(self.n > 0, lap, torch.ones_like(lap)), torch.zeros_like(lap))
        psx, psy = self.gradient(vrt * inv, a)
        chx, chy = self.gradient(div * inv, a)
        return chx - psy, psx + chy

    def fourier(self, g):  # (f, lat, lon) -> (m, f, lat), with the quadrature weights
        k = 2 * math.pi / self.nlon
        F = torch.complex(torch.einsum("fji,mi->mfj", g, self.c), -torch.einsum("fji,mi->mfj", g, self.s))
        return F * (k * self.w)

    def flat(self, d):  # (m, f, n) -> (f, nlm)
        return d.permute(1, 0, 2).reshape(d.shape[1], -1)[:, self.at].contiguous()

    def anal(self, g):
        return self.flat(self.mul(self.fourier(g), self.P.transpose(1, 2).contiguous()))

    def curl_div(self, u, v, a):
        k = 1 / (a * self.cos)
        U, V = self.fourier(u * k[:, None]), self.fourier(v * k[:, None])
        Pt, Ht, im = self.P.transpose(1, 2).contiguous(), self.H.transpose(1, 2).contiguous(), self.im[:, None, None]
        return (self.flat(im * self.mul(V, Pt) + self.mul(U, Ht)), self.flat(im * self.mul(U, Pt) - self.mul(V, Ht)))


@functools.lru_cache(maxsize=1)
def _sphere(T):
    return _Sphere(T)


def _tendencies(S, st, nl, ak, bk):
    """The hydrostatic primitive equations' tendencies on hybrid levels (Simmons and Burridge's differencing) of one
    member; levels bottom to top outside, top to bottom (k) inside."""
    f32 = lambda x: float(np.float32(x))  # noqa: E731  the constants are single-precision literals
    rd, cp, cvap, omega, a = f32(287.05), f32(1004.6), f32(1846.0), f32(7.2921e-5), RERTH
    kappa = rd / cp
    ak, bk = torch.from_numpy(ak).cuda(), torch.from_numpy(bk).cuda()
    u, v = (x.flip(0) for x in S.winds(st["vrt"], st["div"], a))
    vrt, div, tv = (S.synth(st[k]).flip(0) for k in ("vrt", "div", "tv"))
    tx, ty = (x.flip(0) for x in S.gradient(st["tv"], a))
    px, py = (x[0] for x in S.gradient(st["lnps"][None], a))
    ps = torch.exp(S.synth(st["lnps"][None])[0])
    q1 = S.synth(st["trac"][0]).flip(0) if st["trac"] is not None else None
    col = (slice(None), None, None)
    pk = ak[col] + bk[col] * ps
    p1, p2, dp = pk[:-1], pk[1:], pk[1:] - pk[:-1]
    b1, b2, db = bk[:-1][col], bk[1:][col], (bk[1:] - bk[:-1])[col]
    ck = (ak[1:] * bk[:-1] - ak[:-1] * bk[1:])[col]
    rln = torch.log(p2 / p1)
    rln[0] = f32(99999.99)
    alf = 1 - p1 / dp * rln
    alf[0] = f32(math.log(2.0))
    cg = u * px + v * py
    sdb, scb = torch.cumsum(div * dp, 0), torch.cumsum(cg * db, 0)
    adb, acb = sdb - div * dp, scb - cg * db  # over the layers above
    wb = rln * (adb + ps * acb) + alf * (div * dp + ps * cg * db)
    wc = ps * cg * (db + ck * rln / dp)
    wb[0] = alf[0] * (div[0] * dp[0] + ps * cg[0] * db[0] * db[0])
    wc[0] = ps * cg[0] * db[0]
    om = (wc - wb) / dp
    dlnps = -sdb[-1] / ps - scb[-1]
    et = torch.zeros_like(pk)
    et[1:-1] = (-ps * scb - sdb - ps * b2 * dlnps)[:-1]
    cofa = -(b2 * p1 / p2 - b1 + rln * (b1 - p1 * db / dp)) / dp
    cof0 = -(b1 * rln + alf * db) / dp
    cof0[0] = -(alf[0] * db[0]) / dp[0]
    dbp = b2 / p2 - b1 / p1
    dbp[0] = 0

    def below(x):  # sum over the layers below
        return x.flip(0).cumsum(0).flip(0) - x

    pres = (cof0 - cofa) * rd * tv * ps + below(-rd * dbp * tv) * ps
    gx = pres * px + below(-rd * rln * tx) - rd * alf * tx
    gy = pres * py + below(-rd * rln * ty) - rd * alf * ty

    def vadv(x):
        d = torch.zeros_like(et)
        d[1:-1] = et[1:-1] * (x[1:] - x[:-1])
        return 0.5 / dp * (d[1:] + d[:-1])

    heat = kappa * om * tv
    if q1 is not None:
        heat = heat / (1 + (cvap / cp - 1) * q1)
    dtv = -u * tx - v * ty - vadv(tv) + heat
    z = vrt + 2 * omega * S.mu[:, None]
    fx, fy = u * z + vadv(v) - gy, v * z - vadv(u) + gx
    curl, dive = S.curl_div(fx.flip(0), fy.flip(0), a)
    ke = S.anal((0.5 * (u * u + v * v)).flip(0))
    return [-dive, curl + S.n * (S.n + 1) / a ** 2 * ke, S.anal(dtv.flip(0)), S.anal(dlnps[None])[0]]


def exact(case, seed):
    kind = case["kind"]
    if kind == "advance":
        # implicit steps, physics and damping have no short statement apart from the model itself
        return None
    if kind == "mlp":
        dims, x, t, w = _mlp_data(case, seed)
        x, t = (torch.from_numpy(v).cuda().double() for v in (x, t))
        p = torch.from_numpy(w).cuda().double().requires_grad_(True)
        at, h = 0, x
        for k, (i, o) in enumerate(zip(dims[:-1], dims[1:])):
            h = h @ p[at:at + i * o].reshape(i, o) + p[at + i * o:at + i * o + o]
            at += i * o + o
            if k < len(dims) - 2:
                h = torch.nn.functional.gelu(h)
        loss = ((h - t) ** 2).mean()
        loss.backward()
        return [p.grad, float(loss.detach())]
    T, nlon, nlat, nlm = _sizes(case)
    S, gen = _sphere(T), torch.Generator(device="cuda").manual_seed(seed)
    real, cplx, _ = _types(case)
    if kind == "tend":
        st = {k: None if v is None else v.to(cplx).to(torch.complex128) for k, v in _state(case, seed).items()}
        ak, bk = _vert(case["nlev"])
        out = [_tendencies(S, {k: None if v is None else v[i] for k, v in st.items()}, case["nlev"], ak, bk)
               for i in range(case["nmem"])]
        return [torch.stack(x) for x in zip(*out)] + ([None] if case["ntrac"] else [])
    nf = case["nf"]
    if kind == "host":
        q = _random_spec(gen, T, (nf,), -1.5, False)
        return [S.synth(q).cpu().numpy(), q.cpu().numpy()]
    if kind in ("anal", "vrtdiv"):
        g = [_random_grid(gen, nf, nlat, nlon).to(real).double() for _ in range(2 if kind == "vrtdiv" else 1)]
        return [S.anal(g[0])] if kind == "anal" else list(S.curl_div(g[0], g[1], RERTH))
    amp, slope = (1e-5, -0.5) if kind == "getuv" else (1.0, -1.5)
    q = [(amp * _random_spec(gen, T, (nf,), slope, kind == "getuv")).to(cplx).to(torch.complex128)
         for _ in range(2 if kind == "getuv" else 1)]
    if kind == "getuv":
        return list(S.winds(q[0], q[1], RERTH))
    if kind == "grad":
        return list(S.gradient(q[0], RERTH))
    return [S.synth(q[0])] + ([q[0]] if kind == "roundtrip" else [])
