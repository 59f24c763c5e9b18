"""The column kernels where their addressing and their choice by size can go wrong, against the FP64 oracle."""
import numpy as np
import pytest

import cases
import levels
import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def test_fields_past_4gib():
    """Tendencies where one field's levels take 4.7 GB (768 x 12000 columns, 64 levels, FP64), so that a level's
    offset does not fit 32 bits. At T5 the products of the state are resolved by 96 x 48 columns already: the oracle's
    tendencies there are those of any finer grid to 4e-15, the tracer's, whose limiter is not smooth, to 1.2e-4."""
    import gfsdc
    nl, T = 64, 5
    ak, bk = levels.hybrid_levels(nl)
    o = O.Model(96, 48, T, nl, ak, bk, 600.0, ntrac=1)
    vrt, div, tv, lnps = cases.perturbed_state(o.sht.degree, o.sht.order, nl, seed=3, amp=0.3)
    q = 1e-4 * cases.perturbed_state(o.sht.degree, o.sht.order, nl, seed=12, amp=1.0)[2]
    q[..., 0] = 0.01 * np.linspace(1.0, 0.2, nl) * np.sqrt(4 * np.pi)
    o.set_state(vrt[0], div[0], tv[0], lnps[0], q)
    to = o.getdyntend(1)
    print("context of 768 x 12000 columns", flush=True)
    g = gfsdc.Context(768, 12000, T, gfsdc.FP64, nlev=nl, ak=ak, bk=bk, dt=600.0, ntrac=1)
    try:
        g.set_state(vrt, div, tv, lnps, trac=q[None])
        tg = g.getdyntend(1)
    finally:
        g.close()
    for k, tol in (("dvrt", 1e-9), ("ddiv", 1e-9), ("dtv", 1e-9), ("dlnps", 1e-9), ("dtrac", 1e-3)):
        assert rel(tg[k][0], to[k]) < tol, (k, rel(tg[k][0], to[k]))


# on both sides of the column counts from which a pass takes one thread per column: FP64 without tracers 50 000 in all
# at 33 to 43 levels, 80 000 at more and 100 000 at fewer; FP32, a getdyntend call, 100 000 a member
@pytest.mark.parametrize("vc", ["plain", "vc", "vc_svc"])
@pytest.mark.parametrize("prec,grid,nlev,nmem", [("fp64", (128, 194, 31), 34, 2), ("fp64", (128, 196, 31), 34, 2),
                                                 ("fp64", (256, 156, 21), 44, 2), ("fp64", (256, 160, 21), 44, 2),
                                                 ("fp64", (256, 194, 42), 5, 2), ("fp64", (256, 196, 42), 5, 2),
                                                 ("fp32", (512, 194, 42), 5, 2), ("fp32", (512, 196, 42), 5, 2)])
def test_columns_by_size(prec, grid, nlev, nmem, vc):
    """Tendencies of each member without and with vorticity confinement, and with its svc pattern, against the oracle at
    the bounds of test_gpu_stoch (FP64 1e-9, FP32 2e-4)."""
    import gfsdc
    nlon, nlat, T = grid
    stoch = {"plain": None, "vc": dict(vcamp=8.0),
             "vc_svc": dict(vcamp=8.0, svc=0.7, svc_tau=3 * 3600.0, svc_lscale=5.0e5, iseed_svc=9)}[vc]
    ak, bk = levels.hybrid_levels(nlev)
    p, tol = (gfsdc.FP64, 1e-9) if prec == "fp64" else (gfsdc.FP32, 2e-4)
    g = gfsdc.Context(nlon, nlat, T, p, nlev=nlev, ak=ak, bk=bk, dt=600.0, nmem=nmem)
    st = [cases.perturbed_state(g.degree, g.order, nlev, seed=5 + m, amp=0.3) for m in range(nmem)]
    if stoch:
        g.stoch_init(**stoch)
    g.set_state(*[np.concatenate(x) for x in zip(*st)])
    tg = g.getdyntend(1)
    for m in range(nmem):
        o = O.Model(nlon, nlat, T, nlev, ak, bk, 600.0)
        if stoch:
            o.stoch_init(**{k: v + m if k == "iseed_svc" else v for k, v in stoch.items()})
        o.set_state(*[x[0] for x in st[m]])
        to = o.getdyntend(1)
        for k in ("dvrt", "ddiv", "dtv", "dlnps"):
            assert rel(tg[k][m], to[k]) < tol, (k, m, rel(tg[k][m], to[k]))
