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
