"""The explicit scheme (explicit_ = 1) against the FP64 oracle: no linear terms, every field by its tendencies alone."""
import numpy as np
import pytest

import cases
import levels
import oracle as O

pytestmark = pytest.mark.gpu


# fields of a coefficient below, on and past the lanes of a wavefront; a count of coefficients off its four wavefronts
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nlev,ntrac,nmem", [(2, 0, 3), (21, 2, 1), (64, 1, 2)])
def test_explicit_steps(nlev, ntrac, nmem, prec):
    """Three short steps of each member (2-norm, the bounds of test_gpu_moist: FP64 1e-9, FP32 1e-4), eager and from a
    graph, with the clock moved by three steps."""
    import gfsdc
    ak, bk = levels.hybrid_levels(nlev)
    o = O.Model(64, 32, 21, nlev, ak, bk, 60.0, ntrac=ntrac, explicit_=1)
    p, tol = (gfsdc.FP64, 1e-9) if prec == "fp64" else (gfsdc.FP32, 1e-4)
    x = [np.concatenate(v) for v in zip(*(cases.perturbed_state(o.sht.degree, o.sht.order, nlev, seed=3 + m, amp=0.2)
                                          for m in range(nmem)))]
    q = np.zeros((nmem, ntrac, nlev, o.sht.nlm), complex)
    for t in range(ntrac):
        q[:, t] = 1e-4 * x[2]
        q[:, t, :, 0] = 0.01 * np.linspace(1.0, 0.2, nlev) * np.sqrt(4 * np.pi)
    for graph in (False, True):
        g = gfsdc.Context(64, 32, 21, p, nlev=nlev, ak=ak, bk=bk, dt=60.0, ntrac=ntrac, nmem=nmem, explicit_=1)
        g.set_state(*x, trac=q if ntrac else None)
        g.advance(3, use_graph=graph)
        assert g.time == 180.0
        sg = g.get_state()
        for m in range(nmem):
            o.pdryini = 0.0
            o.set_state(*(v[m] for v in x), *([q[m]] if ntrac else []))
            o.advance(3)
            so = o.get_state()
            for k in ("vrt", "div", "tv", "lnps") + (("trac",) if ntrac else ()):
                e = np.linalg.norm(sg[k][m] - so[k]) / np.linalg.norm(so[k])
                assert e < tol, (graph, k, m, e)
