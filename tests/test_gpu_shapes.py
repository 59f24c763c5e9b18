"""Kernels at the sizes where their tiling can go wrong: partial tiles,
remainders, the smallest and the largest of their range."""
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
