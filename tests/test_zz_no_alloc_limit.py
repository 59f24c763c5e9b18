"""gfsdc_spectogrd_noalloc at the limit of its scratch: the intermediates of a call decide, and nothing else."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import lib, noalloc, rand_spec

pytestmark = pytest.mark.gpu


# the most fields whose extended columns and Fourier buffer fit 128 MiB: 97 280 and 259 072 bytes are left
@pytest.mark.parametrize("prec,shape,nf", [("fp64", (72, 36, 23), 7040), ("fp32", (64, 32, 21), 17088)])
def test_noalloc_takes_what_fits(prec, shape, nf):
    """The call equals gfsdc_spectogrd bit for bit, and one with another column tile is refused."""
    import gfsdc
    ctx = gfsdc.Context(*shape, gfsdc.FP64 if prec == "fp64" else gfsdc.FP32)
    q = rand_spec(ctx.degree, ctx.order, nf, seed=1).astype(np.complex128 if prec == "fp64" else np.complex64)
    print(f"noalloc {prec}: {nf} fields", flush=True)
    got = noalloc(ctx, q, np.float64 if prec == "fp64" else np.float32)
    assert np.array_equal(got, ctx.spectogrd(q, gfsdc.DT_F64 if prec == "fp64" else gfsdc.DT_F32))
    dummy = C.c_void_p(16)  # never dereferenced: the size check comes first
    assert lib().gfsdc_spectogrd_noalloc(ctx.h, dummy, dummy, nf + 64) == -1
