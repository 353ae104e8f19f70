"""Field transfers around the sizes where small ones go without events (two
fields of 8192 cells out, two pieces of 131072 cells in): values bit for bit,
through repeated transfers that use the same pinned slots, with the caller's
arrays overwritten as soon as a call returns."""
import numpy as np
import pytest

import parallelcmacionize_amd as cmi

pytestmark = pytest.mark.gpu
BOX = np.array([0.0, 0.0, 0.0, 3e16, 4e16, 5e16])
SIZES = [[1, 1, 1], [1, 8, 1024], [1, 8192 // 1024 + 1, 911], [2, 8, 1024], [1, 128, 1024],
         [1, 129, 1023], [2, 128, 1024], [2, 131, 1001]]


@pytest.mark.parametrize("ncell", SIZES)
@pytest.mark.parametrize("precision", [cmi.PREC_FP64, cmi.PREC_FP32])
def test_repeated_transfers(ncell, precision):
    n = int(np.prod(ncell))
    rng = np.random.default_rng(n)
    with cmi.Context(BOX, ncell, [1, 1, 1], precision) as ctx:
        nH, xn, J = np.empty(n), np.empty(n), np.empty(n)
        unit = 6.3e-22 * (BOX[3] / ncell[0])
        for k in range(3):
            nH[:] = rng.uniform(1e7, 1e9, n)
            xn[:] = rng.standard_normal(n)
            J[:] = rng.standard_normal(n)
            want_x, want_J = xn.copy(), J.copy()
            if k == 1:
                ctx.set_fields(nH=nH)
                ctx.set_fields(xn=xn)
            else:
                ctx.set_fields(nH, xn)
            ctx.set_intensity(J)
            nH[:] = xn[:] = J[:] = np.nan
            if precision == cmi.PREC_FP32:
                want_J = (want_J * (1.0 / unit)) * unit
            for _ in range(2):
                J1, x1 = ctx.get_fields()
                assert x1.tobytes() == want_x.tobytes() and J1.tobytes() == want_J.tobytes()


@pytest.mark.parametrize("edge", [16, 32, 64])
def test_repeated_transfers_of_a_set(edge):
    rng = np.random.default_rng(edge)
    b = cmi.Batch([BOX] * 3, [[edge] * 3] * 3)
    for k in range(2):
        xs = [rng.standard_normal((edge,) * 3) for _ in range(3)]
        for q, x in enumerate(xs):
            v = x.copy()
            b.set_fields(q, None, v) if k else b.set_fields(q, np.full(x.shape, 1e8), v)
            v[:] = np.nan
        for q, x in enumerate(xs):
            assert b.get_fields(q)[1].tobytes() == x.tobytes()
    b.close()
