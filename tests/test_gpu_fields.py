"""Cell fields in and out at the edges of their transfer pieces (131072 cells)
and for orders of every kind: subgrids that are and are not whole tiles, tiles
of one cell, re-laid tiles, problem sets.  Values come back bit for bit (J of
FP32 contexts times its unit and back, each one rounding), and land in the
cells the walk reads (a one-packet walk per probe against the oracle)."""
import numpy as np
import pytest

import oracle_lib as O
import parallelcmacionize_amd as cmi
from parallelcmacionize_amd import workloads as W

pytestmark = pytest.mark.gpu
SIGMA = 6.3e-22
GRIDS = [([1, 1, 1], [1, 1, 1]), ([3, 5, 7], [1, 5, 7]), ([64, 64, 32], [4, 1, 2]),
         ([64, 64, 33], [2, 4, 1]), ([48, 40, 70], [3, 2, 7]), ([96, 112, 80], [2, 7, 5])]


def _special(n, rng):
    v = rng.standard_normal(n) * 10.0 ** rng.integers(-300, 300, n)
    v[::max(1, n // 7)] = np.inf
    v[n // 2] = np.nan
    v[n // 3] = -0.0
    return v


@pytest.mark.parametrize("ncell,nsub", GRIDS)
@pytest.mark.parametrize("precision", [cmi.PREC_FP64, cmi.PREC_FP32])
def test_fields_round_trip(ncell, nsub, precision):
    rng = np.random.default_rng(sum(ncell))
    n = int(np.prod(ncell))
    box = np.array([0.0, 0.0, 0.0, 3e16, 4e16, 5e16])
    with cmi.Context(box, ncell, nsub, precision) as ctx:
        J0, x0 = ctx.get_fields()
        assert np.all(J0 == 0) and np.all(x0 == 1e-6)
        x, J = _special(n, rng), rng.standard_normal(n)
        ctx.set_fields(xn=x)
        ctx.set_intensity(J)
        J1, x1 = ctx.get_fields()
        assert x1.tobytes() == x.tobytes()
        unit = SIGMA * (box[3] / nsub[0] / (ncell[0] // nsub[0]))
        want = J if precision == cmi.PREC_FP64 else (J * (1.0 / unit)) * unit
        assert J1.tobytes() == want.tobytes()
        # another tile shape: the same values in the caller's order
        if precision == cmi.PREC_FP32:
            ctx.set_engine(cmi.ENGINE_TILES, tile=[1, 1, 1])
            assert ctx.get_fields()[1].tobytes() == x.tobytes()


@pytest.mark.parametrize("ncell,nsub", GRIDS)
def test_fields_reach_their_cells(ncell, nsub):
    rng = np.random.default_rng(1 + sum(ncell))
    n = int(np.prod(ncell))
    box = W.box_10pc()
    dens, xn = 1e8 * np.exp(rng.normal(0, 1, n)), 10 ** rng.uniform(-5, -1, n)
    with cmi.Context(box, ncell, nsub, cmi.PREC_FP64) as ctx:
        ctx.set_fields(dens, xn)
        ctx.set_sources([[0.11 * W.PC, -0.2 * W.PC, 0.3 * W.PC]], [1e49])
        pk, ss = ctx.emit(300, 1, 0)
        po, st, cr, _, _ = ctx.transport_packets(pk, ss)
        J, _ = ctx.get_fields()
    og = O.OracleGrid(O.load_oracle(), box, ncell, nsub)
    og.n[:] = dens
    og.xn[:] = xn
    og.J[:] = 0
    st_o, cr_o, _ = og.transport(pk, ss)
    assert np.array_equal(st, st_o) and np.array_equal(cr, cr_o)
    assert np.array_equal(po["tau"], pk["tau"])  # the oracle's, walked in place
    assert np.all(np.abs(J - og.J) <= 600 * 2.3e-16 * np.maximum(J, og.J))


def test_problem_set_fields_round_trip():
    rng = np.random.default_rng(8)
    ncells = [[16, 16, 16], [48, 32, 96], [64, 64, 32], [32, 80, 64]]
    b = cmi.Batch([[0, 0, 0, 1e17, 2e17, 3e17]] * len(ncells), ncells)
    xs = [_special(int(np.prod(c)), rng).reshape(c) for c in ncells]
    for q, x in enumerate(xs):
        J0, x0 = b.get_fields(q)
        assert np.all(J0 == 0) and np.all(x0 == 1e-6)
        b.set_fields(q, xn=x)
    for q, x in enumerate(xs):
        assert b.get_fields(q)[1].tobytes() == x.tobytes()
    b.close()
