"""The walk engine's emission kernel against the oracle on the packets it
emits: packet counts around its wave and serve-batch sizes, one source (every
first deposit in one cell) and the most sources a context takes (more hot
cells than the deposit table has entries for), with and without reemission."""
import numpy as np
import pytest

import oracle_lib as O
import parallelcmacionize_amd as cmi
from parallelcmacionize_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npackets,nsrc,nsub", [
    (1, 1, [1, 1, 1]), (31, 1, [2, 1, 3]), (33, 2, [3, 2, 1]), (4097, 1, [4, 4, 4]),
    (40000, 64, [3, 2, 4]), (200000, 7, [2, 2, 2])])
def test_emitted_transport_matches_oracle(npackets, nsrc, nsub):
    rng = np.random.default_rng(npackets)
    ncell = [12, 8, 24]
    box = np.array([-5 * W.PC, -4 * W.PC, -6 * W.PC, 10 * W.PC, 8 * W.PC, 12 * W.PC])
    nc = int(np.prod(ncell))
    n = 1e8 * np.exp(rng.normal(0, 1, nc))
    xn = 10 ** rng.uniform(-5, -1, nc)
    pos = box[:3] + rng.uniform(0.05, 0.95, (nsrc, 3)) * box[3:]
    with cmi.Context(box, ncell, nsub, cmi.PREC_FP64) as ctx:
        ctx.set_fields(n, xn)
        ctx.set_sources(pos, np.full(nsrc, 1e48))
        pk, ss = ctx.emit(npackets, 3, 1)
        s = ctx.transport(npackets, 3, 1)
        J, _ = ctx.get_fields()
    og = O.OracleGrid(O.load_oracle(), box, ncell, nsub)
    og.n[:] = n
    og.xn[:] = xn
    og.J[:] = 0
    st, cr, hp = og.transport(pk, ss)
    assert s["crossings"] == int(cr.sum()) and s["hops"] == int(hp.sum())
    assert s["absorbed"] == int((st == 0).sum()) and s["escaped"] == int((st == 1).sum())
    assert s["errors"] == 0
    # a cell sums at most npackets x 2 positive FP64 deposits in another order
    assert np.all(np.abs(J - og.J) <= 2 * npackets * 2.3e-16 * np.maximum(J, og.J))


@pytest.mark.parametrize("npackets", [1, 64, 20000])
def test_emitted_reemission_equals_list(npackets):
    """The same packets as an explicit list (its own kernel), reemission on:
    identical counts, J to the order of the sums."""
    ncell, nsub = [16, 16, 16], [2, 1, 4]
    box = W.box_10pc()
    with cmi.Context(box, ncell, nsub, cmi.PREC_FP64) as ctx:
        ctx.set_fields(np.full(4096, 1e8), np.full(4096, 1e-3))
        ctx.set_sources([[0.1 * W.PC, 0.0, -0.2 * W.PC]], [1e49])
        ctx.set_reemission(0.6, seed=5, iteration=2)
        pk, ss = ctx.emit(npackets, 5, 2)
        a = ctx.transport(npackets, 5, 2)
        Ja, _ = ctx.get_fields()
        ctx.reset_intensity()
        _, _, _, _, b = ctx.transport_packets(pk, ss)
        Jb, _ = ctx.get_fields()
    for k in ("crossings", "hops", "absorbed", "escaped", "reemitted"):
        assert a[k] == b[k], k
    # at most 64 deposits of a packet in one cell (0.6^64 of the packets more)
    assert np.all(np.abs(Ja - Jb) <= 64 * npackets * 2.3e-16 * np.maximum(Ja, Jb))
