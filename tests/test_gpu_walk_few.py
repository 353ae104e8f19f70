"""The walk engine's emission kernel where packets are few: lanes and waves left
out, at the counts where one more lane of a wave takes packets (multiples of
the waves that fill the chip, and of a custom grid's), in both precisions.  The
same packets as an explicit list go through the same arithmetic: counts are
identical, J to the order of its FP64 sums."""
import numpy as np
import pytest

import parallelcmacionize_amd as cmi
from parallelcmacionize_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [cmi.PREC_FP64, cmi.PREC_FP32])
@pytest.mark.parametrize("blocks", [0, 1, 3, 16])
@pytest.mark.parametrize("reemission", [0.0, 0.7])
def test_few_packets_equal_list(precision, blocks, reemission):
    ncell, nsub = [16, 24, 32], [2, 3, 4]
    n = int(np.prod(ncell))
    rng = np.random.default_rng(11)
    with cmi.Context(W.box_10pc(), ncell, nsub, precision) as ctx:
        ctx.set_engine(cmi.ENGINE_WALK, walk_blocks=blocks)
        ctx.set_fields(1e8 * np.exp(rng.normal(0, 1, n)), 10 ** rng.uniform(-4.5, -2, n))
        ctx.set_sources(rng.uniform(-4 * W.PC, 4 * W.PC, (3, 3)), np.full(3, 1e48))
        ctx.set_reemission(reemission, seed=9, iteration=4)
        for npackets in (1, 2, 5, 8, 9, 63, 65, 511, 513, 1023, 1024, 1025, 2049, 65537):
            ctx.reset_intensity()
            a = ctx.transport(npackets, 9, 4)
            Ja, _ = ctx.get_fields()
            pk, ss = ctx.emit(npackets, 9, 4)
            ctx.reset_intensity()
            b = ctx.transport_packets(pk, ss)[-1]
            Jb, _ = ctx.get_fields()
            assert a["errors"] == 0 and a["absorbed"] + a["escaped"] == npackets
            for k in ("crossings", "hops", "absorbed", "escaped", "reemitted"):
                assert a[k] == b[k], (npackets, k)
            # a packet deposits at most 64 times in a cell (0.7^64 of them more)
            assert np.all(np.abs(Ja - Jb) <= 64 * npackets * 2.3e-16 * np.maximum(Ja, Jb))
