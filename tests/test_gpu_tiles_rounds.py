"""Rounds of the tiles engine at the edges of their pieces: chunks around the
placement's 4096-slot pieces and beyond one launch's workgroups, packet counts
around waves and chunks, 256 and 512 threads, 16^3 and other tiles, with the
walk-out off, on, and from the start.  Per-visit sums are exact integers, so
counts and J are the same bit for bit however a round is cut."""
import numpy as np
import pytest

import parallelcmacionize_amd as cmi
from parallelcmacionize_amd import workloads as W

pytestmark = pytest.mark.gpu
KEYS = ("crossings", "hops", "absorbed", "escaped", "errors")


def _context(ncell, nsub, nsrc):
    rng = np.random.default_rng(sum(ncell) + nsrc)
    n = int(np.prod(ncell))
    ctx = cmi.Context(W.box_10pc(), ncell, nsub, cmi.PREC_FP32)
    ctx.set_fields(1e8 * np.exp(rng.normal(0, 1, n)), 10 ** rng.uniform(-6, -2.5, n))
    ctx.set_sources(rng.uniform(-4 * W.PC, 4 * W.PC, (nsrc, 3)), np.full(nsrc, 1e48))
    return ctx


def _run(ctx, npackets, **tuning):
    ctx.set_engine(cmi.ENGINE_TILES, **tuning)
    ctx.reset_intensity()
    s = ctx.transport(npackets, 11, 3)
    return [s[k] for k in KEYS], ctx.get_fields()[0]


@pytest.mark.parametrize("npackets", [1, 63, 257, 4097, 150000])
@pytest.mark.parametrize("ncell,nsub,nsrc", [([48, 32, 64], [3, 2, 4], 1),
                                             ([40, 24, 24], [1, 1, 1], 5)])
def test_cuts_do_not_change_results(npackets, ncell, nsub, nsrc):
    with _context(ncell, nsub, nsrc) as ctx:
        ref, J = _run(ctx, npackets, finish_packets=-1)
        assert ref[2] + ref[3] == npackets and ref[4] == 0
        for t in ({"chunk_min": 256}, {"chunk_min": 4095}, {"chunk_min": 4097},
                  {"chunk_min": 100000}, {"block_threads": 256},
                  {"block_threads": 256, "chunk_min": 5000}):
            got, Jg = _run(ctx, npackets, finish_packets=-1, **t)
            assert got == ref, t
            assert Jg.tobytes() == J.tobytes(), t
        for finish in (0, 1000, npackets):
            got, Jg = _run(ctx, npackets, finish_packets=finish)
            assert got == ref and Jg.tobytes() == J.tobytes(), finish


@pytest.mark.parametrize("npackets", [300, 60000])
def test_list_equals_emission(npackets):
    """The same packets as an explicit list (per-packet outputs, its own round
    0): identical fates.  A list's records carry the start rounded from FP64
    positions as the emission's do."""
    with _context([48, 32, 64], [3, 2, 4], 3) as ctx:
        ref, J = _run(ctx, npackets)
        pk, ss = ctx.emit(npackets, 11, 3)
        ctx.reset_intensity()
        _, st, cr, hp, s = ctx.transport_packets(pk, ss)
        assert int((st == 0).sum()) == s["absorbed"] and int((st == 1).sum()) == s["escaped"]
        assert int(cr.sum()) == s["crossings"] and int(hp.sum()) == s["hops"]
        assert abs(s["crossings"] - ref[0]) <= 2 * npackets * 1e-3
        assert abs(ctx.get_fields()[0].sum() / J.sum() - 1) < 1e-5


@pytest.mark.parametrize("npackets", [1, 65, 4097, 100000])
@pytest.mark.parametrize("p", [0.364, 0.95])
def test_reemission_is_the_same_in_every_kernel(npackets, p):
    """Reemitted at the refill of a wave: the kernel of 16^3 tiles (512 threads)
    and the general one (256) draw the same packets' numbers, so counts and J
    agree bit for bit, whatever the waves' neighbours are."""
    with _context([48, 32, 64], [3, 2, 4], 2) as ctx:
        ctx.set_reemission(p)
        ref, J = _run(ctx, npackets)
        assert ref[2] + ref[3] == npackets and ref[4] == 0
        for t in ({"block_threads": 256}, {"block_threads": 256, "chunk_min": 300},
                  {"chunk_min": 100000}, {"refill_batch": 1}, {"refill_batch": 64}):
            got, Jg = _run(ctx, npackets, **t)
            assert got == ref, t
            assert Jg.tobytes() == J.tobytes(), t


@pytest.mark.parametrize("ncell", [[64, 64, 128], [64, 64, 132], [4, 4, 4], [4, 8, 12],
                                   [128, 32, 36]])
def test_plans_of_many_tiles(ncell):
    """4^3 tiles: 8192 and 8448 of them (plan and placement in one launch and in
    two), 1, 6 and 2304 (a thread's tiles not all in range), against the same
    packets walked out by one launch."""
    rng = np.random.default_rng(sum(ncell))
    n = int(np.prod(ncell))
    with cmi.Context(W.box_10pc(), ncell, [1, 1, 1], cmi.PREC_FP32) as ctx:
        ctx.set_fields(1e8 * np.exp(rng.normal(0, 1, n)), 10 ** rng.uniform(-6, -2.5, n))
        ctx.set_sources(rng.uniform(-4 * W.PC, 4 * W.PC, (3, 3)), np.full(3, 1e48))
        ref, J = _run(ctx, 30000, tile=[4, 4, 4], finish_packets=30000)
        assert ref[2] + ref[3] == 30000 and ref[4] == 0
        for t in ({}, {"finish_packets": -1}, {"finish_packets": -1, "chunk_min": 300}):
            got, Jg = _run(ctx, 30000, tile=[4, 4, 4], **t)
            assert got == ref, t
            assert Jg.tobytes() == J.tobytes(), t
