"""The placement's shares of a round's visits: the arithmetic on the host, and
rounds of more visits times pieces than 32 bits hold on the GPU."""
import os
import subprocess

import numpy as np
import pytest

import parallelcmacionize_amd as cmi
from parallelcmacionize_amd import workloads as W

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("program", ["place_shares", "place_blocks"])
def test_shares_and_workgroups(tmp_path, program):
    exe = str(tmp_path / program)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-o", exe,
                    os.path.join(HERE, "cpp", program + ".cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_unsplit_chunks_on_many_tiles():
    """2^18 tiles of 4 cells, a packet in each, and chunks of up to 2^26
    packets (no visit is ever split): counts, fates and J as with the default
    chunk and as walked out by one launch, bit for bit."""
    ncell, tile = [128, 128, 64], [1, 2, 2]
    rng = np.random.default_rng(8)
    n = int(np.prod(ncell))
    assert n == 4 << 18
    with cmi.Context(W.box_10pc(), ncell, [1, 1, 1], cmi.PREC_FP32) as ctx:
        # a mean free path of a few cells
        dx = 10 * W.PC / 128
        ctx.set_fields(np.full(n, 1e8), rng.uniform(0.1, 1.0, n) / (6.3e-22 * 1e8 * dx))
        p = np.zeros(1 << 18, cmi.PHOTON_DTYPE)
        t = np.stack(np.unravel_index(np.arange(1 << 18), (128, 64, 32)), axis=1)
        cell = np.array([10 * W.PC / c for c in ncell])
        p["pos"] = -5 * W.PC + (t + rng.uniform(0.05, 0.95, t.shape)) * cell * tile
        d = rng.normal(size=t.shape)
        p["dir"] = d / np.linalg.norm(d, axis=1)[:, None]
        p["tau"] = rng.uniform(0.1, 4.0, len(p))
        p["sigma"] = 6.3e-22
        p["weight"] = 1.0
        ss = np.zeros(len(p), np.uint32)

        def run(**tuning):
            ctx.set_engine(cmi.ENGINE_TILES, tile=tile, **tuning)
            ctx.reset_intensity()
            _, st, cr, hp, s = ctx.transport_packets(p, ss)
            return st, cr, hp, s, ctx.get_fields()[0]

        st, cr, hp, s, J = run(finish_packets=len(p))
        assert s["errors"] == 0 and s["absorbed"] + s["escaped"] == len(p)
        assert s["hops"] > 3 * len(p)
        for chunk in (0, 1 << 20, 1 << 26):
            got = run(finish_packets=-1, chunk_min=chunk)
            assert all(got[3][k] == s[k] for k in
                       ("crossings", "hops", "absorbed", "escaped", "errors")), chunk
            for a, b in ((got[0], st), (got[1], cr), (got[2], hp), (got[4], J)):
                assert a.tobytes() == b.tobytes(), chunk
