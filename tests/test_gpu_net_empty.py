"""Volumes without voxels: no logits, a NaN mean loss and zero gradients, with
either forward kernel; the network works on afterwards.  Negative extents are
refused."""
import ctypes as C

import numpy as np
import pytest

import parallelcmacionize_amd as cmi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("fresh", [True, False])
@pytest.mark.parametrize("shape", [(0, 8, 32), (0, 5, 32), (8, 0, 32), (8, 8, 0), (0, 0, 0)])
def test_empty_volume(shape, fresh, tiled):
    net = cmi.WarmStartNet(seed=5)
    net.set_tiled(tiled)
    rng = np.random.default_rng(1)
    f = rng.normal(size=(1, 5, 6, 32, 2)).astype(np.float32)
    t = rng.normal(size=(1, 5, 6, 32)).astype(np.float32)
    ref = None if fresh else (net.predict(f[0]), net.loss_and_grad(f, t))
    assert net.predict(np.zeros(shape + (2,), np.float32)).size == 0
    for batch in (1, 3):
        loss, g = net.loss_and_grad(np.zeros((batch,) + shape + (2,), np.float32),
                                    np.zeros((batch,) + shape, np.float32))
        assert np.isnan(loss) and not g.any()
    if not fresh:
        assert np.array_equal(net.predict(f[0]), ref[0])
        loss, g = net.loss_and_grad(f, t)
        assert abs(loss / ref[1][0] - 1) < 1e-6
        assert np.allclose(g, ref[1][1], rtol=0, atol=1e-5 * np.abs(g).max())
    net.close()


@pytest.mark.parametrize("dim", [(-1, -1, 32), (-8, 4, 32), (4, 4, -32)])
def test_negative_extents_are_refused(dim):
    net = cmi.WarmStartNet(seed=5)
    d = (C.c_int * 3)(*dim)
    buf = (C.c_float * 64)()
    g = (C.c_float * net.nparam)()
    lib = cmi.load_library()
    assert lib.cmi_net_predict(net.h, buf, d, buf) == -1
    assert lib.cmi_net_loss_and_grad(net.h, buf, buf, 1, d, buf, g) == -1
    net.close()
