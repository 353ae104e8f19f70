"""Sub-lattices smaller than a block: packed blocks (several residues to a
block) at every number of residues, ragged residues, axes packed and not, and
the per-run kernel that takes over where blocks stay mostly empty.  Volumes of
more than 20480 voxels, which smaller ones leave to the per-run kernel.  The
forward pass against the per-run kernel bit for bit; gradients against PyTorch
CPU autograd with the bars of test_gpu_net.py."""
import numpy as np
import pytest

import parallelcmacionize_amd as cmi
import test_gpu_net as T

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _net(seed, dil):
    n = cmi.WarmStartNet(seed=seed)
    n.set_normalisation([0.0, 0.0], [1.0, 1.0], 1.0)
    n.set_dilation(dil)
    return n


@pytest.mark.parametrize("shape,dil", [
    ((21, 30, 64), (1, 2, 4, 8)), ((40, 27, 32), (7, 9, 3, 8)), ((48, 33, 96), (16, 12, 16, 11)),
    ((64, 64, 64), (24, 21, 32, 64)), ((9, 70, 64), (5, 4, 3, 8)), ((64, 5, 96), (1, 2, 4, 64)),
    ((130, 3, 64), (1, 2, 43, 8)), ((8, 128, 128), (4, 8, 16, 3)), ((128, 9, 128), (3, 4, 8, 5)),
    ((10, 96, 160), (2, 33, 9, 61)), ((96, 96, 96), (32, 33, 31, 48)),
    ((128, 64, 64), (17, 33, 13, 64))])
def test_forward_identical_to_per_run(shape, dil):
    n = _net(7, dil)
    feat = np.random.default_rng(3).normal(size=shape + (2,)).astype(np.float32)
    z1 = n.predict(feat)
    n.set_tiled(False)
    z0 = n.predict(feat)
    n.close()
    assert np.isfinite(z0).all() and np.abs(z0).max() > 0
    assert np.array_equal(z0, z1)


@pytest.mark.parametrize("B,shape,dil", [
    (1, (48, 33, 96), (16, 12, 16, 11)), (2, (21, 30, 64), (1, 2, 4, 8)),
    (1, (40, 40, 64), (64, 20, 40, 33)), (1, (8, 70, 64), (3, 16, 8, 24)),
    (3, (6, 50, 96), (2, 25, 13, 32))])
def test_gradients_match_torch(B, shape, dil):
    n = _net(4, dil)
    rng = np.random.default_rng(B)
    feat = rng.normal(size=(B,) + shape + (2,)).astype(np.float32)
    tgt = rng.normal(size=(B,) + shape).astype(np.float32)
    loss, g = n.loss_and_grad(feat, tgt)
    p = n.params()
    n.close()
    zt, ws = T.torch_forward(T.split_params(p), feat, dil)
    lt = ((zt - torch.tensor(tgt)) ** 2).mean()
    lt.backward()
    assert abs(loss / lt.item() - 1) < 1e-2
    gt = T.join_grads(p, [(w.grad.numpy(), b.grad.numpy()) for w, b in ws])
    off = 0
    for li, (cin, cout, nout) in enumerate(T.LAYERS):
        for name, size, real in (("W", 27 * nout * 32, 27 * nout * 32), ("b", nout, cout)):
            a, b = g[off:off + real], gt[off:off + real]
            off += size
            cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30))
            rel = float(np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-30))
            print("layer", li, name, "cos", cos, "rel", rel)
            assert cos >= 0.995 and rel <= 5e-2, (li, name, cos, rel)
    assert np.all(g[gt == 0] == 0)
