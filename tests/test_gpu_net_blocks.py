"""The warm-start network's block kernels at the edges of their blocks: volumes
that the 8^3 and 4x8x8 blocks do not divide, sub-lattices smaller than a block,
dilations larger than the volume, one to 17 samples.  The forward pass against
the per-run kernel bit for bit; loss and gradients against PyTorch CPU autograd
with the bars of test_gpu_net.py (activation gradients are stored in BF16)."""
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
    ((1, 1, 32), (1, 2, 4, 8)), ((7, 9, 32), (1, 2, 4, 8)), ((8, 8, 64), (1, 1, 1, 1)),
    ((17, 5, 96), (2, 3, 5, 7)), ((33, 40, 32), (1, 2, 4, 8)), ((9, 20, 32), (64, 16, 1, 33))])
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
    (1, (5, 7, 32), (1, 2, 4, 8)), (3, (9, 8, 64), (2, 3, 5, 16)),
    (17, (4, 3, 32), (1, 1, 2, 3)), (2, (12, 17, 32), (1, 2, 4, 8))])
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


def test_training_step_is_adam_of_the_gradient():
    """One training step on the only sample: the parameters move as Adam's
    first step on loss_and_grad's gradient, and a second forward uses them."""
    n = _net(9, (1, 2, 4, 8))
    rng = np.random.default_rng(5)
    f = rng.normal(size=(1, 10, 12, 32, 2)).astype(np.float32)
    t = rng.normal(size=(1, 10, 12, 32)).astype(np.float32)
    p0 = n.params()
    loss, g = n.loss_and_grad(f, t)
    n.add_samples(f, t)
    losses = n.train(1, 1, [10, 12, 32], 1e-3, seed=2)
    p1 = n.params()
    loss1, _ = n.loss_and_grad(f, t)
    n.set_params(p1)          # packed anew from the master parameters
    loss2, _ = n.loss_and_grad(f, t)
    n.close()
    assert abs(losses[0] - loss) <= 1e-5 * loss
    # m / c1 = g, v / c2 = g^2 (FP32): a step of lr g / (|g| + eps), up to the
    # order of the gradient's sums where g is far from 0
    far = np.abs(g) > 1e-4 * np.abs(g).max()
    step = -1e-3 * np.sign(g)
    assert np.allclose((p1 - p0)[far], step[far], rtol=0, atol=1e-5)
    assert np.all(p1[g == 0] == p0[g == 0])
    assert abs(loss1 - loss2) <= 1e-6 * loss1
