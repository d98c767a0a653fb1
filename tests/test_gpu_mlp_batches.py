"""The closure network at large batches: from 16384 samples on a wave takes eight of them
(the data gradient of every layer width with a kernel of its own), and above 131072 the
gradient's partials are reduced layer by layer and the Adam step is a launch of its own.
Gradients against the oracle at the tolerances of test_gpu_mlp.py (1e-5 for the loss, 1e-4
per tensor); a training step against Adam's formula on the gradient of the rows that the
seed draws.

Tolerance of the step: the first one moves a parameter by lr g / (|g| + 1e-8), and where
|g| is above 1e-2 of its tensor's largest entry a gradient within 1e-4 of the tensor's norm
has the right sign and size: 1e-3 lr and two roundings of the parameter."""
import numpy as np
import pytest

from oracle import mlp as omlp
from respackdev_amd.closure import Mlp

pytestmark = pytest.mark.gpu


def draws(seed, count):
    """The 64-bit Mersenne Twister (Nishimura and Matsumoto)."""
    mask, mt = (1 << 64) - 1, [seed]
    for i in range(1, 312):
        mt.append((6364136223846793005 * (mt[-1] ^ (mt[-1] >> 62)) + i) & mask)
    out = []
    while len(out) < count:
        for i in range(312):
            x = (mt[i] & 0xFFFFFFFF80000000) | (mt[(i + 1) % 312] & 0x7FFFFFFF)
            mt[i] = mt[(i + 156) % 312] ^ (x >> 1) ^ (0xB5026F5AA96619E9 if x & 1 else 0)
        for x in mt:
            x ^= (x >> 29) & 0x5555555555555555
            x ^= (x << 17) & 0x71D67FFFEDA60000
            x ^= (x << 37) & 0xFFF7EEE000000000
            out.append(x ^ (x >> 43))
    return out[:count]


def net(nin, width, depth, nout, seed):
    m = Mlp(0, nin=nin, width=width, depth=depth, nout=nout, seed=3)
    rng = np.random.default_rng(seed)
    p = (rng.standard_normal(m.nparams) * 0.15).astype(np.float32)
    m.params = p
    return m, p, rng


def tensors(dims):
    lay, _ = omlp.layout(dims)
    for l, (wo, bo) in enumerate(lay):
        yield slice(wo, bo)
        yield slice(bo, bo + dims[l + 1])


@pytest.mark.parametrize("dims", [(8, 16, 2, 2), (16, 64, 2, 8), (8, 128, 2, 2), (32, 32, 1, 16),
                                  (7, 20, 2, 5)])
@pytest.mark.parametrize("n", [16384, 16389, 131400])
def test_gradient_of_large_batches(dims, n):
    m, p, rng = net(*dims, seed=n)
    try:
        x = rng.standard_normal((n, dims[0])).astype(np.float32)
        t = rng.standard_normal((n, dims[3])).astype(np.float32)
        loss, g = m.gradient(x, t)
        lo, go = omlp.gradient(p, m.dims, x, t)
        assert abs(loss - lo) <= 1e-5 * lo
        for s in tensors(m.dims):
            assert np.linalg.norm(g[s] - go[s]) <= 1e-4 * np.linalg.norm(go[s])
    finally:
        m.close()


@pytest.mark.parametrize("batch", [16389, 131400])
def test_steps_of_large_batches(batch):
    m, p, rng = net(8, 16, 2, 2, seed=batch)
    try:
        n, lr = 5003, 1e-3
        x = rng.standard_normal((n, 8)).astype(np.float32)
        t = rng.standard_normal((n, 2)).astype(np.float32)
        rows = np.array([d % n for d in draws(11, 2 * batch)])
        losses = m.train(x, t, 2, batch, lr=lr, seed=11)
        m.params = p
        one = m.train(x, t, 1, batch, lr=lr, seed=11)
        assert one[0] == losses[0]
        lo, go = omlp.gradient(p, m.dims, x[rows[:batch]], t[rows[:batch]])
        assert abs(losses[0] - lo) <= 1e-5 * lo
        p1 = m.params
        want = p - lr * go / (np.abs(go) + 1e-8)
        for s in tensors(m.dims):
            sure = np.abs(go[s]) > 1e-2 * np.abs(go[s]).max()
            assert np.all((np.abs(p1[s] - want[s]) <= 1e-3 * lr + 2.0 ** -23 * np.abs(p[s]))[sure])
        lo, _ = omlp.gradient(p1, m.dims, x[rows[batch:]], t[rows[batch:]])
        assert abs(losses[1] - lo) <= 1e-5 * lo
    finally:
        m.close()
