"""The closure network's kernels at the sizes their dispatch turns on: layer
widths with a kernel of their own (8, 16, 32, 64, 128 inputs), widths without
one (off a 16-byte row), outputs narrower and wider than 16, and batches around
the samples of a wave and the 256-sample chunks of the weight gradient, against
the oracle (FP64, the same BF16-rounded weights) at the tolerances of
test_gpu_mlp.py: 1e-5 for outputs and loss, 1e-4 per gradient tensor."""
import numpy as np
import pytest

from oracle import mlp as omlp
from respackdev_amd.closure import Mlp

pytestmark = pytest.mark.gpu

NETS = [(8, 128, 3, 2), (16, 64, 2, 16), (32, 32, 1, 3), (8, 16, 2, 1), (128, 128, 1, 128),
        (7, 20, 2, 5), (64, 100, 2, 17)]


@pytest.mark.parametrize("net", NETS)
@pytest.mark.parametrize("n", [1, 7, 9, 255, 257, 700])
def test_forward_and_gradient(net, n):
    nin, width, depth, nout = net
    m = Mlp(0, nin=nin, width=width, depth=depth, nout=nout, seed=3)
    try:
        rng = np.random.default_rng(n)
        p = (rng.standard_normal(m.nparams) * 0.15).astype(np.float32)
        m.params = p
        x = rng.standard_normal((n, nin)).astype(np.float32)
        t = rng.standard_normal((n, nout)).astype(np.float32)
        y = m.forward(x)
        yo = omlp.forward(p, m.dims, x)
        assert np.linalg.norm(y - yo) <= 1e-5 * np.linalg.norm(yo)
        loss, g = m.gradient(x, t)
        lo, go = omlp.gradient(p, m.dims, x, t)
        assert abs(loss - lo) <= 1e-5 * lo
        lay, _ = omlp.layout(m.dims)
        for l, (wo, bo) in enumerate(lay):
            for a, b in ((wo, bo), (bo, bo + m.dims[l + 1])):
                assert np.linalg.norm(g[a:b] - go[a:b]) <= 1e-4 * np.linalg.norm(go[a:b])
    finally:
        m.close()
