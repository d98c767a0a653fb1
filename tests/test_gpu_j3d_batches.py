"""calc_j3d over many lattice vectors in one call: the R are taken in batches
whose vectors share each eps^-1, so every R must come out as it does alone, for
column counts off the 16-blocks and 64-tiles of the contraction and a list long
enough for two batches (the last one ragged).

Tolerance: the sums of one (R, q, w) have the same terms whatever the batch;
only the split over q and rows can reorder them, a few hundred 2^-53 of the
largest element."""
import numpy as np
import pytest

from respackdev_amd import gen
from respackdev_amd.chiqw import from_system
from respackdev_amd.w3d import W3d

pytestmark = pytest.mark.gpu


def _open(nk, nwf, ecut_psi, ecut_eps, nen):
    s = gen.make_system(a=7.0, nk=nk, nocc=1, nvir=1, ecut_psi=ecut_psi, seed=60)
    wan, _ = gen.make_wannier(s, nwf, 61)
    w = from_system(s)
    W = np.zeros((len(wan), nwf, max(c.shape[1] for c in wan)), np.complex128)
    for k, c in enumerate(wan):
        W[k, :, :c.shape[1]] = c
    g = W3d(0)
    g.open(w, ecut_eps, np.linspace(0.0, 1.0, nen).astype(np.complex128))
    g.set_wannier(W)
    rng = np.random.default_rng(62)
    for iq, n in enumerate(g.set_q(w.ski)):
        e = rng.standard_normal((nen, n, n)) + 1j * rng.standard_normal((nen, n, n))
        g.set_epsinv(iq, np.eye(n) + 0.2 * e / np.sqrt(n))
    return g


def _rlist(n, m):
    r = np.arange(-m, m + 1)
    return np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)[:n]


@pytest.mark.parametrize("nk,nwf,ecut_psi,ecut_eps,nen,nr", [
    (2, 1, 3.0, 1.0, 1, 1), (2, 1, 6.0, 3.0, 3, 5), (3, 2, 6.0, 4.0, 2, 27), (2, 3, 9.0, 6.7, 1, 4),
    (3, 5, 5.0, 2.7, 1, 13), (4, 9, 14.0, 7.0, 2, 70)])
def test_every_r_as_alone(nk, nwf, ecut_psi, ecut_eps, nen, nr):
    g = _open(nk, nwf, ecut_psi, ecut_eps, nen)
    try:
        rs = _rlist(nr, 2)
        x, j, _, _ = g.j3d(rs)
        pick = sorted({0, 1, nr // 2, nr - 2, nr - 1} & set(range(nr)))
        for i in pick:
            x1, j1, _, _ = g.j3d([rs[i]])
            assert np.abs(x[i] - x1[0]).max() <= 5e-14 * np.abs(x1).max()
            assert np.abs(j[:, i] - j1[:, 0]).max() <= 5e-14 * np.abs(j1).max()
    finally:
        g.close()
