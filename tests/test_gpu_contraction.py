"""The FP64 contraction against its definition in NumPy complex128,
chi(G,G') = sum_K conj(M(G)) d M(G') / volume (chiqw.F:1397-1410), on the pair
densities and weights of the same handle, at G spheres around the 16-blocks and
64-tiles of the kernel, for K with and without padding rows.

Tolerance, element by element: the three real products of a term are at most
2 |a||b| each and enter an element at most three times, every sum has at most K
terms, and forming d a and the final combination adds a few roundings, so both
sides together stay within 16 (K + 16) 2^-53 sum_K |a||d||a'| / volume.
"""
import numpy as np
import pytest

from respackdev_amd import gen
from respackdev_amd.chiqw import Chiqw, from_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    c = Chiqw(0)
    w = from_system(gen.make_system(a=7.0, nk=2, nocc=3, nvir=5, ecut_psi=9.0, seed=42))
    c.open(w, ecut_for_eps=8.0, num_freq_grid=14)
    yield c
    c.close()


# cutoffs (Ry) that give NG 2 .. 128 at q = (0, 0, 1/2): one block, two, the
# odd splits of three to eight blocks, one and two tiles
@pytest.mark.parametrize("ecut", [0.3, 1.0, 1.9, 2.7, 3.5, 4.3, 5.1, 5.9, 6.7, 7.5, 8.0])
@pytest.mark.parametrize("nvir", [1, 5])
def test_fp64_contraction(gpu, ecut, nvir):
    gpu.set_window(ecut, nvir)
    lg = gpu.prepare_q((0.0, 0.0, 0.5))
    m = gpu.pair_densities()[0].astype(np.complex128)
    d = gpu.weights()
    chi = gpu.accumulate("fp64")[0]
    vol, k, ng = gpu.info["volume"], m.shape[0], len(lg)
    assert chi.shape == (len(d), ng, ng)
    for w in range(len(d)):
        ref = (m.conj().T @ (d[w][:, None] * m)) / vol
        bound = (np.abs(m).T @ (np.abs(d[w])[:, None] * np.abs(m))) / vol
        err = np.abs(chi[w].T - ref)
        assert np.all(err <= 16.0 * (k + 16) * 2.0 ** -53 * bound), (ng, w)
