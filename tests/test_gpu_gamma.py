"""The three directions of q -> 0: the library forms chi once and only row and
column G = 0 again per direction; the pair densities it reports per direction
give every element of all three (chiqw.F:1780-1848), at G spheres of one and
several tiles of each contraction."""
import numpy as np
import pytest

from respackdev_amd import gen
from respackdev_amd.chiqw import Chiqw, from_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    c = Chiqw(0)
    w = from_system(gen.make_system(a=7.0, nk=2, nocc=3, nvir=5, ecut_psi=13.9, seed=43))
    c.open(w, ecut_for_eps=12.5, num_freq_grid=14)
    yield c
    c.close()


# FP64: element-wise bound of the FP64 contraction; FP32 and split-BF16: the
# mixed path's 1e-5 relative norm
@pytest.mark.parametrize("ecut", [0.5, 4.0, 7.0, 12.5])
@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16x3"])
def test_three_directions(gpu, ecut, prec):
    gpu.set_window(ecut, 0)
    lg = gpu.prepare_q((0.0, 0.0, 0.0))
    m3 = gpu.pair_densities().astype(np.complex128)
    d = gpu.weights()
    chi = gpu.accumulate(prec)
    g0 = int(np.where((lg == 0).all(1))[0][0])
    vol, k = gpu.info["volume"], m3.shape[1]
    assert chi.shape[0] == 3
    keep = np.arange(len(lg)) != g0
    for ix in range(3):
        m = m3[ix]
        if ix:  # the directions differ, and only in the G = 0 column
            assert not np.array_equal(m[:, g0], m3[0][:, g0])
            np.testing.assert_array_equal(m[:, keep], m3[0][:, keep])
        for w in range(0, len(d), 4):
            ref = (m.conj().T @ (d[w][:, None] * m)) / vol
            err = chi[ix, w].T - ref
            if prec == "fp64":
                bound = (np.abs(m).T @ (np.abs(d[w])[:, None] * np.abs(m))) / vol
                assert np.all(np.abs(err) <= 16.0 * (k + 16) * 2.0 ** -53 * bound)
            else:
                assert np.linalg.norm(err) <= 1e-5 * np.linalg.norm(ref)
