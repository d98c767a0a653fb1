"""Large arrays in and out (chi set, eps^-1 read) in chunks over several threads:
sizes below and above the 4 MiB where the chunked copies start, not multiples of
a chunk, every element checked through eps^-1 = (1 - v chi)^-1 in NumPy.

Tolerance: 1 - v chi is the identity plus a term of norm below 1/2, so its
condition is below 3 and both inversions agree to a few hundred 2^-53."""
import numpy as np
import pytest

from respackdev_amd import gen
from respackdev_amd.chiqw import Chiqw, from_system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    c = Chiqw(0)
    w = from_system(gen.make_system(a=7.0, nk=2, nocc=2, nvir=3, ecut_psi=16.0, seed=44))
    c.open(w, ecut_for_eps=15.0, num_freq_grid=14)
    yield c
    c.close()


# NG 20 (0.1 MiB), 118 (3.0), 150 (4.8: the smallest chunked copy), 336 (24.1)
@pytest.mark.parametrize("ecut", [2.0, 7.9, 8.3, 15.0])
def test_chi_in_and_epsinv_out(gpu, ecut):
    gpu.set_window(ecut, 0)
    q = np.array([0.0, 0.0, 0.5])
    lg = gpu.prepare_q(q)
    n, nen = len(lg), gpu.info["nen"]
    qg = np.linalg.norm((q + lg) * (2.0 * np.pi / 7.0), axis=1)
    v = 8.0 * np.pi / np.outer(qg, qg)
    rng = np.random.default_rng(n)
    a = rng.standard_normal((1, nen, n, n)) + 1j * rng.standard_normal((1, nen, n, n))
    chi = a * (0.1 / np.sqrt(n)) / v
    eps = gpu.dyson_from(chi)
    for w in range(nen):
        ref = np.linalg.inv(np.eye(n) - chi[0, w] * v)
        assert np.abs(eps[0, w] - ref).max() <= 1e-13
