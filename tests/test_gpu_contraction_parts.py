"""Real and imaginary part of the FP64 contraction, each by its own norm, against
extended precision on the pair densities and weights of the same handle.  The
imaginary part is 5 to 10 times smaller than the real part here, so a form of the
complex product that ties its rounding to the real sums fails.

Tolerance.  With b = d a(G'), Im chi = Q1 - Q2 for Q1 = sum ar bi, Q2 = sum ai br,
whose terms have either sign.  The launch splits K so that 2048 workgroups run;
a split's n steps of four K round partial sums that grow as a random walk, which
leaves 2^-53 |Q| sqrt(n / 2) of each sum after the splits are added; the bound is
twice that, plus 2 2^-53 for forming b.  Re chi adds the splits' sums of one sign
in turn: 2^-53 |Re| sqrt(S / 3) for S splits, twice that, plus 2 2^-53 |Re|.
"""
import numpy as np
import pytest

from respackdev_amd import gen
from respackdev_amd.chiqw import Chiqw, from_system

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


def norm(x):
    return float(np.sqrt((x * x).sum()))


@pytest.mark.parametrize("nk, nocc, nvir, ecut_psi, ecut, q, nen", [
    (3, 4, 12, 13.0, 8.0, (0.0, 0.0, 1.0 / 3.0), 19), (4, 6, 16, 13.9, 6.9, (0.0, 0.0, 0.25), 16),
    (3, 4, 12, 11.0, 5.0, (0.0, 0.0, 0.0), 14)])
def test_parts_of_chi(nk, nocc, nvir, ecut_psi, ecut, q, nen):
    c = Chiqw(0)
    try:
        c.open(from_system(gen.make_system(a=7.0, nk=nk, nocc=nocc, nvir=nvir, ecut_psi=ecut_psi,
                                           seed=46)), ecut_for_eps=ecut, num_freq_grid=nen)
        lg = c.prepare_q(q)
        m = c.pair_densities()
        d = c.weights()
        chi = c.accumulate("fp64")
        vol = np.longdouble(c.info["volume"])
    finally:
        c.close()
    ng, k = len(lg), m.shape[1]
    ntile = (ng + 63) // 64
    splits = min((k + 31) // 32, -(-2048 // (ntile * ntile * nen)))
    n = 8 * -(-((k + 31) // 32) // splits)
    g0 = int(np.where((lg == 0).all(1))[0][0])
    for ix in range(len(m)):
        ar, ai = m[ix].real.astype(np.longdouble), m[ix].imag.astype(np.longdouble)
        for w in (0, nen // 2, nen - 1):
            dr, di = d[w].real.astype(np.longdouble)[:, None], d[w].imag.astype(np.longdouble)[:, None]
            br, bi = dr * ar - di * ai, dr * ai + di * ar
            q1, q2 = ar.T @ bi / vol, ai.T @ br / vol
            re = (ar.T @ br + ai.T @ bi) / vol
            got = chi[ix, w].T
            parts = [(slice(None), slice(None))]
            if ix > 0:  # this direction's own products
                parts += [(g0, slice(None)), (slice(None), g0)]
            for p in parts:
                qn = np.hypot(norm(q1[p]), norm(q2[p]))
                assert norm((got.imag - (q1 - q2))[p]) <= U * qn * (2.0 * np.sqrt(n / 2.0) + 2.0), (ix, w)
            assert norm(got.real - re) <= U * norm(re) * (2.0 * np.sqrt(splits / 3.0) + 2.0), (ix, w)
