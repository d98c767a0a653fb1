"""Tetrahedron weights over the ways their frequencies are shared by workgroups:
one frequency, slices of one, remainders, one slice for many pairs, and metals
whose pieces fill the list of a workgroup several times (rough Fermi surface on
384 tetrahedra) or hardly at all.  The weights of the first pair (for a metal
the one into the first partially occupied band) against the oracle within 1e-9
of their scale, as in test_gpu_metal.py; the weights of the other pairs finite,
and none left out at some frequencies only: a pair without transitions (of a
metal, from a band into one below it) is zero at all of them, every other at
none, and an insulator has no such pair.
"""
import numpy as np
import pytest

from respackdev_amd import gen
from respackdev_amd.chiqw import Chiqw, from_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nk, nocc, nvir, ncross, nen", [
    (2, 1, 1, 0, 1),      # one workgroup
    (2, 1, 2, 1, 3),      # more slices wanted than frequencies
    (3, 2, 5, 0, 17),     # one frequency per slice
    (3, 9, 20, 0, 29),    # 180 pairs: 8 slices of 4, the last of 1
    (2, 35, 40, 0, 6),    # 1400 pairs: one slice
    (3, 2, 6, 1, 31),
    (4, 3, 4, 2, 13),
    (5, 2, 3, 1, 6),
])
def test_weights_over_slices(nk, nocc, nvir, ncross, nen):
    from oracle import pipeline
    w = from_system(gen.make_system(a=7.0, nk=nk, nocc=nocc, nvir=nvir, ecut_psi=6.0,
                                    seed=77 + nk, n_cross=ncross, rough=ncross > 0))
    q = (0.0, 0.0, 1.0 / nk)
    g = Chiqw(0)
    try:
        info = g.open(w, ecut_for_eps=1.0, num_freq_grid=nen)
        g.prepare_q(q)
        d = g.weights()
        o = pipeline.run_q(w, q, ecut_for_eps=1.0, num_freq_grid=nen)
        ntk = info["ntk"]
        if ncross:
            assert o["pvir"][0] == info["n_docc"]
        want = o["x0"].T / ntk
        np.testing.assert_allclose(d[:, :ntk], want, rtol=0, atol=1e-9 * np.abs(want).max())
        d = d.reshape(nen, -1, ntk)
        assert np.isfinite(d.view(np.float64)).all()
        some = np.abs(d).max(axis=2) > 0
        assert (some.all(axis=0) | ~some.any(axis=0)).all()
        assert ncross or some.all()
    finally:
        g.close()
