"""calc_int's pair sums on regular k meshes against extended precision: meshes with a
different number of points on every axis (one to eight), and k lists of few digits, whose
positions on the mesh are what counts.  func of every q (the sum of rho_i conj(rho_j)
over G), its imaginary part by the size of its own rounding.  And a run whose summed grids
take two passes over q, against the same pairs among fewer.

Tolerance.  A value rho(q+G) carries the roundings of some 16 steps in turn (up to nine
passes along mesh axes, three phases, the transform), 4 2^-53 as a random walk; N terms
of func add theirs as another: 4 2^-53 / sqrt(N) of the sum of N terms of one sign.  The
real part, where a factor's own rounding is common to every term, is held to 8 2^-53.
The single-precision grids u_k(r) are rounded here as on the GPU.
"""
import numpy as np
import pytest
import scipy.fft

from respackdev_amd import gen
from respackdev_amd.chiqw import WfnData
from respackdev_amd.w3d import W3d

pytestmark = pytest.mark.gpu

A0 = 7.0
B0 = 2.0 * np.pi / A0
LD, CL = np.longdouble, np.clongdouble
PI = LD("3.14159265358979323846264338327950288")


def sphere(q, ecut):
    m = int(np.sqrt(ecut) / B0) + 3
    r = np.arange(-m, m + 1)
    g = np.stack(np.meshgrid(r, r, r, indexing="ij"), -1).reshape(-1, 3)
    e = (((np.asarray(q) + g) * B0) ** 2).sum(1)
    return g[e <= ecut].astype(np.int32), e[e <= ecut]


def mesh(n, digits):
    """One of every +-k pair of the n1 x n2 x n3 mesh, rounded to `digits` digits."""
    out, seen = [], set()
    for i in np.ndindex(*n):
        if i in seen:
            continue
        seen.add(tuple(-x % m for x, m in zip(i, n)))
        k = [(x / m if 2 * x <= m else x / m - 1.0) for x, m in zip(i, n)]
        out.append([round(v, digits) for v in k])
    return np.array(out)


def system(n, nwf, ecut, digits=16, seed=81):
    ski = mesh(n, digits)
    kg = [sphere(k, ecut)[0] for k in ski]
    ngi = np.array([len(g) for g in kg], np.int32)
    kgi = np.zeros((len(ski), int(ngi.max()), 3), np.int32)
    for i, g in enumerate(kg):
        kgi[i, :len(g)] = g
    w = WfnData(lattice=np.eye(3) * A0, rg=np.eye(3, dtype=np.int32).reshape(1, 9).copy(),
                pg=np.zeros((1, 3), np.int32), nnp=1, ski=ski, ngi=ngi, kgi=kgi,
                eig=np.zeros((len(ski), 1)), wfn=np.zeros((len(ski), 1, kgi.shape[1]), np.complex128),
                ef=0.0, ecut=ecut)
    sk0, trs = gen.full_kmesh(ski)
    full = [sphere(k * t, ecut)[0] * t for k, t in zip(sk0, trs)]
    wan, _ = gen.wannier_on(sk0, full, np.eye(3) * B0, nwf, seed)
    W = np.zeros((len(sk0), nwf, max(c.shape[1] for c in wan)), np.complex128)
    for k, c in enumerate(wan):
        W[k, :, :c.shape[1]] = c
    return w, sk0, full, wan, W


def exact_func(n, w, sk0, full, wan, nw, ecut_eps):
    nwf = len(wan[0])
    u = np.zeros((len(sk0), nwf, *nw[::-1]), CL)  # [z][y][x]
    for k, g in enumerate(full):
        g = g % np.array(nw)
        u[k][:, g[:, 2], g[:, 1], g[:, 0]] = wan[k]
    u = scipy.fft.ifftn(u, axes=(2, 3, 4)) * (nw[0] * nw[1] * nw[2])
    u = u.astype(np.complex64).astype(CL)
    key = {tuple(np.rint(k * n).astype(int) % n): i for i, k in enumerate(sk0)}
    qs = [(q, q, 1) for q in w.ski]
    have = {tuple(np.rint(q * n).astype(int) % n) for q in w.ski}
    qs += [(-q, q, -1) for q in w.ski if tuple(np.rint(-q * n).astype(int) % n) not in have]
    r = [np.arange(m).astype(LD) / m for m in nw]
    out = []
    for q, q0, t in qs:
        ge, _ = sphere(q0, ecut_eps)
        gp, e = sphere(q0, w.ecut)
        lst = np.concatenate([ge, gp[e > ecut_eps]]) * t
        qg = np.sqrt((((q + lst) * B0) ** 2).sum(1)).astype(LD)
        iq = np.where(qg == 0, 0, 1 / np.where(qg == 0, 1, qg))
        acc = np.zeros((nwf, *nw[::-1]), CL)
        for k in range(len(sk0)):
            j = key[tuple(np.rint((sk0[k] + q) * n).astype(int) % n)]
            s = np.rint(sk0[k] + q - sk0[j]).astype(LD)
            th = 2 * PI * (s[2] * r[2][:, None, None] + s[1] * r[1][:, None] + s[0] * r[0])
            acc += u[j].conj() * (np.cos(th) + 1j * np.sin(th)) * u[k]
        g = lst % np.array(nw)
        m = scipy.fft.ifftn(acc, axes=(1, 2, 3))[:, g[:, 2], g[:, 1], g[:, 0]]
        rho = m * iq / len(sk0)
        out.append((rho @ rho.conj().T).T)
    return np.array(out)


def norm(x):
    return float(np.sqrt((abs(x) ** 2).sum()))


@pytest.mark.parametrize("n, nwf, ecut, digits", [
    ((3, 3, 3), 4, 8.0, 16), ((3, 3, 3), 4, 8.0, 13), ((3, 3, 3), 3, 8.0, 10), ((6, 1, 3), 3, 7.0, 9),
    ((2, 3, 4), 4, 8.0, 16), ((4, 3, 2), 2, 9.0, 16), ((5, 1, 2), 5, 10.0, 16), ((1, 6, 7), 2, 6.0, 16),
    ((8, 2, 1), 3, 9.0, 16), ((3, 5, 1), 9, 13.0, 16)])
def test_func_on_a_mesh(n, nwf, ecut, digits):
    w, sk0, full, wan, W = system(n, nwf, ecut, digits)
    ecut_eps = 0.55 * ecut
    g = W3d(0)
    try:
        g.open(w, ecut_eps, np.zeros(1, np.complex128))
        g.set_wannier(W)
        for iq, m in enumerate(g.set_q(w.ski)):
            g.set_epsinv(iq, np.eye(m, dtype=np.complex128)[None])
        func, _ = g.funcs()
        inf = g.info()
    finally:
        g.close()
    assert (inf["nkb1"], inf["nkb2"], inf["nkb3"]) == n
    ref = exact_func(np.array(n), w, sk0, full, wan, (inf["nwx"], inf["nwy"], inf["nwz"]), ecut_eps)
    u = 2.0 ** -53
    ng = min(w.ngi)
    assert norm(func.imag - ref.imag) <= 4.0 * u / np.sqrt(ng) * norm(ref.real)
    assert norm(func.real - ref.real) <= 8.0 * u * norm(ref.real)


def test_q_in_two_passes():
    """Nine functions on 6^3 k and a 16^3 grid: 1.1 GiB of summed grids, more than the
    1 GiB held at once.  Two R; tolerance as in test_gpu_j3d_batches.py."""
    n, rs = (6, 6, 6), [(0, 0, 0), (1, 0, -1)]
    out = []
    for nwf in (9, 3):
        w, _, _, _, W = system(n, 9, 45.5)
        g = W3d(0)
        try:
            g.open(w, 2.0, np.zeros(1, np.complex128))
            assert g.info()["nwx"] == 16
            g.set_wannier(W[:, :nwf])
            for iq, m in enumerate(g.set_q(w.ski)):
                g.set_epsinv(iq, 0.7 * np.eye(m, dtype=np.complex128)[None])
            x, j, _, _ = g.j3d(rs)
            out.append((x, j))
        finally:
            g.close()
    (x9, j9), (x3, j3) = out
    assert np.abs(x9[:, :3, :3] - x3).max() <= 5e-14 * np.abs(x3).max()
    assert np.abs(j9[:, :, :3, :3] - j3).max() <= 5e-14 * np.abs(j3).max()


def test_most_k_and_most_functions():
    """256 k (8 x 8 x 4) and sixteen functions, the largest that the LDS of the mesh
    transforms holds, against the first two functions alone (eight grid points at a time
    instead of one): rho of a pair takes the same operations whatever its company, the
    sums over G and the contraction at most a few hundred 2^-53 of the largest element."""
    n, out = (8, 8, 4), []
    w, _, _, _, W1 = system(n, 1, 4.0)
    rng = np.random.default_rng(82)
    W = (rng.standard_normal((W1.shape[0], 16, W1.shape[2])) +
         1j * rng.standard_normal((W1.shape[0], 16, W1.shape[2])))
    W *= (np.abs(W1) > 0)  # the plane waves of each k
    for nwf in (16, 2):
        g = W3d(0)
        try:
            g.open(w, 2.0, np.zeros(1, np.complex128))
            g.set_wannier(W[:, :nwf])
            for iq, m in enumerate(g.set_q(w.ski)):
                g.set_epsinv(iq, 0.7 * np.eye(m, dtype=np.complex128)[None])
            out.append(g.funcs() + g.j3d([(1, 0, -1)])[:2])
        finally:
            g.close()
    for a, b in zip(*out):
        assert np.abs(a[..., :2, :2] - b).max() <= 5e-14 * np.abs(b).max()
