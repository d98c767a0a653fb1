"""Calls that meet an allocation that fails: hipMalloc or hipHostMalloc refused from a
size on by alloc_limits.c, in a process of its own (the refusal comes from the host;
every kernel runs as usual).  What the caller asked for still arrives, or an error and
what was computed before it.  And what a call leaves allocated."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes as C, sys
sys.path.insert(0, sys.argv[2])
lim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lim.alloc_limits.argtypes = [C.c_size_t, C.c_size_t]
lim.alloc_live.restype = C.c_size_t
ALL = 2 ** 64 - 1
import numpy as np
from respackdev_amd import _lib, gen
from respackdev_amd.chiqw import Chiqw, from_system
def opened(ecut, nen=14, **kw):
    c = Chiqw(0)
    c.open(from_system(gen.make_system(a=7.0, seed=47, **kw)), ecut_for_eps=ecut, num_freq_grid=nen)
    return c
def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))
"""


def run(tmp_path, body):
    so = str(tmp_path / "alloc_limits.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", os.path.join(HERE, "alloc_limits.c"), "-o", so, "-ldl"],
                   check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, so, os.path.dirname(HERE)],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split()[-1:] == ["done"], r.stdout + r.stderr


def test_chi_arrives_when_the_dyson_step_fails(tmp_path):
    run(tmp_path, """
c = opened(4.0, nk=2, nocc=2, nvir=3, ecut_psi=9.0)
q = (0.0, 0.0, 0.5)
lg = c.prepare_q(q); c.pair_densities(False); c.weights(False)
ref = c.accumulate("fp64")
lim.alloc_limits(0, ALL)  # eps^-1 has no buffer yet
chi = np.zeros_like(ref); eps = np.zeros_like(ref); qq = np.array(q)
rc = _lib.lib().rp_chiqw_q(c._h, _lib.ptr(qq), 0, _lib.ptr(eps), _lib.ptr(chi), None)
assert rc != 0 and lim.alloc_refused() > 0, (rc, lim.alloc_refused())
assert rel(chi, ref) <= 1e-13, rel(chi, ref)  # the weights' sums meet in any order
lim.alloc_limits(ALL, ALL)
assert rel(c.run_q(q, "fp64", want_chi=True)["chi"], ref) <= 1e-13
c.close(); print("done")
""")


# NG ~ 300, 200 frequencies, K 38400: partial sums of 0.3 GB per split of K, four splits
# (twice that is above the 2 GiB bound), one where it must be
LARGE = """
c = opened(14.0, nen=200, nk=4, nocc=10, nvir=60, ecut_psi=14.5)
ng = len(c.prepare_q((0.0, 0.0, 0.25))); c.pair_densities(False); c.weights(False)
per = 16 * ng * ng * 200
"""


def test_tuner_stays_within_the_bound_of_the_partial_sums(tmp_path):
    run(tmp_path, LARGE + """
lim.alloc_limits(2 ** 31, ALL)
c.autotune(True); c.accumulate("fp64", copy=False)
t = c.tune_table()[0]
assert t["heuristic_nsplit"] == 4 and 8 * per > 2 ** 31 and lim.alloc_refused() == 0, t
c.close(); print("done")
""")


def test_tuner_passes_over_what_does_not_fit(tmp_path):
    run(tmp_path, """
c = opened(6.9, nk=4, nocc=4, nvir=8, ecut_psi=9.0)
ng = len(c.prepare_q((0.0, 0.0, 0.25))); c.pair_densities(False); c.weights(False)
ref = c.accumulate("fp64"); c.close()
c = opened(6.9, nk=4, nocc=4, nvir=8, ecut_psi=9.0)
c.autotune(True)
c.prepare_q((0.0, 0.0, 0.25)); c.pair_densities(False); c.weights(False)
sp = min(4 * 8 * 64 // 32, -(-2048 // ((-(-ng // 64)) ** 2 * 14)))
lim.alloc_limits(sp * 16 * ng * ng * 14, ALL)  # the heuristic's partials, not twice them
chi = c.accumulate("fp64")
t = c.tune_table()[0]
assert t["heuristic_nsplit"] == sp and t["nsplit"] <= sp and lim.alloc_refused() > 0, t
assert rel(chi, ref) <= 1e-13
c.close(); print("done")
""")


def test_fewer_splits_when_memory_is_short(tmp_path):
    run(tmp_path, LARGE + """
ref = c.accumulate("fp64"); c.close()
c = opened(14.0, nen=200, nk=4, nocc=10, nvir=60, ecut_psi=14.5)
c.prepare_q((0.0, 0.0, 0.25)); c.pair_densities(False); c.weights(False)
lim.alloc_limits(3 * per, ALL)
chi = c.accumulate("fp64")
assert lim.alloc_refused() > 0 and rel(chi, ref) <= 1e-13, rel(chi, ref)
c.close(); print("done")
""")


def test_exchange_gives_large_buffers_back(tmp_path):
    """Nine functions on 6^3 k, four R: 1.1 GB of vectors at a time."""
    run(tmp_path, """
from respackdev_amd.w3d import W3d
s = gen.make_system(a=7.0, nk=6, nocc=1, nvir=1, ecut_psi=30.0, seed=64)
wan, _ = gen.make_wannier(s, 9, 65)
w = from_system(s)
W = np.zeros((len(wan), 9, max(c.shape[1] for c in wan)), np.complex128)
for k, c in enumerate(wan):
    W[k, :, :c.shape[1]] = c
rs = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]
g = W3d(0)
g.open(w, 1.5, np.zeros(1, np.complex128))
g.set_wannier(W)
for iq, n in enumerate(g.set_q(w.ski)):
    g.set_epsinv(iq, 0.7 * np.eye(n, dtype=np.complex128)[None])
x1 = g.j3d(rs[:1])[0]
one = lim.alloc_live()
x4 = g.j3d(rs)[0]
assert one > 2 ** 20 and lim.alloc_live() <= one, (one, lim.alloc_live())
assert np.array_equal(x4, g.j3d(rs)[0])
assert np.abs(x4[0] - x1[0]).max() <= 5e-14 * np.abs(x1).max()
g.close()
assert lim.alloc_live() == 0, lim.alloc_live()
print("done")
""")


# chi in and eps^-1 out are 4.8 MiB each: by chunks over several threads
COPIES = """
c = opened(8.3, nk=2, nocc=2, nvir=3, ecut_psi=16.0)
n = len(c.prepare_q((0.0, 0.0, 0.5)))
rng = np.random.default_rng(48)
chi = 1e-3 * (rng.standard_normal((1, 14, n, n)) + 1j * rng.standard_normal((1, 14, n, n)))
assert chi.nbytes > 4 << 20
"""


def test_large_copies_without_pinned_memory(tmp_path):
    run(tmp_path, COPIES + """
lim.alloc_limits(ALL, 0)
plain = c.dyson_from(chi)
assert lim.alloc_refused() > 0
lim.alloc_limits(ALL, ALL)
assert np.array_equal(c.dyson_from(chi), plain)
c.close(); print("done")
""")


def test_pinned_arrays_take_no_chunks(tmp_path):
    run(tmp_path, COPIES + """
hip = C.CDLL("libamdhip64.so.7")
hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
hip.hipHostFree.argtypes = [C.c_void_p]
ps = [C.c_void_p(), C.c_void_p()]
for p in ps:
    assert hip.hipHostMalloc(C.byref(p), chi.nbytes, 0) == 0
a, b = [np.frombuffer((C.c_char * chi.nbytes).from_address(p.value), np.complex128).reshape(chi.shape)
        for p in ps]
a[:] = chi
lim.alloc_limits(ALL, 0)  # the handle has no chunks yet
_lib.check(_lib.lib().rp_chi_set(c._h, ps[0])); _lib.check(_lib.lib().rp_dyson(c._h, ps[1]))
assert lim.alloc_refused() == 0
lim.alloc_limits(ALL, ALL)
assert np.array_equal(c.dyson_from(chi), b)
c.close()
for p in ps:
    hip.hipHostFree(p)
print("done")
""")
