"""Snapshot-to-snapshot stepping of small operators: when it is taken, and what
happens when it cannot be."""
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT, crandn, load_pkg, rel

pytestmark = pytest.mark.gpu

SHIM = """
#include <stddef.h>
static int (*next)(void **, size_t);
static size_t size;
static int skip, refused;
void shim_set(void *f, size_t bytes, int after) { next = (int (*)(void **, size_t))f; size = bytes; skip = after; }
int shim_refused(void) { return refused; }
int rsvdt_hip_malloc(void **p, size_t bytes)
{
    if (bytes == size && skip-- == 0) { refused++; *p = NULL; return 103; }
    return next(p, bytes);
}
"""


def operator(N, real, width=3):
    import scipy.sparse as sp
    rng = np.random.default_rng(N)
    offs = range(-(width // 2), width - width // 2)
    d = [rng.standard_normal(N - abs(o)) + (0 if real else 1j * rng.standard_normal(N - abs(o))) for o in offs]
    return (sp.diags(d, list(offs), shape=(N, N)) - (1 + width) * sp.eye(N)).tocsr().astype(np.complex128)


KW = dict(k=3, q=0, Nw=16, w=0.7, TL=1.0, dt=0.04)


def refusing(shim, what, removal):
    """Child process: one direct action with one allocation refused."""
    import ctypes
    S = ctypes.CDLL(shim, mode=ctypes.RTLD_GLOBAL)      # before the library, whose calls then bind to it
    pkg = load_pkg()
    L = pkg.lib()
    S.shim_set.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    real = ctypes.cast(L.rsvdt_hip_malloc, ctypes.c_void_p)
    S.shim_set(real, 0, 0)
    N = 301
    A = operator(N, True)
    out = {}
    for fuse in (0, 1):
        s = pkg.Session(A, transient_removal=removal, fuse_small=fuse, **KW)
        if not fuse:
            F = crandn(np.random.default_rng(0), N, s.k * s.Nw_eff)
        s.set_sketch(F)
        if fuse:        # the propagator, or the harmonic responses (as large as the forcing's two work blocks)
            S.shim_set(real, N * N * 16 if what == "E" else N * s.k * s.Nw_eff * 16, 0)
        s.direct()
        out[fuse] = s.get_Y()
        st = pkg.action_stats()
        s.close()
    assert S.shim_refused() == 1
    assert st["chunk_steps"] != s.RR, "the action leapt"
    assert rel(out[1], out[0]) < (1e-9 if removal else 1e-12)


@pytest.mark.parametrize("what", ["E", "H"])
@pytest.mark.parametrize("removal", [0, 1])
def test_steps_without_room_to_leap(tmp_path, what, removal):
    """When the propagator or the responses cannot be allocated the action steps
    one by one, as before the forcing was folded in place."""
    cc = shutil.which("gcc")
    if cc is None:
        pytest.skip("no C compiler")
    (tmp_path / "shim.c").write_text(SHIM)
    so = str(tmp_path / "shim.so")
    subprocess.run([cc, "-shared", "-fPIC", "-O1", "-o", so, str(tmp_path / "shim.c")], check=True)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), so, what, str(removal)], cwd=ROOT, timeout=100,
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]


def action(pkg, A, removal=False, fuse=1, F=None, **kw):
    s = pkg.Session(A, transient_removal=removal, fuse_small=fuse, q=0, w=0.7, **kw)
    if F is None:
        F = crandn(np.random.default_rng(1), A.shape[0], s.k * s.Nw_eff)
    s.set_sketch(F)
    s.direct()
    out, st = s.get_Y(), pkg.action_stats()
    leapt = st["chunk_steps"] == s.RR and st["rk4_launches"] < st["steps"]
    s.close()
    return out, F, leapt


def steps(n):
    """The step size of n steps a period, at w = 0.7."""
    return 2 * np.pi / 0.7 / n


@pytest.mark.parametrize("N,real,k,Nw,RR,leaps", [
    (64, True, 1, 64, 8, False),         # 64 products of 5 us, 512 steps of 0.5 us
    (1024, True, 10, 64, 8, False),      # 13 us, 1.5 us
    (600, True, 100, 16, 6, False),
    (64, True, 1, 64, 24, True),
    (500, False, 10, 64, 16, True),
    (1100, False, 10, 16, 32, True),     # rows beyond the stepper's registers
    (1300, True, 33, 32, 24, True),
])
def test_leap_rule(pkg, N, real, k, Nw, RR, leaps):
    """Leaps where products cost less than steps, steps where they do not; both
    give the stage kernels' result."""
    A = operator(N, real)
    kw = dict(k=k, Nw=Nw, TL=0.0, dt=steps(Nw * RR) * 1.0001)
    out, F, leapt = action(pkg, A, **kw)
    assert leapt == leaps
    ref, _, _ = action(pkg, A, fuse=0, F=F, **kw)
    assert rel(out, ref) < 1e-12


@pytest.mark.parametrize("N,k,Nw,RR", [(1024, 64, 16, 12), (500, 10, 16, 32), (1100, 3, 16, 32)])
def test_leap_rule_removal(pkg, N, k, Nw, RR):
    """The removal's e^{A dT} of a leaping action: as products of the whole basis
    (the second) or, where these cost more, as steps."""
    A = operator(N, True)
    kw = dict(k=k, Nw=Nw, TL=1.0, dt=steps(Nw * RR) * 1.0001)
    out, F, leapt = action(pkg, A, removal=True, **kw)
    assert leapt
    ref, _, _ = action(pkg, A, removal=True, fuse=0, F=F, **kw)
    assert rel(out, ref) < 1e-9


def test_chunk_option(pkg):
    """Chunks of a size the caller sets are chunks of steps."""
    A = operator(64, True)
    kw = dict(k=3, Nw=16, TL=1.0, dt=0.04)
    ref, F, leapt = action(pkg, A, **kw)
    assert leapt
    out, _, leapt = action(pkg, A, F=F, chunk_steps=7, **kw)
    assert not leapt and pkg.action_stats()["chunk_steps"] == 7
    assert rel(out, ref) < 1e-12


def test_stats_name_the_shape(pkg):
    """The launch shape that the statistics name does not depend on the way."""
    A = operator(64, True)
    kw = dict(k=3, Nw=16, TL=1.0, dt=0.04)
    shape = {}
    for chunk in (0, 7):
        _, _, leapt = action(pkg, A, chunk_steps=chunk, **kw)
        assert leapt == (chunk == 0)
        st = pkg.action_stats()
        shape[chunk] = [st[f] for f in ("spmm_lanes", "spmm_variant", "spmm_xcd_remap", "rk4_form")]
    assert shape[0] == shape[7] and shape[7][1:3] == [3, 1]


@pytest.mark.parametrize("direct", [True, False])
def test_propagator_follows_the_steps(pkg, direct):
    """One Mat stepped with one step size, another, another number of steps and the
    first again: the kept propagator is the one of the call."""
    A = operator(200, False)
    first = pkg.Session(A, q=0, w=0.7, transient_removal=False, k=4, Nw=16, TL=1.0, dt=0.04)
    for Nw, dt in ((16, 0.04), (16, 0.02), (8, 0.02), (16, 0.04)):
        kw = dict(q=0, w=0.7, transient_removal=False, k=4, Nw=Nw, TL=1.0, dt=dt)
        s = pkg.Session(A, **kw)
        own, s.LNS.A = s.LNS.A, first.LNS.A
        F = crandn(np.random.default_rng(Nw), 200, 4 * s.Nw_eff)
        s.set_sketch(F)
        s.direct() if direct else s.adjoint()
        out = s.get_Y()
        assert pkg.action_stats()["rk4_launches"] < s.Ns // 4
        s.LNS.A = own
        s.set_sketch(F)
        s.direct() if direct else s.adjoint()
        assert np.array_equal(out, s.get_Y())      # a Mat of its own: the same kernels, the same bits
        s.close()
    first.close()


if __name__ == "__main__":
    refusing(sys.argv[1], sys.argv[2], bool(int(sys.argv[3])))
