"""Kernels whose launch shape follows the size, at the sizes where the shape
changes: tile edges, remainders, the smallest and largest of each range."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from conftest import crandn, rel
from gpu_util import Desc, Dev, init, tiled_form

pytestmark = pytest.mark.gpu
V, I64 = ctypes.c_void_p, ctypes.c_int64
EPS = 2.2e-16


@pytest.fixture(scope="module")
def L(pkg):
    return init(pkg)


@pytest.mark.parametrize("n", [1, 2, 3, 15, 16, 17, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("rank_def", [False, True])
def test_jacobi_svd_sizes(L, pkg, n, rank_def):
    """Singular values against numpy, U orthonormal and diagonalising R R^H
    (a graded spectrum over four decades; with a zero column when rank_def)."""
    rng = np.random.default_rng(n)
    nb = 3
    s = 10.0 ** (-4.0 * (np.arange(n) + 0.3 * rng.random((nb, n))) / n)
    R = np.stack([np.triu(np.linalg.qr((np.linalg.qr(crandn(rng, n, n))[0] * s[b]) @ crandn(rng, n, n))[1])
                  for b in range(nb)])
    if rank_def:
        R[:, :, n // 2] = 0
    dR, dU, ds = Dev(pkg, R), Dev(pkg, nbytes=R.nbytes), Dev(pkg, nbytes=nb * n * 8)
    L.rsvdt_hip_bjacobi_svd.argtypes = [I64, I64, V, V, V, V]
    assert L.rsvdt_hip_bjacobi_svd(nb, n, dR.p, dU.p, ds.p, None) == 0
    U, sg = dU.get(np.complex128, R.shape), ds.get(np.float64, (nb, n))
    tol = 40 * n * EPS
    for b in range(nb):
        ref = np.linalg.svd(R[b], compute_uv=False)
        top = max(ref[0], 1e-300)
        assert np.max(np.abs(sg[b] - ref)) <= tol * top
        live = sg[b] > tol * top
        Ul = U[b][:, live]
        assert np.max(np.abs(Ul.conj().T @ Ul - np.eye(live.sum())), initial=0.0) <= tol
        D = Ul.conj().T @ (R[b] @ R[b].conj().T) @ Ul
        assert np.max(np.abs(D - np.diag(sg[b][live] ** 2)), initial=0.0) <= tol * top * top
        t = Ul.sum(axis=0)
        big = np.abs(t) > 1e-7
        assert np.all(t.real[big] > 0) and np.all(np.abs(t.imag[big]) <= tol * np.sqrt(n))


@pytest.mark.parametrize("na,nc", [(1, 1), (16, 16), (17, 17), (20, 20), (32, 32), (33, 33), (48, 48), (49, 49),
                                   (64, 64), (65, 65), (81, 81), (129, 129), (65, 17), (17, 65), (33, 65), (65, 32),
                                   (40, 64), (64, 40)])
@pytest.mark.parametrize("nb,nr", [(1, 3), (3, 515), (2, 4100)])
@pytest.mark.parametrize("same", [False, True])
def test_gram_tiles(L, pkg, na, nc, nb, nr, same):
    """X^H Z for the macro tiles, the border column (n = 16 T + 1) and the
    triangle of X^H X, on rows that do not fill the waves' steps."""
    if same and na != nc:
        pytest.skip("the triangle needs X = Z")
    rng = np.random.default_rng(na * 1000 + nc + nr)
    X = crandn(rng, nb, nr, na)
    Z = X if same else crandn(rng, nb, nr, nc)
    L.rsvdt_hip_bgram_work_bytes.restype = ctypes.c_size_t
    L.rsvdt_hip_bgram_work_bytes.argtypes = [I64] * 4
    L.rsvdt_hip_bgram.argtypes = [I64] * 4 + [V, I64, I64, I64, V, I64, I64, I64, V, V, V]
    dX = Dev(pkg, X)
    dZ = dX if same else Dev(pkg, Z)
    dG = Dev(pkg, nbytes=nb * na * nc * 16)
    dw = Dev(pkg, nbytes=L.rsvdt_hip_bgram_work_bytes(nb, nr, na, nc))
    for _ in range(2):
        assert L.rsvdt_hip_bgram(nb, nr, na, nc, dX.p, nr * na, na, 1, dZ.p, nr * nc, nc, 1, dG.p, dw.p, None) == 0
    G = dG.get(np.complex128, (nb, na, nc))
    ref = np.einsum("bra,brc->bac", X.conj(), Z)
    # each entry: nr products of modulus ~1, rounded sums of 4 nr real terms
    assert np.max(np.abs(G - ref)) <= 8 * EPS * np.sqrt(nr) * (np.abs(X).max() * np.abs(Z).max()) * np.sqrt(nr)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("nb,nr", [(1, 3), (3, 515), (2, 4100)])
@pytest.mark.parametrize("in_place", [False, True])
def test_apply_gram(L, pkg, n, nb, nr, in_place):
    """Out = X C (C upper triangular) and Out^H Out from one pass, and the
    apply alone, against numpy."""
    rng = np.random.default_rng(n + nr)
    X, C = crandn(rng, nb, nr, n), np.triu(crandn(rng, nb, n, n)) / np.sqrt(n)
    ref = np.einsum("bra,bac->brc", X, C)
    G_ref = np.einsum("bra,brc->bac", ref.conj(), ref)
    L.rsvdt_hip_bgram_work_bytes.restype = ctypes.c_size_t
    L.rsvdt_hip_bgram_work_bytes.argtypes = [I64] * 4
    L.rsvdt_hip_bapply_gram.argtypes = [I64] * 3 + [V, I64, I64, V, V, V, V, V]
    for with_gram in (True, False):
        dX, dC = Dev(pkg, X), Dev(pkg, C)
        dO = dX if in_place else Dev(pkg, nbytes=X.nbytes)
        dG = Dev(pkg, nbytes=C.nbytes)
        dw = Dev(pkg, nbytes=L.rsvdt_hip_bgram_work_bytes(nb, nr, n, n))
        assert L.rsvdt_hip_bapply_gram(nb, nr, n, dX.p, nr * n, n, dC.p, dO.p, dG.p if with_gram else None,
                                       dw.p, None) == 0
        out = dO.get(np.complex128, X.shape)
        # sums of 4 n real products of size max|X| max|C|
        assert np.max(np.abs(out - ref)) <= 8 * EPS * n * np.abs(X).max() * np.abs(C).max()
        if with_gram:
            assert np.max(np.abs(dG.get(np.complex128, C.shape) - G_ref)) <= 16 * EPS * nr * np.abs(ref).max() ** 2


def test_apply_gram_rejects_wide(L, pkg):
    d = Dev(pkg, nbytes=1 << 16)
    L.rsvdt_hip_bapply_gram.argtypes = [I64] * 3 + [V, I64, I64, V, V, V, V, V]
    assert L.rsvdt_hip_bapply_gram(1, 4, 65, d.p, 260, 65, d.p, d.p, None, None, None) == 102
    assert L.rsvdt_hip_bapply_gram(1, 4, 8, d.p, 32, 8, d.p, d.p, d.p, None, None) == 102


@pytest.mark.parametrize("N", [1, 3, 15, 16, 17, 33, 130, 515])
@pytest.mark.parametrize("k,nb", [(1, 1), (10, 1), (16, 1), (17, 2), (16, 16), (257, 1), (13, 25)])
def test_dense_apply_sizes(L, pkg, N, k, nb):
    rng = np.random.default_rng(N + k)
    E, X, F = crandn(rng, N, N) / np.sqrt(N), crandn(rng, nb, N, k), crandn(rng, nb, N, k)
    L.rsvdt_hip_dense_apply.argtypes = [I64] * 3 + [V] * 5
    dE, dX, dF, dO = Dev(pkg, E), Dev(pkg, X), Dev(pkg, F), Dev(pkg, nbytes=X.nbytes)
    for f in (None, dF):
        assert L.rsvdt_hip_dense_apply(N, k, nb, dE.p, dX.p, f.p if f else None, dO.p, None) == 0
        ref = np.einsum("ra,bac->brc", E, X) + (F if f else 0)
        assert np.max(np.abs(dO.get(np.complex128, X.shape) - ref)) <= 8 * EPS * (N + 1) * np.abs(E).max() * np.abs(X).max() + 4 * EPS * np.abs(F).max()
    assert L.rsvdt_hip_dense_apply(N, k, nb, dE.p, dX.p, None, dX.p, None) == 102      # never in place


def _band_operator(N, real, width, rng):
    import scipy.sparse as sp
    offs = range(-(width // 2), width // 2 + 1)
    d = [rng.standard_normal(max(N - abs(o), 0)) + (0 if real else 1j * rng.standard_normal(max(N - abs(o), 0)))
         for o in offs]
    return (sp.diags(d, list(offs), shape=(N, N)) - (1 + width) * sp.eye(N)).tocsr().astype(np.complex128)


@pytest.mark.parametrize("N,real,width", [(20, False, 3), (64, True, 3), (129, False, 7), (500, False, 3), (700, True, 5)])
@pytest.mark.parametrize("k,Nw,TL,removal", [(1, 8, 0.0, False), (3, 16, 1.0, True), (16, 15, 2.37, False), (5, 16, 7.9, True)])
@pytest.mark.parametrize("direct", [True, False])
def test_leaps_match_steps(pkg, N, real, width, k, Nw, TL, removal, direct):
    """Snapshots by dense propagator products (one per snapshot) against the
    stage kernels' step-by-step run: whole and partial leaps before the first
    snapshot, none at all, odd numbers of frequencies, both directions."""
    if removal and Nw + 1 > N:
        pytest.skip("more snapshots than rows")
    rng = np.random.default_rng(N + k)
    A = _band_operator(N, real, width, rng)
    kw = dict(k=k, q=0, Nw=Nw, w=0.7, TL=TL, dt=0.04, transient_removal=removal)
    out = {}
    for fuse in (1, 0):
        s = pkg.Session(A, fuse_small=fuse, **kw)
        if fuse == 1:
            F = crandn(rng, N, k * s.Nw_eff)
        s.set_sketch(F)
        s.direct() if direct else s.adjoint()
        out[fuse] = s.get_Y()
        st = pkg.action_stats()
        if fuse:
            assert st["chunk_steps"] == s.RR and st["rk4_launches"] < st["steps"] // 2
        s.close()
    assert rel(out[1], out[0]) < (1e-9 if removal else 1e-12)


@pytest.mark.parametrize("na,nc", [(1, 1), (5, 17), (16, 16), (33, 48), (65, 65), (65, 32), (65, 33), (64, 64), (129, 129),
                                   (129, 64), (140, 65), (146, 64), (146, 97), (4, 200)])
@pytest.mark.parametrize("nb,nr", [(1, 3), (3, 515), (2, 4100)])
@pytest.mark.parametrize("with_y", [False, True])
def test_apply_tiles(L, pkg, na, nc, nb, nr, with_y):
    """Out = alpha Y + X C over column tiles, the border column and row
    remainders; the entries of X past a row's end (the next row, or NaN after
    the last) must not reach the result."""
    rng = np.random.default_rng(na * 7 + nc + nr)
    X, C, Y = crandn(rng, nb, nr, na), crandn(rng, nb, na, nc) / np.sqrt(na), crandn(rng, nb, nr, nc)
    pad = np.full(64, np.nan + 1j * np.nan)
    dX, dC, dY = Dev(pkg, np.concatenate([X.ravel(), pad])), Dev(pkg, C), Dev(pkg, Y)
    dO = Dev(pkg, nbytes=Y.nbytes)
    L.rsvdt_hip_bapply.argtypes = [I64] * 4 + [V, I64, I64, I64, V, ctypes.c_double, V, I64, I64, I64, V, I64, I64, I64, V]
    assert L.rsvdt_hip_bapply(nb, nr, na, nc, dX.p, nr * na, na, 1, dC.p, 0.5, dY.p if with_y else None, nr * nc, nc, 1,
                              dO.p, nr * nc, nc, 1, None) == 0
    ref = np.einsum("bra,bac->brc", X, C) + (0.5 * Y if with_y else 0)
    assert np.max(np.abs(dO.get(np.complex128, Y.shape) - ref)) <= 8 * EPS * (na + 1) * np.abs(X).max() * max(np.abs(C).max(), 1)


@pytest.mark.parametrize("n", [1, 16, 17, 65, 140, 141, 150])
def test_trmm_sizes(L, pkg, n):
    rng = np.random.default_rng(n)
    A, B = np.triu(crandn(rng, 3, n, n)), np.triu(crandn(rng, 3, n, n))
    dA, dB, dC = Dev(pkg, A), Dev(pkg, B), Dev(pkg, nbytes=A.nbytes)
    L.rsvdt_hip_btrmm_upper.argtypes = [I64, I64, V, V, V, V]
    assert L.rsvdt_hip_btrmm_upper(3, n, dA.p, dB.p, dC.p, None) == 0
    out = dC.get(np.complex128, A.shape)
    assert np.max(np.abs(out - A @ B)) <= 8 * EPS * (n + 1) * np.abs(A).max() * np.abs(B).max()
    assert np.all(np.tril(out, -1) == 0)


@pytest.mark.parametrize("n,kt,b0,kb", [(1, 1, 0, 1), (65, 16, 8, 8), (65, 9, 2, 7), (3, 100, 1, 60), (129, 32, 0, 32),
                                        (17, 5, 4, 1), (2, 3, 0, 3), (481, 16, 0, 16)])
@pytest.mark.parametrize("N", [1, 2, 515])
def test_transpose_row_groups(L, pkg, n, kt, b0, kb, N):
    rng = np.random.default_rng(n + N)
    src = crandn(rng, n, N, kt)
    dS, dD, dB = Dev(pkg, src), Dev(pkg, nbytes=kb * N * n * 16), Dev(pkg, np.zeros_like(src))
    L.rsvdt_hip_transpose_rows.argtypes = [I64] * 5 + [V, V, ctypes.c_int, V]
    assert L.rsvdt_hip_transpose_rows(N, n, kt, b0, kb, dS.p, dD.p, 0, None) == 0
    assert np.array_equal(dD.get(np.complex128, (kb, N, n)), src[:, :, b0:b0 + kb].transpose(2, 1, 0))
    assert L.rsvdt_hip_transpose_rows(N, n, kt, b0, kb, dD.p, dB.p, 1, None) == 0
    back = np.zeros_like(src)
    back[:, :, b0:b0 + kb] = src[:, :, b0:b0 + kb]
    assert np.array_equal(dB.get(np.complex128, src.shape), back)


@pytest.mark.parametrize("ntile,nb,bpw", [(63, 2, 8), (64, 3, 1), (511, 3, 2), (513, 2, 1), (1100, 3, 8)])
def test_tiles_of_several_blocks(L, pkg, ntile, nb, bpw):
    """The Horner stage on several blocks, its tiles dealt to the XCDs in runs
    (one run each, or runs of 64 and a rest): every tile once, no tile twice."""
    rng = np.random.default_rng(ntile)
    N, k, c = 32 * ntile - 5, 6, 0.03
    A = sp.diags([rng.standard_normal(N - abs(o)) for o in (-40, -1, 0, 1, 40)], [-40, -1, 0, 1, 40], format="csr")
    y = crandn(rng, nb, N, k)
    tptr, tcol, lidx, hmax, emax = tiled_form(A, 32)
    held = [Dev(pkg, x) for x in (A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, tptr, tcol, lidx, y)]
    rp, ci, v, tp, tc, li, dy = (h.p for h in held)
    out = Dev(pkg, nbytes=y.nbytes)
    d = Desc(N, k, nb, rp, ci, v, 1, 64, 8, 0, 9, 0, None, None, None, 32, hmax, emax, tp, tc, li, bpw)
    L.rsvdt_hip_horner_stage.argtypes = [ctypes.POINTER(Desc), V, V, V, V, ctypes.c_double, V, V, V]
    assert L.rsvdt_hip_horner_stage(ctypes.byref(d), dy, dy, None, None, c, out.p, None, None) == 0
    ref = np.stack([y[b] + c * (A @ y[b]) for b in range(nb)])
    assert rel(out.get(np.complex128, y.shape), ref) < 1e-14


@pytest.mark.parametrize("off,pad", [(0, 0), (0, 4), (1, 0), (0, 3)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (64, 64, 64), (68, 60, 68), (65, 63, 66), (132, 72, 130), (40, 64, 4100)])
@pytest.mark.parametrize("ak,bk", [(True, True), (True, False), (False, True), (False, False)])
def test_gemm_bf16_loads(L, pkg, M, N, K, ak, bk, off, pad):
    """Both load widths of the BF16 GEMM: operands on and off a 16-byte
    boundary (off), padded leading dimensions (pad), K-steps and tiles that do
    not divide, and a split reduction."""
    rng = np.random.default_rng(M + K)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)

    def put(X):                        # row-major with a padded row, `off` floats into its buffer
        ld = X.shape[1] + pad
        buf = np.full(off + X.shape[0] * ld, np.nan, np.float32)
        buf[off:].reshape(X.shape[0], ld)[:, :X.shape[1]] = X
        d = Dev(pkg, buf)
        return d, d.p.value + 4 * off if isinstance(d.p, V) else d.p + 4 * off, ld

    dA, pA, lda = put(A if ak else A.T)
    dB, pB, ldb = put(B.T if bk else B)
    dC = Dev(pkg, nbytes=M * N * 4)
    L.rsvdt_hip_gemm_bf16.argtypes = [I64] * 3 + [V, I64, I64, V, I64, I64, V, I64, ctypes.c_int, V, V, I64, V]
    assert L.rsvdt_hip_gemm_bf16(M, N, K, pA, lda if ak else 1, 1 if ak else lda, pB, 1 if bk else ldb,
                                 ldb if bk else 1, dC.p, N, 0, None, None, 0, None) == 0

    def bf16(X):
        u = X.view(np.uint32).astype(np.uint64)
        return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32).astype(np.float64)
    ref = bf16(A) @ bf16(B)
    assert np.max(np.abs(dC.get(np.float32, (M, N)) - ref)) <= 6e-8 * 4 * np.sqrt(K) * max(1.0, np.max(np.abs(ref)))


@pytest.mark.parametrize("M", [1, 3, 31, 127, 128, 129, 1000])
@pytest.mark.parametrize("N,lda", [(1, 1), (63, 70), (64, 64), (200, 200)])
def test_colsum_sizes(L, pkg, M, N, lda):
    """Column sums over row chunks that the four row slots do not divide."""
    rng = np.random.default_rng(M + N)
    A = rng.standard_normal((M, lda)).astype(np.float32)
    dA, out = Dev(pkg, A), Dev(pkg, np.full(N, np.nan, np.float32))
    L.rsvdt_hip_colsum.argtypes = [I64, I64, V, I64, V, V]
    assert L.rsvdt_hip_colsum(M, N, dA.p, lda, out.p, None) == 0
    ref = A[:, :N].astype(np.float64).sum(0)
    assert np.max(np.abs(out.get(np.float32, (N,)) - ref)) <= 6e-8 * M * np.max(np.abs(A))


@pytest.mark.parametrize("P,K,ncol", [(1, 1, 1), (5, 3, 65), (16, 4, 63), (17, 5, 64), (64, 52, 700), (31, 3, 140001),
                                      (64, 64, 133000), (130, 20, 1000)])
@pytest.mark.parametrize("prec,beta", [(64, 0.0), (64, 0.5), (32, 0.0)])
def test_coef_gemm_stream(L, pkg, P, K, ncol, prec, beta):
    """The streamed coefficient product: fewer and more K-steps than are in
    flight, one and several column tiles a workgroup, ragged last tiles."""
    rng = np.random.default_rng(P + K + ncol)
    cmod = P + 3
    C, X, Y = crandn(rng, K, cmod), crandn(rng, K, ncol), crandn(rng, P, ncol)
    cdt = np.complex128 if prec == 64 else np.complex64
    dC, dX, dY = Dev(pkg, C), Dev(pkg, X), Dev(pkg, Y.astype(cdt))
    L.rsvdt_hip_coef_gemm.argtypes = [I64, I64, I64, V, I64, I64, I64, ctypes.c_int, I64, ctypes.c_double, V, I64, V,
                                      I64, ctypes.c_int, ctypes.c_double, V]
    assert L.rsvdt_hip_coef_gemm(P, K, ncol, dC.p, cmod, 1, 2, -1, cmod, 0.7, dX.p, ncol, dY.p, ncol, prec, beta,
                                 None) == 0
    ref = 0.7 * (C[:, (2 - np.arange(P)) % cmod].T @ X) + beta * Y
    tol = (4 * K * EPS if prec == 64 else 2.4e-7) * max(1.0, np.max(np.abs(ref)))
    assert np.max(np.abs(dY.get(cdt, (P, ncol)) - ref)) <= tol


@pytest.mark.parametrize("rows,cols,k,nb", [(1, 1, 1, 1), (37, 90, 7, 3), (500, 500, 64, 4), (513, 200, 100, 5),
                                            (33, 40, 256, 2), (20, 31, 257, 6), (70000, 70000, 3, 9)])
@pytest.mark.parametrize("wmax", [0, 1, 2, 7])
def test_spmm_blocks_shapes(L, pkg, rows, cols, k, nb, wmax):
    """Out_b = M In_b with 0 .. wmax entries a row (empty rows among them), for
    rows that do not fill a workgroup and blocks that do not fill a group."""
    rng = np.random.default_rng(rows + wmax)
    cnt = rng.integers(0, min(wmax, cols) + 1, rows)
    rp = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    ci = np.concatenate([np.sort((rng.integers(cols) + np.arange(c)) % cols) for c in cnt] + [[0]]).astype(np.int32)
    v, x = crandn(rng, len(ci)), crandn(rng, nb, cols, k)
    M = sp.csr_matrix((v[:-1], ci[:-1], rp), shape=(rows, cols))
    held = [Dev(pkg, a) for a in (rp, ci, v, x)]
    out = Dev(pkg, np.full((nb, rows, k), np.nan + 0j))
    L.rsvdt_hip_spmm_blocks.argtypes = [I64] * 3 + [V, V, V, V, I64, V, I64, V]
    assert L.rsvdt_hip_spmm_blocks(rows, k, nb, *[h.p for h in held], cols * k, out.p, rows * k, None) == 0
    got = out.get(np.complex128, (nb, rows, k))
    ref = np.stack([M @ x[b] for b in range(nb)])
    assert np.max(np.abs(got - ref)) <= 30 * EPS * max(wmax, 1) * 4


@pytest.mark.parametrize("rows,cols,kb", [(1, 1, 1), (5, 6, 3), (31, 40, 10), (32, 64, 32), (33, 66, 33), (500, 640, 10),
                                          (70001, 66, 2), (4200003, 3, 3)])
def test_dense_round_trip(L, pkg, rows, cols, kb):
    """A host matrix to blocks on the device and back: the blocks' layout and
    every entry, for ragged tiles and more columns than one transfer takes."""
    rng = np.random.default_rng(rows)
    F = np.asfortranarray(rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols)))
    m = pkg.mat_from_dense(F, kb)
    assert np.array_equal(pkg.mat_to_dense(m), F)
    pkg.destroy(m)
    if rows * cols > 10 ** 6:
        return
    nblk = cols // kb
    dc, db = Dev(pkg, np.ascontiguousarray(F.T)), Dev(pkg, nbytes=F.nbytes)
    L.rsvdt_hip_cm_relayout.argtypes = [I64] * 3 + [ctypes.c_int, I64, I64, V, V, ctypes.c_int, V]
    for order in (0, 1):
        assert L.rsvdt_hip_cm_relayout(rows, kb, nblk, order, 0, cols, dc.p, db.p, 0, None) == 0
        c = np.arange(cols).reshape((nblk, kb) if order == 0 else (kb, nblk))
        ref = F[:, c if order == 0 else c.T].transpose(1, 0, 2)
        assert np.array_equal(db.get(np.complex128, (nblk, rows, kb)), ref)
        back = Dev(pkg, nbytes=F.nbytes)
        assert L.rsvdt_hip_cm_relayout(rows, kb, nblk, order, 0, cols, back.p, db.p, 1, None) == 0
        assert np.array_equal(back.get(np.complex128, (cols, rows)), F.T)


@pytest.mark.parametrize("M,N,K", [(64 * 7, 190, 40), (64 * 8, 190, 40), (64 * 17 - 3, 70, 20), (130, 70, 64 * 72)])
def test_gemm_bf16_tile_order(L, pkg, M, N, K):
    """Fewer than eight, eight, and eight and a rest of the groups of tiles (or
    of splits) that go to one XCD: every tile of C once."""
    rng = np.random.default_rng(M)
    A, B = (rng.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (K, N)))
    dA, dB, dC = Dev(pkg, A), Dev(pkg, B), Dev(pkg, np.full((M, N), np.nan, np.float32))
    L.rsvdt_hip_gemm_bf16.argtypes = [I64] * 3 + [V, I64, I64, V, I64, I64, V, I64, ctypes.c_int, V, V, I64, V]
    assert L.rsvdt_hip_gemm_bf16(M, N, K, dA.p, K, 1, dB.p, N, 1, dC.p, N, 0, None, None, 0, None) == 0
    assert np.array_equal(dC.get(np.float32, (M, N)), A @ B)     # whole numbers: exact


@pytest.mark.parametrize("kb,k,Nw,Nwe", [(1, 1, 1, 1), (2, 5, 8, 4), (3, 3, 15, 15), (4, 7, 64, 32), (1, 2, 300, 300)])
@pytest.mark.parametrize("direct", [True, False])
def test_removal_windows(L, pkg, kb, k, Nw, Nwe, direct):
    """The Galerkin projection's window coefficients and shifts against numpy."""
    rng = np.random.default_rng(Nw)
    dft, RR, sw, dT = crandn(rng, Nw, Nwe), 16.0, 0.05 if direct else -0.05, 1.9
    dd, dC, dp = Dev(pkg, dft), Dev(pkg, nbytes=2 * kb * (Nw + 1) * Nwe * 16), Dev(pkg, nbytes=k * Nwe * 16)
    D = ctypes.c_double
    L.rsvdt_hip_tr_windows.argtypes = [I64] * 4 + [V, D, D, D, ctypes.c_int, ctypes.c_int, V, V, V]
    w1, w2 = (0, 1) if direct else (1, 0)
    assert L.rsvdt_hip_tr_windows(kb, k, Nw, Nwe, dd.p, RR, sw, dT, w1, w2, dC.p, dp.p, None) == 0
    C, ph = dC.get(np.complex128, (2, kb, Nw + 1, Nwe)), dp.get(np.complex128, (k, Nwe))
    ref = np.exp(1j * (sw * np.arange(Nwe) * dT))
    d = np.zeros((2, Nw + 1, Nwe), complex)
    d[0, w1:w1 + Nw], d[1, w2:w2 + Nw] = RR * dft, RR * dft
    assert np.max(np.abs(ph - ref)) <= 2 * EPS
    assert np.array_equal(C[0], np.broadcast_to(d[0], C[0].shape))
    assert np.max(np.abs(C[1] - (ref * d[0] - d[1]))) <= 6 * EPS * np.max(np.abs(d))
