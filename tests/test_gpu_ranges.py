"""What the kernels keep over the whole range of their arguments: sums in a
fixed order, entries they must not read, sizes beyond one launch."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from conftest import crandn, rel
from gpu_util import Dev, init

pytestmark = pytest.mark.gpu
V, I64 = ctypes.c_void_p, ctypes.c_int64
EPS = 2.2e-16


@pytest.fixture(scope="module")
def L(pkg):
    return init(pkg)


def at(d, nbytes):
    """The device pointer nbytes into a buffer."""
    return V(d.p.value + nbytes)


@pytest.mark.parametrize("M", [3, 200, 256, 257, 300, 384, 385, 511, 512])
def test_colsum_order(L, pkg, M):
    """Up to 512 rows a column is the sum of at most two chunks of 256 rows
    (four row slots each), and so the same bits on every run: two addends onto
    zero in either order."""
    rng = np.random.default_rng(M)
    N = 70
    A = rng.standard_normal((M, N)).astype(np.float32)
    L.rsvdt_hip_colsum.argtypes = [I64, I64, V, I64, V, V]
    dA, out = Dev(pkg, A), Dev(pkg, np.full(N, np.nan, np.float32))
    ref = np.zeros(N, np.float32)
    for m0 in range(0, M, 256):
        slot = np.zeros((4, N), np.float32)
        for m in range(m0, min(m0 + 256, M)):
            slot[(m - m0) % 4] += A[m]
        ref += (slot[0] + slot[1]) + (slot[2] + slot[3])
    for _ in range(3):
        assert L.rsvdt_hip_colsum(M, N, dA.p, N, out.p, None) == 0
        assert np.array_equal(out.get(np.float32, (N,)), ref)


@pytest.mark.parametrize("n", [2, 17, 65, 140, 141])
def test_trmm_reads_the_upper_triangles(L, pkg, n):
    """Whatever lies below the diagonals is not read, and an infinite entry
    reaches only the entries that its row and column form."""
    rng = np.random.default_rng(n)
    A, B = crandn(rng, 3, n, n), crandn(rng, 3, n, n)
    low = np.tril_indices(n, -1)
    ref = np.triu(A) @ np.triu(B)
    A[0][low], B[1][low] = np.nan, np.inf
    A[2, 0, n - 1] = np.inf                # enters Out(0, n-1) alone
    dA, dB, dC = Dev(pkg, A), Dev(pkg, B), Dev(pkg, nbytes=A.nbytes)
    L.rsvdt_hip_btrmm_upper.argtypes = [I64, I64, V, V, V, V]
    assert L.rsvdt_hip_btrmm_upper(3, n, dA.p, dB.p, dC.p, None) == 0
    out = dC.get(np.complex128, A.shape)
    assert not np.isfinite(out[2, 0, n - 1])
    out[2, 0, n - 1] = ref[2, 0, n - 1] = 0
    assert np.max(np.abs(out - ref)) <= 8 * EPS * (n + 1) * 36        # |entries| < 6
    assert np.all(np.tril(out, -1) == 0)


def test_spmm_blocks_many_rows(L, pkg):
    """More rows than one launch has workgroups for (one row each above 128
    columns): the rows around the seam and at both ends."""
    rows, k, cols = (1 << 24) + 100, 171, 5
    rng = np.random.default_rng(1)
    at_rows = [0, (1 << 24) - 2, (1 << 24) - 1, 1 << 24, rows - 1]
    cnt = np.zeros(rows + 1, np.int32)
    cnt[np.array(at_rows) + 1] = 1
    rp = np.cumsum(cnt, dtype=np.int64).astype(np.int32)
    ci = np.arange(5, dtype=np.int32)
    v, x = crandn(rng, 5), crandn(rng, cols, k)
    held = [Dev(pkg, a) for a in (rp, ci, v, x)]
    out = Dev(pkg, nbytes=rows * k * 16)
    L.rsvdt_hip_spmm_blocks.argtypes = [I64] * 3 + [V, V, V, V, I64, V, I64, V]
    span = 4
    for r in at_rows:
        r0 = min(r, rows - span)
        nan = np.full((span, k), np.nan + 0j)
        assert L.rsvdt_hip_memcpy_h2d(at(out, r0 * k * 16), nan.ctypes.data_as(V), nan.nbytes) == 0
    assert L.rsvdt_hip_spmm_blocks(rows, k, 1, *[h.p for h in held], cols * k, out.p, rows * k, None) == 0
    for r in at_rows:
        r0 = min(r, rows - span)
        got = np.empty((span, k), complex)
        assert L.rsvdt_hip_memcpy_d2h(got.ctypes.data_as(V), at(out, r0 * k * 16), got.nbytes) == 0
        ref = np.zeros((span, k), complex)
        for q in range(span):
            if r0 + q in at_rows:
                e = at_rows.index(r0 + q)
                ref[q] = v[e] * x[e]
        assert np.max(np.abs(got - ref)) <= 4 * EPS * 36


def test_gemm_bf16_many_tiles(L, pkg):
    """More tiles of C than one grid dimension has workgroups for."""
    M, N = 65, (1 << 29) + 70
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    L.rsvdt_hip_mem_info.argtypes = [V, V]
    assert L.rsvdt_hip_mem_info(ctypes.byref(free), ctypes.byref(total)) == 0
    if free.value < 150e9:
        pytest.skip("needs 150 GB of device memory")
    a = np.arange(1, M + 1, dtype=np.float32)         # whole numbers: exact in BF16
    b = np.array([3], np.float32)
    dA, dB, dC = Dev(pkg, a), Dev(pkg, b), Dev(pkg, nbytes=M * N * 4)
    L.rsvdt_hip_gemm_bf16.argtypes = [I64] * 3 + [V, I64, I64, V, I64, I64, V, I64, ctypes.c_int, V, V, I64, V]
    places = [(0, 0), (0, (1 << 29) - 64), (0, N - 128), (64, 0), (64, (1 << 29) - 64), (64, N - 128)]
    for m, n in places:
        nan = np.full(128, np.nan, np.float32)
        assert L.rsvdt_hip_memcpy_h2d(at(dC, (m * N + n) * 4), nan.ctypes.data_as(V), nan.nbytes) == 0
    assert L.rsvdt_hip_gemm_bf16(M, N, 1, dA.p, 1, 1, dB.p, 1, 0, dC.p, N, 0, None, None, 0, None) == 0
    for m, n in places:
        got = np.empty(128, np.float32)
        assert L.rsvdt_hip_memcpy_d2h(got.ctypes.data_as(V), at(dC, (m * N + n) * 4), got.nbytes) == 0
        assert np.array_equal(got, np.full(128, 3.0 * a[m], np.float32))


def test_colsum_many_columns(L, pkg):
    """More columns than one launch has threads for: both ends."""
    M, N = 2, (1 << 30) + 72
    A = np.arange(M * 256, dtype=np.float32).reshape(M, 256)
    dA, out = Dev(pkg, nbytes=M * N * 4), Dev(pkg, nbytes=N * 4)
    L.rsvdt_hip_colsum.argtypes = [I64, I64, V, I64, V, V]
    places = [0, N - 256]
    for n in places:
        for m in range(M):
            assert L.rsvdt_hip_memcpy_h2d(at(dA, (m * N + n) * 4), A[m].ctypes.data_as(V), 1024) == 0
    assert L.rsvdt_hip_colsum(M, N, dA.p, N, out.p, None) == 0
    for n in places:
        got = np.empty(256, np.float32)
        assert L.rsvdt_hip_memcpy_d2h(got.ctypes.data_as(V), at(out, n * 4), 1024) == 0
        assert np.array_equal(got, A.sum(0))


def test_relayout_many_rows(L, pkg):
    """More rows than one launch has threads for: both ends, both ways."""
    rows, kb = (1 << 29) + 33, 1
    rng = np.random.default_rng(2)
    src, dst = Dev(pkg, nbytes=rows * 16), Dev(pkg, nbytes=rows * 16)
    x = crandn(rng, 100)
    L.rsvdt_hip_cm_relayout.argtypes = [I64] * 3 + [ctypes.c_int, I64, I64, V, V, ctypes.c_int, V]
    places = [0, rows - 100]
    for to_cm in (0, 1):
        for r in places:
            assert L.rsvdt_hip_memcpy_h2d(at(src, r * 16), x.ctypes.data_as(V), x.nbytes) == 0
            nan = np.full(100, np.nan + 0j)
            assert L.rsvdt_hip_memcpy_h2d(at(dst, r * 16), nan.ctypes.data_as(V), nan.nbytes) == 0
        cm, blk = (dst, src) if to_cm else (src, dst)
        assert L.rsvdt_hip_cm_relayout(rows, kb, 1, 0, 0, 1, cm.p, blk.p, to_cm, None) == 0
        for r in places:
            got = np.empty(100, complex)
            assert L.rsvdt_hip_memcpy_d2h(got.ctypes.data_as(V), at(dst, r * 16), got.nbytes) == 0
            assert np.array_equal(got, x)


@pytest.mark.parametrize("n", [16449, 23200])
def test_gram_many_tiles(L, pkg, n):
    """More macro tiles than one grid dimension takes, and more entries than
    one launch of the reduction: corners of X^H Z."""
    nr = 3
    rng = np.random.default_rng(n)
    X, Z = crandn(rng, nr, n), crandn(rng, nr, n)
    L.rsvdt_hip_bgram_work_bytes.restype = ctypes.c_size_t
    L.rsvdt_hip_bgram_work_bytes.argtypes = [I64] * 4
    L.rsvdt_hip_bgram.argtypes = [I64] * 4 + [V, I64, I64, I64, V, I64, I64, I64, V, V, V]
    dX, dZ, dG = Dev(pkg, X), Dev(pkg, Z), Dev(pkg, nbytes=n * n * 16)
    dw = Dev(pkg, nbytes=L.rsvdt_hip_bgram_work_bytes(1, nr, n, n))
    assert L.rsvdt_hip_bgram(1, nr, n, n, dX.p, nr * n, n, 1, dZ.p, nr * n, n, 1, dG.p, dw.p, None) == 0
    for a in (0, 63, n // 2, 16383, 16384, n - 2, n - 1):
        row = np.empty(n, complex)
        assert L.rsvdt_hip_memcpy_d2h(row.ctypes.data_as(V), at(dG, a * n * 16), row.nbytes) == 0
        assert np.max(np.abs(row - X[:, a].conj() @ Z)) <= 8 * EPS * nr * 36


@pytest.mark.parametrize("rows,k", [(700, 85), (700, 86), (515, 128), (515, 129), (300, 171), (300, 320), (300, 321),
                                    (40000, 121)])
@pytest.mark.parametrize("nb", [1, 2, 9])
def test_spmm_blocks_wide(L, pkg, rows, k, nb):
    """Lanes of several columns each (one block of 86 to 320 columns) and blocks
    of wide rows, with 0 to 7 entries a row: against scipy, and a block of a
    group the same bits as the block alone."""
    rng = np.random.default_rng(rows + k)
    cnt = rng.integers(0, 8, rows)
    rp = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    ci = np.concatenate([np.sort((rng.integers(rows) + np.arange(c)) % rows) for c in cnt]).astype(np.int32)
    v, x = crandn(rng, len(ci)), crandn(rng, nb, rows, k)
    held = [Dev(pkg, a) for a in (rp, ci, v)]
    dx, out, one = Dev(pkg, x), Dev(pkg, np.full((nb, rows, k), np.nan + 0j)), Dev(pkg, nbytes=rows * k * 16)
    L.rsvdt_hip_spmm_blocks.argtypes = [I64] * 3 + [V, V, V, V, I64, V, I64, V]
    p = [h.p for h in held]
    assert L.rsvdt_hip_spmm_blocks(rows, k, nb, *p, dx.p, rows * k, out.p, rows * k, None) == 0
    got = out.get(np.complex128, (nb, rows, k))
    M = sp.csr_matrix((v, ci, rp), shape=(rows, rows))
    for b in (0, nb - 1):
        assert np.max(np.abs(got[b] - M @ x[b])) <= 4 * 7 * EPS * 36      # sums of 7 products of |.| < 6 each
        assert L.rsvdt_hip_spmm_blocks(rows, k, 1, *p, at(dx, b * rows * k * 16), rows * k, one.p, rows * k, None) == 0
        assert np.array_equal(got[b], one.get(np.complex128, (rows, k)))


@pytest.mark.parametrize("rows,nb", [(4096, 8), (4096, 13), (4096, 33), (9000, 11), (70000, 17)])
def test_spmm_blocks_groups(L, pkg, rows, nb):
    """Two, three and eight blocks a workgroup, in groups of two and four that do
    not fill, entries walked again for each group, and outputs beyond the
    last-level cache (the last): every block the same bits as the block alone."""
    k = 16
    rng = np.random.default_rng(rows + nb)
    cnt = rng.integers(0, 6, rows)
    rp = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32)
    ci = rng.integers(0, rows, rp[-1]).astype(np.int32)
    v, x = crandn(rng, len(ci)), crandn(rng, nb, rows, k)
    held = [Dev(pkg, a) for a in (rp, ci, v)]
    dx, out, one = Dev(pkg, x), Dev(pkg, np.full((nb, rows, k), np.nan + 0j)), Dev(pkg, nbytes=rows * k * 16)
    L.rsvdt_hip_spmm_blocks.argtypes = [I64] * 3 + [V, V, V, V, I64, V, I64, V]
    p = [h.p for h in held]
    assert L.rsvdt_hip_spmm_blocks(rows, k, nb, *p, dx.p, rows * k, out.p, rows * k, None) == 0
    got = out.get(np.complex128, (nb, rows, k))
    M = sp.csr_matrix((v, ci, rp), shape=(rows, rows))
    for b in range(nb):
        assert L.rsvdt_hip_spmm_blocks(rows, k, 1, *p, at(dx, b * rows * k * 16), rows * k, one.p, rows * k, None) == 0
        assert np.array_equal(got[b], one.get(np.complex128, (rows, k)))
    assert np.max(np.abs(got[-1] - M @ x[-1])) <= 4 * 5 * EPS * 36


def test_transpose_beyond_cache(L, pkg):
    """Nontemporal row transposes, 290 MB a side, both ways."""
    N, n, kt, b0, kb = 35000, 65, 9, 1, 8
    rng = np.random.default_rng(3)
    src = rng.standard_normal((n, N, kt)) + 0j
    dS, dD, dB = Dev(pkg, src), Dev(pkg, nbytes=kb * N * n * 16), Dev(pkg, np.zeros_like(src))
    L.rsvdt_hip_transpose_rows.argtypes = [I64] * 5 + [V, V, ctypes.c_int, V]
    assert L.rsvdt_hip_transpose_rows(N, n, kt, b0, kb, dS.p, dD.p, 0, None) == 0
    assert np.array_equal(dD.get(np.complex128, (kb, N, n)), src[:, :, b0:].transpose(2, 1, 0))
    assert L.rsvdt_hip_transpose_rows(N, n, kt, b0, kb, dD.p, dB.p, 1, None) == 0
    src[:, :, 0] = 0
    assert np.array_equal(dB.get(np.complex128, src.shape), src)


@pytest.mark.parametrize("in_place", [False, True])
def test_apply_gram_beyond_cache(L, pkg, in_place):
    """Nontemporal rows of a CholeskyQR pass: 300 MB."""
    nb, nr, n = 2, 290001, 33
    rng = np.random.default_rng(4)
    X, C = crandn(rng, nb, nr, n), np.triu(crandn(rng, nb, n, n)) / np.sqrt(n)
    L.rsvdt_hip_bgram_work_bytes.restype = ctypes.c_size_t
    L.rsvdt_hip_bgram_work_bytes.argtypes = [I64] * 4
    L.rsvdt_hip_bapply_gram.argtypes = [I64] * 3 + [V, I64, I64, V, V, V, V, V]
    dX, dC, dG = Dev(pkg, X), Dev(pkg, C), Dev(pkg, nbytes=C.nbytes)
    dO = dX if in_place else Dev(pkg, nbytes=X.nbytes)
    dw = Dev(pkg, nbytes=L.rsvdt_hip_bgram_work_bytes(nb, nr, n, n))
    assert L.rsvdt_hip_bapply_gram(nb, nr, n, dX.p, nr * n, n, dC.p, dO.p, dG.p, dw.p, None) == 0
    out, G, ref = dO.get(np.complex128, X.shape), dG.get(np.complex128, C.shape), X @ C
    assert np.max(np.abs(out - ref)) <= 8 * EPS * n * np.abs(X).max() * np.abs(C).max()
    assert np.max(np.abs(G - ref.conj().transpose(0, 2, 1) @ ref)) <= 16 * EPS * nr * np.abs(ref).max() ** 2


class QrWork(ctypes.Structure):
    _fields_ = [(f, V) for f in ("G", "R", "Ri", "Ra", "Rt", "work", "info")]


@pytest.mark.parametrize("npass", [1, 2, 3])
@pytest.mark.parametrize("n", [16, 33, 64, 65])
def test_cholqr_from_another_array(L, pkg, n, npass):
    """CholeskyQR passes that start from an array of their own and end in X after
    odd and even numbers, with the product of their factors."""
    nb, nr = 2, 700
    rng = np.random.default_rng(n)
    X0 = crandn(rng, nb, nr, n)
    L.rsvdt_hip_bgram_work_bytes.restype = ctypes.c_size_t
    L.rsvdt_hip_bgram_work_bytes.argtypes = [I64] * 4
    mat = nb * n * n * 16
    d0, dX, dT, dR = Dev(pkg, X0), Dev(pkg, nbytes=X0.nbytes), Dev(pkg, nbytes=X0.nbytes), Dev(pkg, nbytes=mat)
    held = [Dev(pkg, nbytes=mat) for _ in range(5)] + [Dev(pkg, nbytes=L.rsvdt_hip_bgram_work_bytes(nb, nr, n, n)),
                                                       Dev(pkg, nbytes=256)]
    w = QrWork(*[h.p for h in held])
    f = L.rsvdt_cholqr_bufs
    f.argtypes = [I64] * 3 + [V, V, I64, I64, I64, V, ctypes.c_int, ctypes.c_int, ctypes.c_double, V, ctypes.c_size_t,
                              V, V, ctypes.c_int]
    assert f(nb, nr, n, d0.p, dX.p, nr * n, n, 1, dR.p, npass, 0, 0.0, dT.p, X0.nbytes, ctypes.byref(w), None, 0) == 0
    Q, R = dX.get(np.complex128, X0.shape), dR.get(np.complex128, (nb, n, n))
    assert np.array_equal(d0.get(np.complex128, X0.shape), X0)
    cond = max(np.linalg.cond(X0[b]) for b in range(nb))
    for b in range(nb):
        # one pass of CholeskyQR loses cond^2, two are at rounding
        assert np.max(np.abs(Q[b].conj().T @ Q[b] - np.eye(n))) <= 8 * n * EPS * (cond ** 2 if npass == 1 else 8)
        assert np.max(np.abs(Q[b] @ R[b] - X0[b])) <= 8 * n * EPS * np.linalg.norm(X0[b], 2) * 4
        assert np.all(np.tril(R[b], -1) == 0) and np.all(np.diag(R[b]).real > 0)


@pytest.mark.parametrize("n,drop", [(17, 3), (33, 5), (64, 9), (65, 9)])
def test_basis_of_dependent_columns(pkg, n, drop):
    """QRDecomposition of dependent columns (the second level of the span basis):
    orthonormal columns, zeros for what is left out, the span kept to rounding."""
    nr = 900
    rng = np.random.default_rng(n)
    X = crandn(rng, nr, n)
    where = rng.choice(n - 1, drop, replace=False) + 1
    for c in where:
        X[:, c] = X[:, :c] @ crandn(rng, c) / np.sqrt(c)
    m = pkg.mat_from_dense(np.asfortranarray(X), n)
    f = pkg.lib().QRDecomposition
    f.argtypes = [V]
    assert f(m) == 0
    Q = pkg.mat_to_dense(m)
    pkg.destroy(m)
    G = Q.conj().T @ Q
    live = np.diag(G).real > 0.5
    assert n - drop <= live.sum() <= n
    assert np.max(np.abs(G - np.diag(live.astype(float)))) <= 64 * n * EPS
    assert np.linalg.norm(X - Q @ (Q.conj().T @ X)) <= 64 * n * EPS * np.linalg.norm(X)
