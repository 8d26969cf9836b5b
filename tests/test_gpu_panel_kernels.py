"""The panel kernels of the factorizations at the sizes and values where they
branch: block edges, ragged last blocks, pivots outside the range of the fast
reciprocal square root, failed pivots.  References are numpy in FP64."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Dev:
    """A host array's device copy (column-major)."""

    def __init__(self, dm, a):
        self.dm = dm
        self.a = np.asfortranarray(a)
        self.buf = dm.DeviceBuffer(max(self.a.nbytes, 8))
        if self.a.nbytes:
            dm._lib.call("dm_memcpy_h2d", C.c_void_p(self.buf.ptr),
                         self.a.ctypes.data_as(C.c_void_p), C.c_size_t(self.a.nbytes), None)

    @property
    def p(self):
        return C.c_void_p(self.buf.ptr)

    def get(self):
        out = np.empty_like(self.a, order="F")
        if out.nbytes:
            self.dm._lib.call("dm_memcpy_d2h", out.ctypes.data_as(C.c_void_p), self.p,
                              C.c_size_t(out.nbytes), None)
        return out


def _spd(n, dtype, seed):
    rng = np.random.default_rng(seed)
    G = rng.standard_normal((n, n))
    return (G @ G.T / n + np.eye(n)).astype(dtype).astype(np.float64)


def _potrf(dm, A, uplo, dtype):
    n = A.shape[0]
    d, info = Dev(dm, A.astype(dtype)), dm.DeviceInt(1)
    fn = "dm_dpotrf" if dtype == np.float64 else "dm_spotrf"
    dm._lib.call(fn, uplo.encode(), n, d.p, max(n, 1), C.c_void_p(info.ptr), None)
    return d.get(), int(info.get()[0])


# factor error of a well-conditioned matrix: a few n eps, n <= 200
TOL = {np.float64: 2e-13, np.float32: 1e-4}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 56, 57, 63, 64, 65, 127, 128, 129, 200])
@pytest.mark.parametrize("scaling", ["none", "tiny", "huge", "mixed"])
def test_potrf_panel(dm, dtype, uplo, n, scaling):
    """D A D has the factor U D for a diagonal D of powers of two: with huge or
    tiny D the pivots leave the fast range, with a mixed one only some do.  The
    other triangle stays as it was."""
    A = _spd(n, dtype, n)
    e = {"none": 0, "tiny": -1, "huge": 1, "mixed": 1}[scaling] * (485 if dtype == np.float64 else 49)
    k = np.full(n, e)
    if scaling == "mixed":
        k = np.where(np.arange(n) % 11 == 3, e, np.where(np.arange(n) % 13 == 5, -e, 0))
    D = np.ldexp(1.0, k)
    got, info = _potrf(dm, A * D[:, None] * D[None, :], uplo, dtype)
    assert info == 0
    U = np.linalg.cholesky(A).T
    # undo the scaling (exact): U D -> U
    F = got.astype(np.float64)
    F = np.triu(F) / D[None, :] if uplo == "U" else (np.tril(F) / D[:, None]).T
    assert np.abs(F - U).max() <= TOL[dtype] * np.abs(U).max()
    other = np.tril(got, -1) if uplo == "U" else np.triu(got, 1)
    want = (A * D[:, None] * D[None, :]).astype(dtype)
    assert np.array_equal(other, np.tril(want, -1) if uplo == "U" else np.triu(want, 1))


@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n,bad", [(1, 0), (64, 0), (64, 63), (70, 66), (150, 64), (150, 100),
                                   (200, 199)])
@pytest.mark.parametrize("value", [0.0, -3.0, np.nan])
def test_potrf_failed_pivot(dm, uplo, n, bad, value):
    """info is the 1-based order of the first pivot that is not positive, and
    the rows of the factor before it are final."""
    A = np.diag(np.arange(1.0, n + 1))
    A[bad, bad] = value
    got, info = _potrf(dm, A, uplo, np.float64)
    assert info == bad + 1
    assert np.allclose(np.diag(got)[:bad], np.sqrt(np.arange(1.0, bad + 1)), rtol=1e-15, atol=0)


def _leading_factor(dm, uplo, n, bad):
    """potrf of a dense matrix whose pivot `bad` is negative: the factor of its
    leading bad x bad minor, and numpy's."""
    A = _spd(n, np.float64, n)
    A[bad, bad] = -1.0
    got, info = _potrf(dm, A, uplo, np.float64)
    assert info == bad + 1
    F = (np.triu(got) if uplo == "U" else np.tril(got).T)[:bad, :bad]
    return F, np.linalg.cholesky(A[:bad, :bad]).T


@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n,bad", [(200, 150), (200, 195), (330, 200), (330, 329)])
def test_potrf_failed_pivot_earlier_rows(dm, uplo, n, bad):
    """The panel before the last one that was factored is finished by the
    launch in which the pivot fails, whichever of its workgroups is first."""
    F, U = _leading_factor(dm, uplo, n, bad)
    rows = bad // 64 * 64 - 64
    assert np.abs(F - U)[:rows].max() <= TOL[np.float64] * np.abs(U).max()


@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n,bad", [(150, 40), (150, 64), (150, 100), (200, 128), (200, 150),
                                   (200, 199), (330, 256), (330, 300)])
def test_potrf_failed_pivot_leading_factor(dm, uplo, n, bad):
    """The factor of the leading minor before a failed pivot is whole, wherever
    in the second, third or last panel the pivot fails."""
    F, U = _leading_factor(dm, uplo, n, bad)
    assert np.abs(F - U).max() <= TOL[np.float64] * np.abs(U).max()


@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("dtype,n", [(np.float64, 2048), (np.float64, 2113), (np.float64, 2300),
                                     (np.float32, 3073), (np.float32, 3200)])
def test_potrf_large_tile(dm, dtype, n, uplo):
    """Around the size from which a panel's row, update and next diagonal block
    are launches of their own: the factor by its backward error (sqrt(n) u, see
    test_potrf_backward_error), the other triangle untouched."""
    A = _smooth(n, 1.0).astype(dtype)
    got, info = _potrf(dm, A, uplo, dtype)
    assert info == 0
    U = (np.triu(got) if uplo == "U" else np.tril(got).T).astype(np.float64)
    # FP64: the product that checks has an error of its own of as much
    rms = np.sqrt(np.mean((U.T @ U - A) ** 2))
    assert rms <= (2 if dtype == np.float64 else 1) * 2 * np.sqrt(n) * np.finfo(dtype).eps / 2
    other = np.tril(got, -1) if uplo == "U" else np.triu(got, 1)
    assert np.array_equal(other, np.tril(A, -1) if uplo == "U" else np.triu(A, 1))


@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("bad", [63, 64, 200, 320, 1000, 2299])
def test_potrf_failed_pivot_large_tile(dm, uplo, bad):
    """The leading factor before a failed pivot where panels have launches of
    their own, at the change to one launch (column 256) and after it."""
    F, U = _leading_factor(dm, uplo, 2300, bad)
    assert np.abs(F - U).max() <= 10 * TOL[np.float64] * np.abs(U).max()


def _smooth(n, nugget):
    """A covariance matrix of close points: exp(-(x - y)^2 / 0.02) and a nugget
    on the diagonal.  Its condition is about n / nugget, and most of that lies
    within any few neighbouring rows."""
    x = np.linspace(0.0, 1.0, n)
    return np.exp(-(x[:, None] - x) ** 2 / 0.02) + nugget * np.eye(n)


@pytest.mark.parametrize("dtype,nugget", [(np.float64, 1e-6), (np.float64, 1e-13),
                                          (np.float32, 1e-4)])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n", [65, 256, 300])
def test_potrf_backward_error(dm, dtype, nugget, uplo, n):
    """The error of U^T U - A does not grow with A's condition.  An element is
    a sum of at most n products with partial sums of at most 1, each rounded to
    u = eps / 2: a random walk of sqrt(n) u."""
    A = _smooth(n, nugget).astype(dtype)
    got, info = _potrf(dm, A, uplo, dtype)
    assert info == 0
    U = (np.triu(got) if uplo == "U" else np.tril(got).T).astype(np.longdouble)
    rms = np.sqrt(np.mean((U.T @ U - A) ** 2))
    assert rms <= np.sqrt(n) * np.finfo(dtype).eps / 2


def _trsm(dm, dtype, side, uplo, trans, diag, L, nv, alpha, pad):
    """One tile solve against its residual.  Substitution through inverted
    16 x 16 blocks is backward stable up to those blocks' condition (below 4
    here): |T X - alpha B| <= 4 (L + 16) eps |T| |X|."""
    rng = np.random.default_rng(1000 * L + nv)
    A = 0.5 * rng.standard_normal((L + pad, L)) / np.sqrt(L)
    A[np.arange(L), np.arange(L)] = 1.5 + rng.random(L)
    A = A.astype(dtype)
    m, n = (L, nv) if side == "L" else (nv, L)
    B = rng.standard_normal((m + pad, n)).astype(dtype)
    dA, dB = Dev(dm, A), Dev(dm, B)
    p = "d" if dtype == np.float64 else "s"
    a = C.c_double(alpha) if p == "d" else C.c_float(alpha)
    dm._lib.call(f"dm_{p}trsm", side.encode(), uplo.encode(), trans.encode(), diag.encode(), m, n,
                 a, dA.p, L + pad, dB.p, m + pad, None)
    got = dB.get()
    assert np.array_equal(got[m:], B[m:])
    T = A[:L].astype(np.float64)
    T = np.triu(T) if uplo == "U" else np.tril(T)
    if diag == "U":
        np.fill_diagonal(T, 1)
    op = T.T if trans == "T" else T
    X, R = got[:m].astype(np.float64), alpha * B[:m].astype(np.float64)
    if side == "R":
        op, X, R = op.T, X.T, R.T
    bound = 4 * (L + 16) * np.finfo(dtype).eps * (np.abs(op) @ np.abs(X))
    assert (np.abs(op @ X - R) <= bound).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("diag", ["N", "U"])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("side", ["L", "R"])
def test_trsm_leaf(dm, dtype, side, uplo, trans, diag):
    """Around the block rows of 16, the 256 rows a wave set covers once and the
    512 of a leaf; vectors around the 16 a workgroup takes; odd strides."""
    for L, nv, pad in [(1, 1, 0), (15, 3, 1), (16, 16, 0), (17, 17, 3), (33, 1, 0), (255, 31, 0),
                       (256, 1, 1), (257, 5, 0), (300, 16, 1), (496, 33, 0), (511, 2, 3),
                       (512, 48, 0), (513, 7, 0), (1041, 18, 1)]:
        _trsm(dm, dtype, side, uplo, trans, diag, L, nv, 0.75, pad)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("side,uplo,trans", [("L", "U", "T"), ("L", "L", "T"), ("R", "U", "T"),
                                             ("R", "L", "N")])
@pytest.mark.parametrize("L,nv", [(1, 131073), (16, 131103), (17, 65600), (130, 16389),
                                  (256, 16400)])
def test_trsm_many_vectors(dm, dtype, side, uplo, trans, L, nv):
    """Short triangles whose vectors take more than a round of the chip: a
    workgroup loops over several blocks of them, the last one over fewer."""
    _trsm(dm, dtype, side, uplo, trans, "N", L, nv, 0.5, 1)


@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("L", [1, 8, 40])
def test_trsm_zero_diagonal(dm, uplo, trans, L):
    """A zero in the first row that is solved makes that row infinite, with the
    right-hand side's sign, not NaN."""
    T = np.eye(L) * 2.0
    first = 0 if (uplo == "L") == (trans == "N") else L - 1
    T[first, first] = 0.0
    B = np.ones((L, 3))
    B[:, 1] = -1.0
    dA, dB = Dev(dm, T), Dev(dm, B)
    dm._lib.call("dm_dtrsm", b"L", uplo.encode(), trans.encode(), b"N", L, 3, 1.0, dA.p, L, dB.p, L,
                 None)
    assert np.array_equal(dB.get()[first], np.array([np.inf, -np.inf, np.inf]))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("trans", ["N", "T"])
@pytest.mark.parametrize("side", ["L", "R"])
@pytest.mark.parametrize("nv", [8191, 8192, 8193, 8223])
def test_trsm_wide(dm, dtype, side, trans, nv):
    """From 8192 vectors on a workgroup takes two blocks of 16, the last of
    them partly or wholly past the end."""
    for L in (16, 48, 290):
        _trsm(dm, dtype, side, "U", trans, "N", L, nv, -1.0, 1)


def _getf2(A, pivot):
    """Column by column, the operations of the panel in their order."""
    A, piv = A.astype(np.float64).copy(), []
    for k in range(min(A.shape)):
        p = k + int(np.argmax(np.abs(A[k:, k]))) if pivot else k
        piv.append(p + 1)
        A[[k, p]] = A[[p, k]]
        if A[k, k] != 0:
            A[k + 1:, k] /= A[k, k]
        A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
    return A, np.array(piv)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("pivot", [True, False])
@pytest.mark.parametrize("m,n", [(1, 1), (7, 7), (33, 32), (63, 40), (512, 9), (513, 33), (1024, 8),
                                 (1025, 31), (2048, 17), (2049, 32), (4096, 32), (4097, 7),
                                 (8193, 5), (16384, 3), (16385, 3), (20, 50)])
def test_lu_panel(dm, dtype, pivot, m, n):
    """One tile of m x n around the rows at which a leaf changes its kernel:
    the pivots exactly, ties (small integers) included, the factors within
    32 n eps of the growth that partial pivoting (or a dominant diagonal)
    bounds on these inputs."""
    rng = np.random.default_rng(m + n)
    A = rng.integers(-3, 4, (m, n)).astype(dtype) if n <= 9 else rng.standard_normal((m, n))
    A = (A if pivot else A + 4 * n * np.eye(m, n)).astype(dtype)
    if n <= 9:
        A[:, 1:] += rng.standard_normal((m, n - 1)).astype(dtype) / 4  # ties in the first column
    b = max(m, n)
    DA = dm.DArray.from_array(A, dm.Blocks(b, b))
    F = dm.lu_(DA, dm.RowMaximum() if pivot else dm.NoPivot(), check=False, allowsingular=True)
    want, piv = _getf2(A, pivot)
    assert np.array_equal(F.ipiv, piv)
    assert np.abs(DA.collect() - want).max() <= 32 * n * np.finfo(dtype).eps * np.abs(want).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m", [8192, 8193, 16384])
@pytest.mark.parametrize("n", [1, 2, 3, 4])
def test_lu_panel_narrow(dm, dtype, m, n):
    """Around the columns and rows at which a leaf goes from registers to
    memory: test_lu_panel's pivots and bound."""
    A = np.random.default_rng(m + n).standard_normal((m, n)).astype(dtype)
    DA = dm.DArray.from_array(A, dm.Blocks(m, m))
    F = dm.lu_(DA, dm.RowMaximum(), check=False)
    want, piv = _getf2(A, True)
    assert np.array_equal(F.ipiv, piv)
    assert np.abs(DA.collect() - want).max() <= 32 * n * np.finfo(dtype).eps * np.abs(want).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_lu_panel_values(dm, dtype):
    """Columns of zeros, NaN and infinities, pivots too small to invert."""
    rng = np.random.default_rng(3)
    A = rng.standard_normal((600, 12)).astype(dtype)
    A[:, 5] = 0
    DA = dm.DArray.from_array(A, dm.Blocks(600, 600))
    F = dm.lu_(DA, dm.RowMaximum(), check=False, allowsingular=True)
    want, piv = _getf2(A, True)
    assert F.info == 6 and np.array_equal(F.ipiv[:5], piv[:5]) and F.ipiv[5] == 6
    T = np.finfo(dtype)
    B = np.full((40, 1), T.smallest_subnormal * 4, dtype)  # 1 / pivot overflows
    B[17] = T.smallest_subnormal * 16
    DB = dm.DArray.from_array(B, dm.Blocks(40, 40))
    F = dm.lu_(DB, dm.RowMaximum(), check=False)
    assert F.ipiv[0] == 18 and np.array_equal(DB.collect()[1:, 0], np.full(39, 0.25, dtype))
    N = np.full((40, 1), np.nan, dtype)                    # no candidate: the row stays
    DN = dm.DArray.from_array(N, dm.Blocks(40, 40))
    assert dm.lu_(DN, dm.RowMaximum(), check=False, allowsingular=True).ipiv[0] == 1
    N[30], N[35] = -np.inf, np.inf                         # NaN never wins, the first tie does
    DN = dm.DArray.from_array(N, dm.Blocks(40, 40))
    assert dm.lu_(DN, dm.RowMaximum(), check=False, allowsingular=True).ipiv[0] == 31


@pytest.mark.parametrize("m,n,nb,steps", [(1, 1, 1, 1), (1300, 9, 100, 1300), (600, 5, 64, 37),
                                          (700, 3, 700, 512), (1025, 6, 256, 513)])
@pytest.mark.parametrize("kind", ["pivots", "one row", "any"])
def test_row_swaps(dm, m, n, nb, steps, kind):
    """The swaps in order, exactly: the rows a pivoted panel names, all steps
    naming one row, and lists with earlier rows and indices out of range."""
    rng = np.random.default_rng(m)
    B = rng.standard_normal((m, n))
    piv = np.array([rng.integers(p, m) for p in range(steps)]) + 1
    if kind == "one row":
        piv[:] = m
    elif kind == "any":
        piv = rng.integers(-3, m + 5, steps)
    D, ip = dm.DArray.from_array(B, dm.Blocks(nb, nb)), Dev(dm, piv.astype(np.int32))
    t = D.tiled()
    dm._lib.call("dm_tiled_laswp", C.byref(t), ip.p, steps, None)
    for p, q in enumerate(piv - 1):
        if 0 <= q < m:
            B[[p, q]] = B[[q, p]]
    assert np.array_equal(D.collect(), B)


@pytest.mark.parametrize("m,n,steps", [(3, 524288, 1), (9, 260000, 3), (40, 16385, 17), (300, 1030, 257)])
@pytest.mark.parametrize("kind", ["pivots", "any"])
def test_row_swaps_many_columns(dm, m, n, steps, kind):
    """Fewer steps than threads: sets of them on columns of their own."""
    rng = np.random.default_rng(n)
    B = rng.standard_normal((m, n))
    piv = np.array([rng.integers(p, m) for p in range(steps)]) + 1
    if kind == "any":
        piv = rng.integers(-3, m + 5, steps)
    D, ip = dm.DArray.from_array(B, dm.Blocks(n, n)), Dev(dm, piv.astype(np.int32))
    t = D.tiled()
    dm._lib.call("dm_tiled_laswp", C.byref(t), ip.p, steps, None)
    for p, q in enumerate(piv - 1):
        if 0 <= q < m:
            B[[p, q]] = B[[q, p]]
    assert np.array_equal(D.collect(), B)


def _crand(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -55, 2.0 ** 55])
def test_complex_potrf_leaf(dm, dtype, uplo, n, scale):
    """Blocks around the 16 x 16 threads and the leaf of 64; the scaled ones
    have FP32 pivots outside the range of the fast reciprocal root.  Factor
    error a few n eps of a well-conditioned matrix."""
    rng = np.random.default_rng(n)
    G = _crand(rng, n, n)
    A = (G @ G.conj().T / n + np.eye(n)).astype(dtype)
    U = np.linalg.cholesky(A.astype(complex)).conj().T * scale
    A = (A.astype(complex) * scale * scale).astype(dtype)
    d, info = Dev(dm, A), dm.DeviceInt(1)
    p = "z" if dtype == np.complex128 else "c"
    dm._lib.call(f"dm_{p}potrf", uplo.encode(), n, d.p, n, C.c_void_p(info.ptr), None)
    got = d.get()
    assert int(info.get()[0]) == 0
    F = np.triu(got) if uplo == "U" else np.tril(got).conj().T
    tol = 2e-13 if dtype == np.complex128 else 1e-4
    assert np.abs(F - U).max() <= tol * np.abs(U).max()
    assert not np.diag(got).imag.any()
    other = (lambda M: np.tril(M, -1)) if uplo == "U" else (lambda M: np.triu(M, 1))
    assert np.array_equal(other(got), other(A))


@pytest.mark.parametrize("dtype,nugget", [(np.complex128, 1e-6), (np.complex128, 1e-13),
                                          (np.complex64, 1e-4)])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n", [129, 256, 300])
def test_complex_potrf_backward_error(dm, dtype, nugget, uplo, n):
    """As the real test, with the rows turned in the complex plane: each part
    of an element is a sum of at most 2 n products, both parts sqrt(2) of that."""
    w = np.exp(2j * np.pi * np.random.default_rng(n).random(n))
    A = (w[:, None] * _smooth(n, nugget) * w.conj()).astype(dtype)
    A[np.arange(n), np.arange(n)] = A[np.arange(n), np.arange(n)].real
    d, info = Dev(dm, A), dm.DeviceInt(1)
    p = "z" if dtype == np.complex128 else "c"
    dm._lib.call(f"dm_{p}potrf", uplo.encode(), n, d.p, n, C.c_void_p(info.ptr), None)
    assert int(info.get()[0]) == 0
    got = d.get()
    U = (np.triu(got) if uplo == "U" else np.tril(got).conj().T).astype(np.clongdouble)
    E = np.triu(U.conj().T @ U - (A if uplo == "U" else A.conj().T))
    rms = np.sqrt(2 * np.mean(np.abs(E) ** 2))
    assert rms <= 2 * np.sqrt(n) * np.finfo(dtype).eps / 2


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("trans", ["N", "T", "C"])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("side", ["L", "R"])
def test_complex_trsm_leaf(dm, dtype, side, uplo, trans):
    """Around the block rows of 16 and the leaf of 256, by the residual:
    |T X - alpha B| <= 8 (L + 16) eps |T| |X|, as for the real kernel with the
    two products of each part."""
    eps = np.finfo(dtype).eps
    for L, nv, diag in [(1, 1, "N"), (15, 3, "U"), (16, 16, "N"), (17, 17, "N"), (64, 1, "U"),
                        (65, 33, "N"), (255, 2, "N"), (256, 31, "U"), (257, 16, "N"),
                        (530, 5, "N")]:
        rng = np.random.default_rng(L)
        A = (0.5 * _crand(rng, L + 1, L) / np.sqrt(2 * L)).astype(dtype)
        A[np.arange(L), np.arange(L)] = 1.5 + rng.random(L) + 0.5j * rng.random(L)
        m, n = (L, nv) if side == "L" else (nv, L)
        B = _crand(rng, m + 2, n).astype(dtype)
        dA, dB = Dev(dm, A), Dev(dm, B)
        p, R = ("z", np.float64) if dtype == np.complex128 else ("c", np.float32)
        alpha = np.array([0.75, -0.5], R)
        dm._lib.call(f"dm_{p}trsm", side.encode(), uplo.encode(), trans.encode(), diag.encode(),
                     m, n, alpha.ctypes.data_as(C.c_void_p), dA.p, L + 1, dB.p, m + 2, None)
        got = dB.get()
        assert np.array_equal(got[m:], B[m:])
        T = A[:L].astype(complex)
        T = np.triu(T) if uplo == "U" else np.tril(T)
        if diag == "U":
            np.fill_diagonal(T, 1)
        op = {"N": T, "T": T.T, "C": T.conj().T}[trans]
        X, rhs = got[:m].astype(complex), (0.75 - 0.5j) * B[:m].astype(complex)
        if side == "R":
            op, X, rhs = op.T, X.T, rhs.T
        bound = 8 * (L + 16) * eps * (np.abs(op) @ np.abs(X))
        assert (np.abs(op @ X - rhs) <= bound).all(), (L, nv, diag)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("side,uplo,trans", [("L", "U", "C"), ("L", "L", "T"), ("R", "U", "C"),
                                             ("R", "L", "N")])
@pytest.mark.parametrize("L,nv", [(1, 98305), (4, 98320), (6, 131), (16, 98303), (17, 49200),
                                  (32, 49153)])
def test_complex_trsm_many_vectors(dm, dtype, side, uplo, trans, L, nv):
    """Short triangles: a workgroup loops over its vectors once they take more
    than two rounds of the chip; the bound of test_complex_trsm_leaf."""
    rng = np.random.default_rng(L)
    A = (0.5 * _crand(rng, L, L) / np.sqrt(2 * L)).astype(dtype)
    A[np.arange(L), np.arange(L)] = 1.5 + rng.random(L) + 0.5j * rng.random(L)
    m, n = (L, nv) if side == "L" else (nv, L)
    B = _crand(rng, m + 1, n).astype(dtype)
    dA, dB = Dev(dm, A), Dev(dm, B)
    p, R = ("z", np.float64) if dtype == np.complex128 else ("c", np.float32)
    alpha = np.array([1.0, 0.5], R)
    dm._lib.call(f"dm_{p}trsm", side.encode(), uplo.encode(), trans.encode(), b"N", m, n,
                 alpha.ctypes.data_as(C.c_void_p), dA.p, L, dB.p, m + 1, None)
    got = dB.get()
    assert np.array_equal(got[m:], B[m:])
    T = (np.triu(A) if uplo == "U" else np.tril(A)).astype(complex)
    op = {"N": T, "T": T.T, "C": T.conj().T}[trans]
    X, rhs = got[:m].astype(complex), (1.0 + 0.5j) * B[:m].astype(complex)
    if side == "R":
        op, X, rhs = op.T, X.T, rhs.T
    bound = 8 * (L + 16) * np.finfo(dtype).eps * (np.abs(op) @ np.abs(X))
    assert (np.abs(op @ X - rhs) <= bound).all()


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("ta", ["N", "T", "C"])
@pytest.mark.parametrize("tb", ["N", "T", "C"])
def test_complex_gemm_tiles(dm, dtype, ta, tb):
    """Tiles of 32 and (from 256 of them on) of 64, remainders in every
    direction, by the product's bound 4 (k + 4) eps (|A| |B| + |C|)."""
    op = {"N": lambda M: M, "T": lambda M: M.T, "C": lambda M: M.conj().T}
    p, R = ("z", np.float64) if dtype == np.complex128 else ("c", np.float32)
    for m, n, k in [(1, 1, 1), (33, 31, 17), (64, 70, 0), (1024, 1024, 9), (1023, 1025, 8),
                    (960, 1024, 16)]:
        rng = np.random.default_rng(m + n)
        A = _crand(rng, *((m, k) if ta == "N" else (k, m))).astype(dtype)
        B = _crand(rng, *((k, n) if tb == "N" else (n, k))).astype(dtype)
        Cm = _crand(rng, m, n).astype(dtype)
        dA, dB, dC = Dev(dm, A), Dev(dm, B), Dev(dm, Cm)
        al, be = np.array([0.75, -0.5], R), np.array([0.5, 0.25], R)
        dm._lib.call(f"dm_{p}gemm", ta.encode(), tb.encode(), m, n, k,
                     al.ctypes.data_as(C.c_void_p), dA.p, max(A.shape[0], 1), dB.p,
                     max(B.shape[0], 1), be.ctypes.data_as(C.c_void_p), dC.p, m, None)
        a, b, c = op[ta](A.astype(complex)), op[tb](B.astype(complex)), Cm.astype(complex)
        ref = (0.75 - 0.5j) * (a @ b) + (0.5 + 0.25j) * c
        bound = 4 * (k + 4) * np.finfo(dtype).eps * (np.abs(a) @ np.abs(b) + np.abs(c))
        assert (np.abs(dC.get() - ref) <= bound).all(), (m, n, k)


@pytest.mark.parametrize("inc", [1, 3])
def test_gemv_n(dm, inc):
    """Around the 32 rows of a workgroup and the 256 columns of one round of
    loads, by the product's bound 4 (n + 4) eps (|A| |x| + |y|)."""
    for m, n in [(1, 1), (31, 5), (32, 255), (33, 256), (70, 257), (512, 600), (64, 0)]:
        rng = np.random.default_rng(m + n)
        A = rng.standard_normal((m, max(n, 1)))
        x, y = rng.standard_normal(max(n, 1) * inc), rng.standard_normal(m * inc)
        dA, dx, dy = Dev(dm, A), Dev(dm, x), Dev(dm, y)
        dm._lib.call("dm_dgemv", b"N", m, n, 0.5, dA.p, m, dx.p, inc, -2.0, dy.p, inc, None)
        got, a, v, w = dy.get(), A[:, :n], x[::inc][:n], y[::inc]
        bound = 4 * (n + 4) * np.finfo(float).eps * (np.abs(a) @ np.abs(v) + 2 * np.abs(w))
        assert (np.abs(got[::inc] - (0.5 * (a @ v) - 2.0 * w)) <= bound).all(), (m, n)
        rest = np.arange(len(y)) % inc != 0
        assert np.array_equal(got[rest], y[rest])


@pytest.mark.parametrize("m", [33, 65535, 65536, 65537])
@pytest.mark.parametrize("n", [0, 1, 8, 9, 16, 17, 128, 129, 300])
def test_gemv_n_groups(dm, m, n):
    """Around the columns and rows at which a workgroup's shape changes, by the
    product's bound 4 (n + 4) eps (|A| |x| + |y|)."""
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, max(n, 1)))
    x, y = rng.standard_normal(max(n, 1)), rng.standard_normal(m)
    dA, dx, dy = Dev(dm, A), Dev(dm, x), Dev(dm, y)
    dm._lib.call("dm_dgemv", b"N", m, n, 0.5, dA.p, m, dx.p, 1, -2.0, dy.p, 1, None)
    a, v = A[:, :n], x[:n]
    bound = 4 * (n + 4) * np.finfo(float).eps * (np.abs(a) @ np.abs(v) + 2 * np.abs(y))
    assert (np.abs(dy.get() - (0.5 * (a @ v) - 2.0 * y)) <= bound).all()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n,nb", [(1, 1), (15, 15), (16, 16), (17, 17), (63, 63), (64, 64), (65, 65),
                                  (200, 130), (129, 64)])
def test_inverted_tiles(dm, dtype, uplo, n, nb):
    """ldiv! through the inverted diagonal tiles around their leaf of 64 and its
    blocks of 16; the matrix has condition about 5, the error bound is 64 n eps."""
    A, rng = _spd(n, dtype, n), np.random.default_rng(n)
    b = rng.standard_normal((n, 3)).astype(dtype)
    DA = dm.DArray.from_array(A.astype(dtype), dm.Blocks(nb, nb))
    DB = dm.DArray.from_array(b, dm.Blocks(nb, 3))
    dm.ldiv_(dm.cholesky_(DA, uplo), DB)
    want = np.linalg.solve(A, b.astype(np.float64))
    assert np.abs(DB.collect() - want).max() <= 64 * n * np.finfo(dtype).eps * np.abs(want).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,k", [(1793, 1800, 17), (1920, 1792, 16), (127, 129, 40), (65, 1, 3)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_gemm_ragged_tiles(dm, dtype, m, n, k, beta):
    """Whole and ragged tiles of 128 and 64 (beta = 0 reads no C), by the
    product's bound 4 (k + 4) eps (|A| |B| + |C|); rows past C stay."""
    rng = np.random.default_rng(m + n)
    A, B = rng.standard_normal((k, m)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
    Cm = rng.standard_normal((m + 1, n)).astype(dtype)
    if beta == 0.0:
        Cm[:m] = np.nan
    dA, dB, dC = Dev(dm, A), Dev(dm, B), Dev(dm, Cm)
    p, real = ("d", C.c_double) if dtype == np.float64 else ("s", C.c_float)
    dm._lib.call(f"dm_{p}gemm", b"T", b"N", m, n, k, real(-1.5), dA.p, k, dB.p, k, real(beta), dC.p,
                 m + 1, None)
    got, a, b = dC.get(), A.astype(np.float64), B.astype(np.float64)
    c = np.nan_to_num(Cm[:m].astype(np.float64)) * beta
    bound = 4 * (k + 4) * np.finfo(dtype).eps * (1.5 * np.abs(a.T) @ np.abs(b) + np.abs(c))
    assert (np.abs(got[:m] - (c - 1.5 * (a.T @ b))) <= bound).all()
    assert np.array_equal(got[m], Cm[m])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("uplo", ["U", "L"])
@pytest.mark.parametrize("n", [1, 129, 2433])
def test_syrk_diagonal_tiles(dm, dtype, uplo, n):
    """Tiles on the diagonal store their triangle and leave the other alone."""
    rng, k = np.random.default_rng(n), 19
    A, Cm = rng.standard_normal((k, n)).astype(dtype), rng.standard_normal((n, n)).astype(dtype)
    dA, dC = Dev(dm, A), Dev(dm, Cm)
    p, real = ("d", C.c_double) if dtype == np.float64 else ("s", C.c_float)
    dm._lib.call(f"dm_{p}syrk", uplo.encode(), b"T", n, k, real(-1.0), dA.p, k, real(1.0), dC.p, n,
                 None)
    got, a = dC.get(), A.astype(np.float64)
    tri = np.triu if uplo == "U" else np.tril
    bound = 4 * (k + 4) * np.finfo(dtype).eps * (np.abs(a.T) @ np.abs(a) + np.abs(Cm))
    assert (np.abs(tri(got - (Cm - a.T @ a))) <= bound).all()
    assert np.array_equal(got - tri(got), Cm - tri(Cm))
