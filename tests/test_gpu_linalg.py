"""GPU parity: FP64 LU (the library's blocked getrf and substitution, rocBLAS
updates) and decoupling through the C ABI.

Reference: decouple_covmat (src/covariance.jl:8-14) and `\\`
(src/blockspectralmatrix.jl:101-129).
"""
import numpy as np
import pytest
from helpers import mask_like_W, rel_err

pytestmark = pytest.mark.gpu


def test_decouple_reference_kat(ctx):
    """test/test_covmat.jl:11-17 of the reference, matrices inline there."""
    A = np.array([[1.0, 0.2, 0.3], [0.4, 2.0, 0.15], [0.3, 0.1, 1.44]])
    B1 = np.array([[1.2, 0.6, 0.1], [0.3, 1.4, 0.5], [0.44, 0.2, 1.3]])
    B2 = np.array([[1.6, 0.4, 0.1], [0.3, 1.4, 0.9], [0.45, 0.8, 1.7]])
    Cref = np.linalg.inv(B1) @ A @ np.linalg.inv(B2).T
    C = ctx.decouple_covmat(A, B1, B2)
    assert np.allclose(C, Cref, rtol=1.5e-8, atol=0)
    assert rel_err(C, Cref) < 1e-13


def test_decouple_matches_oracle_and_numpy(ctx, oracle):
    rng = np.random.default_rng(2)
    n = 400
    Y = rng.standard_normal((n, n))
    Y = Y @ Y.T
    B1 = np.eye(n) + 0.1 * rng.standard_normal((n, n))
    B2 = np.eye(n) + 0.1 * rng.standard_normal((n, n))
    C = ctx.decouple_covmat(Y, B1, B2)
    R = oracle.decouple_covmat(Y, B1, B2)
    N = np.linalg.solve(B1, Y) @ np.linalg.inv(B2).T
    assert np.linalg.norm(C - R) / np.linalg.norm(R) < 1e-11
    assert np.linalg.norm(C - N) / np.linalg.norm(N) < 1e-11


def test_decouple_invariant_with_gpu_mcm(ctx):
    """test/test_covmat.jl:115-127: C_coupled = M C_dec M^T for a TT MCM M."""
    lmax = 300
    M = ctx.mcm(0, 0, lmax, mask_like_W(lmax + 1, seed=9))
    rng = np.random.default_rng(0)
    X = rng.uniform(size=M.shape)
    Cc = X.T @ X
    Cd = ctx.decouple_covmat(Cc, M, M)
    back = M @ Cd @ M.T
    assert np.linalg.norm(back - Cc) / np.linalg.norm(Cc) < 1e-9


def test_lu_solve(ctx, oracle):
    rng = np.random.default_rng(5)
    n = 513
    A = np.eye(n) * 3 + rng.standard_normal((n, n))
    b = rng.standard_normal(n)
    x = ctx.lu_solve(A, b)
    assert np.linalg.norm(A @ x - b) / np.linalg.norm(b) < 1e-12
    B = rng.standard_normal((n, 3))
    X = ctx.lu_solve(A, B)
    R = oracle.lu_solve(A, B)
    assert np.linalg.norm(X - R) / np.linalg.norm(R) < 1e-11


def test_singular(ctx, pkg):
    A = np.ones((4, 4))
    with pytest.raises(pkg.SingularException):
        ctx.lu_solve(A, np.ones(4))
    with pytest.raises(pkg.SingularException):
        ctx.decouple_covmat(np.eye(4), np.zeros((4, 4)), np.eye(4))
    with pytest.raises(pkg.AxisError):
        ctx.lu_solve(np.eye(4), np.ones(3))


@pytest.mark.parametrize("n", [1, 5, 16, 17, 32, 33, 256, 257, 289, 300, 513, 1000, 1025, 2100,
                               3072, 3100, 4100])
def test_lu_factor_vs_lapack(ctx, n):
    """The blocked getrf (leaf kernels + rocBLAS updates) against LAPACK's
    getrf (scipy): the same row interchanges and factors to rounding.  Up to
    3072 leaf rows one workgroup factors a 16-column leaf in registers; above
    that each column is a launch over many workgroups (n = 3100 and 4100 run
    both, switching when the remaining rows drop to 3072)."""
    import scipy.linalg as sl
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    LU, ipiv = ctx.lu_factor(A)
    lu_ref, piv_ref = sl.lu_factor(A)
    assert np.array_equal(ipiv - 1, piv_ref)
    assert np.linalg.norm(LU - lu_ref) / np.linalg.norm(lu_ref) < 1e-12


def test_lu_factor_mcm_and_solve(ctx):
    """A TT mode-coupling matrix at lmax 1500 (no row interchanges expected
    beyond LAPACK's): factors as LAPACK, and `M \\ b` through psx_lu_solve."""
    import scipy.linalg as sl
    lmax = 1500
    M = ctx.mcm(0, 0, lmax, mask_like_W(lmax + 1, seed=3))
    LU, ipiv = ctx.lu_factor(M)
    lu_ref, piv_ref = sl.lu_factor(M)
    assert np.array_equal(ipiv - 1, piv_ref)
    assert np.linalg.norm(LU - lu_ref) / np.linalg.norm(lu_ref) < 1e-12
    b = M @ (1.0 / (np.arange(lmax + 1) + 1.0) ** 2)
    x = ctx.lu_solve(M, b)
    assert np.linalg.norm(x - sl.lu_solve((lu_ref, piv_ref), b)) / np.linalg.norm(x) < 1e-12


def test_lu_factor_singular(ctx, pkg):
    with pytest.raises(pkg.SingularException):
        ctx.lu_factor(np.ones((40, 40)))


@pytest.mark.parametrize("n,k", [(2100, 2000), (3100, 5), (4100, 3500), (4100, 700)])
def test_lu_factor_zero_column_position(ctx, pkg, n, k):
    """An exactly zero column k stays zero through every update, so the first
    zero pivot is column k + 1 (LAPACK's info): found by the one-workgroup
    leaf (n = 2100), by the per-column leaf (n = 3100, k = 5), and by each of
    them after the other has run (n = 4100).  The solve refuses it too."""
    rng = np.random.default_rng(n + k)
    A = rng.standard_normal((n, n))
    A[:, k] = 0.0
    with pytest.raises(pkg.SingularException, match=rf"position {k + 1} "):
        ctx.lu_factor(A)
    with pytest.raises(pkg.SingularException, match=rf"position {k + 1} "):
        ctx.lu_solve(A, np.ones(n))


def test_lu_factor_structured_pivots(ctx):
    """Pivoting that moves rows across leaves and blocks: a matrix whose
    largest entry of every column sits in the bottom rows (LAPACK swaps it up
    at every step), against scipy."""
    import scipy.linalg as sl
    n = 600
    rng = np.random.default_rng(1)
    A = rng.uniform(0.0, 1.0, (n, n))
    A[n - 64:, :] += 10.0 * np.arange(1, 65)[:, None]
    LU, ipiv = ctx.lu_factor(A)
    lu_ref, piv_ref = sl.lu_factor(A)
    assert np.array_equal(ipiv - 1, piv_ref)
    assert np.linalg.norm(LU - lu_ref) / np.linalg.norm(lu_ref) < 1e-12


def test_lu_solve_device_buffers(ctx):
    """psx_lu_solve_d on device buffers equals psx_lu_solve on host buffers."""
    rng = np.random.default_rng(4)
    n = 700
    A = np.asfortranarray(np.eye(n) * 2 + rng.standard_normal((n, n)))
    b = rng.standard_normal(n)
    want = ctx.lu_solve(A, b)
    dA, dB = ctx.alloc(8 * n * n), ctx.alloc(8 * n)
    try:
        ctx.h2d(dA, A.ravel(order="F"))
        ctx.h2d(dB, b)
        ctx.check(ctx.lib.psx_lu_solve_d(ctx.handle, n, dA, n, dB, n, 1), "lu_solve_d")
        got = np.empty(n)
        ctx.d2h(got, dB)
    finally:
        ctx.free(dA)
        ctx.free(dB)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 320, 511, 777, 2100])
def test_lu_solve_substitution_sizes(ctx, n):
    """Solves with 1-4 right-hand sides run the library's forward and back
    substitution (128-row diagonal blocks, one launch per block); 5 run its
    many-right-hand-side triangular solve (64-row diagonal blocks, rocBLAS
    updates).  Both against LAPACK (scipy lu_solve)."""
    import scipy.linalg as sl
    rng = np.random.default_rng(100 + n)
    A = rng.standard_normal((n, n)) + np.diag(rng.uniform(1.0, 2.0, n)) * np.sqrt(n)
    ref_lu = sl.lu_factor(A)
    for nrhs in (1, 2, 4, 5):
        B = rng.standard_normal((n, nrhs))
        X = ctx.lu_solve(A, B)
        R = sl.lu_solve(ref_lu, B)
        assert np.linalg.norm(X - R) / np.linalg.norm(R) < 1e-12, (n, nrhs)


def test_lu_solve_substitution_padded_lda(ctx):
    """psx_lu_solve_d with lda and ldb larger than n, and pivoting across
    blocks.  The matrix has cond ~ 6e6 (numpy and scipy solves differ by
    5e-12), so the check is the normwise backward error
    |A x - b| / (|A| |x| + |b|), which a stable LU solve keeps near machine
    epsilon whatever the conditioning, and the forward error against scipy
    within cond x 1e-15."""
    import scipy.linalg as sl
    n, lda, ldb = 600, 613, 640
    rng = np.random.default_rng(8)
    A = rng.uniform(0.0, 1.0, (n, n))
    A[n - 64:, :] += 10.0 * np.arange(1, 65)[:, None]
    b = rng.standard_normal((n, 2))
    Ap = np.zeros((lda, n), order="F")
    Ap[:n] = A
    bp = np.full((ldb, 2), 7.0, order="F")
    bp[:n] = b
    dA, dB = ctx.alloc(8 * lda * n), ctx.alloc(8 * ldb * 2)
    try:
        ctx.h2d(dA, Ap)
        ctx.h2d(dB, bp)
        ctx.check(ctx.lib.psx_lu_solve_d(ctx.handle, n, dA, lda, dB, ldb, 2), "lu_solve_d")
        got = np.empty((ldb, 2), order="F")
        ctx.d2h(got, dB)
    finally:
        ctx.free(dA)
        ctx.free(dB)
    x = got[:n]
    eta = np.linalg.norm(A @ x - b) / (np.linalg.norm(A, 2) * np.linalg.norm(x)
                                        + np.linalg.norm(b))
    assert eta < 1e-15
    R = sl.lu_solve(sl.lu_factor(A), b)
    assert np.linalg.norm(x - R) / np.linalg.norm(R) < np.linalg.cond(A) * 1e-15
    assert (got[n:] == 7.0).all()


def _ill_conditioned(n, cond, seed):
    """Q1 diag(logspace(0, -log10 cond)) Q2 + a small identity part: cond(A) ~ cond."""
    rng = np.random.default_rng(seed)
    q1, _ = np.linalg.qr(rng.standard_normal((n, n)))
    q2, _ = np.linalg.qr(rng.standard_normal((n, n)))
    return (q1 * np.logspace(0.0, -np.log10(cond), n)) @ q2


@pytest.mark.parametrize("n,nrhs", [(300, 37), (700, 700)])
def test_lu_solve_many_rhs_backward_error(ctx, n, nrhs):
    """More than 4 right-hand sides run the blocked substitution (diagonal blocks
    solved by substitution, rocBLAS GEMM updates).  On cond ~ 1e10 the normwise
    backward error stays within 10x of numpy's LAPACK solve (~1e-16)."""
    A = _ill_conditioned(n, 1e10, n)
    B = np.random.default_rng(1).standard_normal((n, nrhs))
    X = ctx.lu_solve(A, B)
    R = np.linalg.solve(A, B)
    eta = lambda Z: np.linalg.norm(A @ Z - B) / (np.linalg.norm(A, 2) * np.linalg.norm(Z)
                                                 + np.linalg.norm(B))
    assert eta(X) < 10 * eta(R) + 1e-16, (eta(X), eta(R))
    assert np.linalg.norm(X - R) / np.linalg.norm(R) < 1e10 * 1e-14


def test_decouple_ill_conditioned(ctx):
    """decouple_covmat(Y, B, B) with cond(B) ~ 1e8: B D B^T reproduces Y within
    10x of numpy's two LAPACK solves.  (On the TT mode-coupling matrix of the
    lmax-2508 covariance workload, cond 2.4e8, rocSOLVER's getrs, whose trsm
    inverts diagonal blocks, reproduced Y to 1.4e-7 against numpy's 2.6e-9;
    the substitution gives 2-4e-9.)"""
    n = 600
    Bm = _ill_conditioned(n, 1e8, 3)
    X = np.random.default_rng(2).standard_normal((n, n))
    Y = X @ X.T / n
    D = ctx.decouple_covmat(Y, Bm, Bm)
    R = np.linalg.solve(Bm, np.linalg.solve(Bm, Y).T).T
    rec = lambda Z: np.linalg.norm(Bm @ Z @ Bm.T - Y) / np.linalg.norm(Y)
    assert rec(D) < 10 * rec(R) + 1e-15, (rec(D), rec(R))
    assert np.linalg.norm(D - R) / np.linalg.norm(R) < 1e8 * 1e-14


def test_decouple_shared_matrix_factored_once(ctx):
    """decouple_covmat(Y, M, M) with one array on both sides factors it once;
    the result equals the call with an equal copy as B2 bit for bit."""
    lmax = 400
    M = ctx.mcm(0, 0, lmax, mask_like_W(lmax + 1, seed=12))
    X = np.random.default_rng(6).standard_normal(M.shape)
    Y = np.asfortranarray(X @ X.T)
    same = ctx.decouple_covmat(Y, M, M)
    apart = ctx.decouple_covmat(Y, M, np.array(M, order="F", copy=True))
    assert np.array_equal(same, apart)
    assert np.linalg.norm(M @ same @ M.T - Y) / np.linalg.norm(Y) < 1e-11


@pytest.mark.parametrize("n,nrhs", [(1, 1), (300, 1), (300, 3), (1700, 2)])
def test_lu_solve_pm(ctx, pkg, n, nrhs):
    """psx_lu_solve_pm: [M++ s M--; s M-- M++] X = B with the 2n x 2n matrix
    assembled on the device equals psx_lu_solve on the matrix assembled on the
    host, bit for bit for s = +1, and for s = -1, where it solves the s = +1
    matrix against D B (D = diag(I, -I)) exactly; both against numpy."""
    rng = np.random.default_rng(n + nrhs)
    Mpp = np.eye(n) * 2.0 + rng.standard_normal((n, n)) / np.sqrt(n)
    Mmm = 0.3 * rng.standard_normal((n, n)) / np.sqrt(n)
    B = rng.standard_normal((2 * n, nrhs))
    for sign in (1, -1):
        A = np.block([[Mpp, sign * Mmm], [sign * Mmm, Mpp]])
        X = ctx.lu_solve_pm(Mpp, Mmm, B, sign)
        assert np.array_equal(X, ctx.lu_solve(A, B)), sign
        R = np.linalg.solve(A, B)
        assert np.linalg.norm(X - R) / np.linalg.norm(R) < 1e-12, sign
    x = ctx.lu_solve_pm(Mpp, Mmm, B[:, 0], -1)
    assert x.shape == (2 * n,) and np.array_equal(x, ctx.lu_solve_pm(Mpp, Mmm, B[:, :1], -1)[:, 0])


def test_lu_solve_pm_arguments(ctx, pkg):
    """A sign other than +-1, blocks of different sizes, a right-hand side of
    the wrong length, and M++ = M-- (a singular block matrix) are refused."""
    A = np.eye(4)
    with pytest.raises(pkg.ArgumentError):
        ctx.lu_solve_pm(A, A, np.ones(8), 0)
    with pytest.raises(pkg.AxisError):
        ctx.lu_solve_pm(A, np.eye(3), np.ones(8))
    with pytest.raises(pkg.AxisError):
        ctx.lu_solve_pm(A, A, np.ones(7))
    with pytest.raises(pkg.SingularException):
        ctx.lu_solve_pm(A, A, np.ones(8), 1)


def _permuted(A, ipiv):
    p = np.arange(A.shape[0])
    for i, q in enumerate(np.asarray(ipiv) - 1):
        p[i], p[q] = p[q], p[i]
    return A[p]


# either side of every change of the leaf kernel (512 rows a register row, 32,
# 16 and 8 columns a leaf, the multi-workgroup path above 6144 rows) and of the
# 256-column panel
@pytest.mark.parametrize("n", [8, 9, 255, 256, 257, 511, 512, 513, 1024, 1025, 1536, 1537, 2049,
                               2561, 3072, 3073, 4097, 5121, 6144, 6177])
def test_lu_factor_at_leaf_edges(ctx, n):
    A = np.random.default_rng(n).uniform(-1, 1, (n, n))
    LU, ipiv = ctx.lu_factor(A)
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    assert np.abs(L).max() <= 1.0
    # |P A - L U| <= gamma_n |L| |U| for any order of the updates, and as much
    # again for the product formed here
    err = np.abs(_permuted(A, ipiv) - L @ U)
    bound = 2 * n * np.finfo(float).eps * (np.abs(L) @ np.abs(U))
    assert (err <= bound).all()


@pytest.mark.parametrize("n", [40, 300, 1600])
def test_lu_pivot_ties_zero_columns_and_nan(ctx, n):
    # every |entry| alike: ties go to the row that came first in the matrix
    # the leaf started from (the first 8 columns are one leaf); exact arithmetic
    from fractions import Fraction
    A = np.where(np.random.default_rng(n).uniform(size=(n, n)) < 0.5, -1.0, 1.0)
    _, ipiv = ctx.lu_factor(A)
    M = [[Fraction(int(v)) for v in row[:8]] for row in A]
    at, free = list(range(n)), set(range(n))     # row at each position
    for j in range(7):       # (magnitudes 1, 2, 3, 4: exact in doubles too)
        top = max(abs(M[i][j]) for i in free)
        p = min(i for i in free if abs(M[i][j]) == top)
        assert ipiv[j] - 1 == at.index(p)
        q = at.index(p)
        at[j], at[q] = at[q], at[j]
        free.remove(p)
        for i in free:
            f = M[i][j] / M[p][j]
            M[i] = [a - f * b for a, b in zip(M[i], M[p])]
        if any(v.denominator & (v.denominator - 1) for i in free for v in M[i]):
            break            # entries no longer doubles
    # a zero column is reported where LAPACK reports it
    B = np.random.default_rng(n + 1).uniform(-1, 1, (n, n))
    B[:, n // 2] = 0.0
    with pytest.raises(Exception, match=f"position {n // 2 + 1}"):
        ctx.lu_solve(B, np.ones(n))
    # a NaN is the pivot of its column and reaches the solution
    B = np.random.default_rng(n + 2).uniform(-1, 1, (n, n))
    B[n - 3, 0] = np.nan
    LU, ipiv = ctx.lu_factor(B)
    assert ipiv[0] == n - 2
    assert np.isnan(ctx.lu_solve(B, np.ones(n))).all()
    # pivots whose reciprocals leave the normal range
    S = np.random.default_rng(n + 3).uniform(-1, 1, (n, n)) * 2.0 ** -1010
    x = ctx.lu_solve(S, S @ np.ones(n))
    ref = np.linalg.solve(S * 2.0 ** 1010, (S * 2.0 ** 1010) @ np.ones(n))
    cond = np.linalg.cond(S * 2.0 ** 1010)
    assert np.abs(x - 1).max() <= 1e3 * np.abs(ref - 1).max() + cond * 1e-13


@pytest.mark.parametrize("n,m", [(1, 5), (15, 7), (16, 16), (17, 33), (63, 5), (64, 15), (65, 17),
                                 (240, 16), (255, 31), (256, 5), (257, 18), (511, 6), (513, 65)])
def test_solve_many_right_hand_sides_at_block_edges(ctx, n, m):
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (n, n))
    B = rng.uniform(-1, 1, (n, m))
    X = ctx.lu_solve(A, B)
    LU, ipiv = ctx.lu_factor(A)
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    # backward error of substitution with computed factors: |A X - B| <=
    # 3 gamma_n |P^T L| |U| |X| (Higham, theorem 9.4); doubled for the product here
    R = np.abs(_permuted(A @ X - B, ipiv))
    assert (R <= 6 * n * np.finfo(float).eps * (np.abs(L) @ (np.abs(U) @ np.abs(X)))).all()
    if n > 1 and m == n:
        Y = rng.uniform(-1, 1, (n, n))
        assert np.array_equal(ctx.decouple_covmat(Y, A, A), ctx.decouple_covmat(Y, A, A.copy()))


@pytest.mark.parametrize("n,nrhs", [(5, 1), (40, 1), (300, 4), (700, 6), (6200, 2)])
def test_lu_solve_d_leaves_the_right_hand_sides_of_a_singular_system(ctx, pkg, n, nrhs):
    # a zero pivot is found before the right-hand sides change; padded leading
    # dimensions, and sizes on either side of every row movement
    rng = np.random.default_rng(n)
    lda, ldb = n + 3, n + 5
    A = np.zeros((lda, n), order="F")
    A[:n] = rng.uniform(-1, 1, (n, n))
    A[:n, n // 2] = 0.0
    B = np.asfortranarray(rng.uniform(-1, 1, (ldb, nrhs)))
    dA, dB = ctx.alloc(A.nbytes), ctx.alloc(B.nbytes)
    try:
        ctx.h2d(dA, A)
        ctx.h2d(dB, B)
        with pytest.raises(pkg.SingularException, match=f"position {n // 2 + 1} "):
            ctx.check(ctx.lib.psx_lu_solve_d(ctx.handle, n, dA, lda, dB, ldb, nrhs), "lu_solve_d")
        got = np.empty_like(B)
        ctx.d2h(got, dB)
        assert np.array_equal(got, B)
    finally:
        ctx.free(dA)
        ctx.free(dB)
