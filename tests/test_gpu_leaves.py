"""GPU tests of the leaf kernels at the edges of their ranges:
the Cholesky leaf (64 x 64, four register stages of 16 rows) and the inverted
diagonal blocks of the look-back solves (64 rows FP64, 128 rows FP32, four
stages), and the LU panel leaf (one workgroup up to 512 rows, an exchange of up
to 128 above)."""
import math

import numpy as np
import pytest
import torch

import oracle
import slate_amd
from helpers import dev_rands, say, spd, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 33, 48, 49, 63, 64, 127])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_potrf_leaf_sizes(gpu, n, dtype):
    """A = L L^T to the backward error of a Cholesky factorization, (n + 1) eps
    of the product |L| |L|^T entry by entry (Higham, Accuracy and Stability,
    theorem 10.3, gamma_{n+1}), and the other triangle untouched."""
    say("potrf leaf n=%d %s" % (n, dtype))
    S = spd(70 + n, n)
    A = to_dev(S, dtype)
    S = to_host(A)
    assert slate_amd.potrf(A, opts=slate_amd.Options(block_size=64)) == 0
    R = to_host(A)
    L = np.tril(R)
    eps = float(torch.finfo(dtype).eps)
    assert (np.abs(S - L @ L.T) <= (n + 1) * eps * (np.abs(L) @ np.abs(L.T)) + 1e-300).all()
    np.testing.assert_array_equal(np.triu(R, 1), np.triu(S, 1))


@pytest.mark.parametrize("bad", [0, 15, 16, 31, 47, 63])
def test_potrf_leaf_info(gpu, bad):
    say("potrf leaf n=64 bad pivot %d" % bad)
    S = spd(8, 64)
    S[bad, bad] = -1.0
    A = to_dev(S)
    assert slate_amd.potrf(A, opts=slate_amd.Options(block_size=64)) == bad + 1


@pytest.mark.parametrize("n", [1, 2, 16, 63, 64, 65, 127, 128, 129, 200, 257])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_getrs_vector_block_edges(gpu, n, trans, dtype):
    """One right-hand side at the edges of the look-back blocks: backward error
    against the factors used.  Each block solve multiplies by a computed
    inverse, so the bound is not the substitution's n eps but carries the
    condition of a diagonal block; the factors here (unit lower part with
    entries below 0.5 / n, diagonal of U in [1, 2]) keep every block's
    condition below 8, which gives 8 * 2 n eps."""
    say("getrs vector n=%d trans=%s %s" % (n, trans, dtype))
    F = 0.5 * oracle.rands(90 + n, n, n) / max(n, 1)
    F[np.arange(n), np.arange(n)] = 1.5 + 0.5 * oracle.rands(91, n, 1)[:, 0]
    A = to_dev(F, dtype)
    F = to_host(A)
    L = np.tril(F, -1) + np.eye(n)
    U = np.triu(F)
    ipiv = np.arange(1, n + 1)
    ipiv[0] = n
    B = dev_rands(92, n, 1, dtype)
    b = to_host(B)[:, 0]
    slate_amd.getrs(A, ipiv, B, trans=trans)
    x = to_host(B)[:, 0]
    perm = np.arange(n)
    perm[0], perm[n - 1] = perm[n - 1], perm[0]
    r = b - U.T @ (L.T @ x[perm]) if trans else b[perm] - L @ (U @ x)
    scale = np.abs(L).sum(1).max() * np.abs(U).sum(1).max() * np.abs(x).max()
    assert np.abs(r).max() <= 16 * max(n, 2) * float(torch.finfo(dtype).eps) * scale


@pytest.mark.parametrize("n", [3, 33, 64, 65, 255, 256, 257, 511, 513, 1023, 1025, 2047, 2049])
def test_panel_leaf_row_edges(gpu, n):
    """Leaf shapes by rows: the trailing panels of one factorization run
    through every shape below n.  Pivots equal the oracle's, factors within the
    accumulated rounding of both (the bound of the other getrf tests)."""
    say("panel leaf n=%d" % n)
    A = dev_rands(300 + n, n, n)
    info, ipiv = slate_amd.getrf(A, slate_amd.Options(block_size=128))
    LU_o, ipiv_o, info_o = oracle.getrf(oracle.rands(300 + n, n, n), nb=128, ib=16)
    assert info == info_o == 0
    np.testing.assert_array_equal(ipiv, ipiv_o)
    assert np.abs(to_host(A) - LU_o).max() <= 4 * max(n, 16) * np.finfo(np.float64).eps * np.abs(LU_o).max()


@pytest.mark.parametrize("ib", [5, 16, 32])
@pytest.mark.parametrize("ld", [300, 301])
def test_panel_leaf_widths(gpu, ib, ld):
    """Leaves narrower than the register form, aligned and unaligned rows."""
    say("panel leaf ib=%d ld=%d" % (ib, ld))
    n = 300
    A = slate_amd.empty_colmajor(n, n, torch.float64, ld=ld)
    A.copy_(dev_rands(12, n, n))
    info, ipiv = slate_amd.getrf(A, slate_amd.Options(block_size=64, inner_blocking=ib))
    LU_o, ipiv_o, _ = oracle.getrf(oracle.rands(12, n, n), nb=64, ib=16)
    assert info == 0
    np.testing.assert_array_equal(ipiv, ipiv_o)
    assert np.abs(to_host(A) - LU_o).max() <= 4 * n * np.finfo(np.float64).eps * np.abs(LU_o).max()


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("n", [40, 700])
def test_panel_leaf_non_finite(gpu, value, n):
    """A non-finite entry in column 20 leaves the columns before it, their
    pivots and their rows' U entries as they are without it."""
    say("panel leaf n=%d with %r" % (n, value))
    H = oracle.rands(55, n, n)
    A = to_dev(H)
    slate_amd.getrf(A)
    H2 = H.copy()
    H2[n - 3, 20] = value
    B = to_dev(H2)
    _, piv = slate_amd.getrf(B)
    LU_o, piv_o, _ = oracle.getrf(H2, nb=n, ib=32)
    np.testing.assert_array_equal(piv[:20], piv_o[:20])
    # columns 0 .. 19: U part and multipliers as a set (the interchanges of
    # later columns move the rows of L, and those depend on the bad value)
    a, b = to_host(A)[:, :20], to_host(B)[:, :20]
    np.testing.assert_array_equal(a[:20], b[:20])
    np.testing.assert_array_equal(np.sort(a[20:], axis=0), np.sort(b[20:], axis=0))


@pytest.mark.parametrize("n,dtype", [(520, torch.float64), (8321, torch.float64), (28801, torch.float64),
                                     (8321, torch.float32), (28801, torch.float32)])
def test_panel_leaf_exchange_shapes(gpu, n, dtype):
    """Leaf shapes of several workgroups: every panel of the factorization is
    pivoted strictly (|L| <= 1) and P A = L U within n eps |L| |U| for the
    factorization and as much for the product that checks it."""
    say("panel leaf exchange n=%d %s" % (n, dtype))
    g = torch.Generator("cuda").manual_seed(n)
    A = torch.empty(n, n, dtype=dtype, device="cuda").uniform_(-1, 1, generator=g).t()
    F = A.t().clone().t()
    info, ipiv = slate_amd.getrf(F)
    assert info == 0
    perm = np.arange(n)
    for i, p in enumerate(ipiv):
        perm[i], perm[p - 1] = perm[p - 1], perm[i]
    rows = torch.from_numpy(np.r_[0:200, n // 2:n // 2 + 100, n - 200:n]).cuda()
    L = torch.where(rows[:, None] > torch.arange(n, device="cuda")[None, :], F[rows], 0)
    assert float(L.abs().max()) <= 1.0
    L[torch.arange(len(rows), device="cuda"), rows] = 1.0
    U = F.triu()
    PA = A[torch.from_numpy(perm).cuda()[rows]]
    bound = 2 * n * torch.finfo(dtype).eps * (L.abs() @ U.abs())
    assert bool(((PA - L @ U).abs() <= bound).all())


@pytest.mark.parametrize("n", [512, 1024, 2048])
def test_panel_leaf_ties(gpu, n):
    """A Hadamard matrix is eliminated exactly in powers of two and every
    pivot search is a tie: the first of equals wins, across waves and
    workgroups, and the factors are the oracle's bit by bit."""
    say("panel leaf ties n=%d" % n)
    H = np.array([[1.0]])
    while H.shape[0] < n:
        H = np.block([[H, H], [H, -H]])
    H = np.asfortranarray(H[np.random.default_rng(n).permutation(n)])
    A = to_dev(H)
    info, ipiv = slate_amd.getrf(A)
    LU_o, ipiv_o, info_o = oracle.getrf(H, nb=128, ib=16)
    assert info == info_o == 0
    np.testing.assert_array_equal(ipiv, ipiv_o)
    np.testing.assert_array_equal(to_host(A), LU_o)


@pytest.mark.parametrize("n", [300, 700, 1500])
def test_panel_leaf_threshold(gpu, n):
    """A pivot threshold keeps diagonals; the oracle's pivots, and its factors
    within the accumulated rounding (growth is in max |LU|)."""
    say("panel leaf threshold n=%d" % n)
    A = dev_rands(77, n, n)
    info, ipiv = slate_amd.getrf(A, slate_amd.Options(pivot_threshold=0.5, block_size=128))
    LU_o, ipiv_o, _ = oracle.getrf(oracle.rands(77, n, n), nb=128, ib=16, threshold=0.5)
    assert info == 0
    np.testing.assert_array_equal(ipiv[:64], ipiv_o[:64])
    a, b = to_host(A)[:, :64], LU_o[:, :64]
    if np.array_equal(ipiv, ipiv_o):
        assert np.abs(a - b).max() <= 4 * n * np.finfo(np.float64).eps * np.abs(LU_o).max()


def test_panel_leaf_zero_column(gpu):
    """No candidate but zeros in a column of several workgroups: the diagonal
    stays and info names the column."""
    say("panel leaf zero column")
    n = 1500
    H = oracle.rands(91, n, n).copy(order="F")
    H[:, 40] = 0.0
    A = to_dev(H)
    info, ipiv = slate_amd.getrf(A)
    assert info == 41 and ipiv[40] == 41


# 32 x 64 tiles (few tiles), 64 x 64 and 128 x 128 tiles, each with whole
# tiles, ragged edges, a k tail, and operands one element off 16-byte alignment
@pytest.mark.parametrize("m,n,k", [(70, 130, 200), (64, 128, 128), (1100, 1000, 70), (1088, 1024, 64),
                                   (2100, 2050, 33), (2048, 2176, 48)])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_gemm_tiles(gpu, m, n, k, off, dtype):
    """|computed - exact| <= (k + 2) eps (|A| |B| + |C|), entry by entry."""
    say("gemm tiles %dx%dx%d off=%d %s" % (m, n, k, off, dtype))
    g = torch.Generator("cuda").manual_seed(m + n + k)

    def mat(r, c):
        S = torch.empty(c, r + 3, dtype=dtype, device="cuda").uniform_(-1, 1, generator=g).t()
        return S[off:off + r]

    A, B, C = mat(m, k), mat(k, n), mat(m, n)
    a, b, c0 = A.double(), B.double(), C.double().clone()
    slate_amd.gemm(-1.0, A, B, 0.5, C)
    ref = 0.5 * c0 - a @ b
    bound = (k + 2) * float(torch.finfo(dtype).eps) * (a.abs() @ b.abs() + 0.5 * c0.abs())
    assert bool(((C.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("n", [33, 64, 257, 300, 700])
@pytest.mark.parametrize("nrhs", [2, 5, 9])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_getrs_matrix_edges(gpu, n, nrhs, trans, dtype):
    """Several right-hand sides: column by column up to four, blocked beyond;
    both triangles in both views.  Same factors and bound as the vector test."""
    say("getrs n=%d nrhs=%d trans=%s %s" % (n, nrhs, trans, dtype))
    F = 0.5 * oracle.rands(90 + n, n, n) / n
    F[np.arange(n), np.arange(n)] = 1.5 + 0.5 * oracle.rands(91, n, 1)[:, 0]
    A = to_dev(F, dtype)
    F = to_host(A)
    L = np.tril(F, -1) + np.eye(n)
    U = np.triu(F)
    ipiv = np.arange(1, n + 1)
    ipiv[0] = n
    B = dev_rands(92, n, nrhs, dtype)
    b = to_host(B)
    slate_amd.getrs(A, ipiv, B, trans=trans)
    x = to_host(B)
    perm = np.arange(n)
    perm[0], perm[n - 1] = perm[n - 1], perm[0]
    r = b - U.T @ (L.T @ x[perm]) if trans else b[perm] - L @ (U @ x)
    scale = np.abs(L).sum(1).max() * np.abs(U).sum(1).max() * np.abs(x).max()
    assert np.abs(r).max() <= 16 * n * float(torch.finfo(dtype).eps) * scale


@pytest.mark.parametrize("n", [40, 300, 1000])
@pytest.mark.parametrize("nrhs", [4, 6])
@pytest.mark.parametrize("uplo", [slate_amd.LOWER, slate_amd.UPPER])
def test_posv_matrix_edges(gpu, n, nrhs, uplo):
    say("posv n=%d nrhs=%d uplo=%d" % (n, nrhs, uplo))
    S = spd(4, n)
    A = to_dev(S)
    B = dev_rands(5, n, nrhs)
    b = to_host(B)
    assert slate_amd.posv(A, B, uplo=uplo) == 0
    x = to_host(B)
    scale = np.abs(S).sum(1).max() * np.abs(x).max()
    assert np.abs(b - S @ x).max() <= 16 * n * np.finfo(np.float64).eps * scale


def test_getrs_matrix_extreme_diagonal(gpu):
    """Diagonal entries whose reciprocal overflows take the dividing branch of
    the one-launch solve; rows next to them keep full accuracy."""
    n, nrhs = 64, 8
    F = np.eye(n)
    F[5, 5] = 1e-310
    F[40, 40] = 1e300
    A = to_dev(F)
    b = np.ones((n, nrhs))
    b[5] = 3e-310
    B = to_dev(b)
    slate_amd.getrs(A, np.arange(1, n + 1), B)
    ref = b / np.diag(F)[:, None]
    np.testing.assert_allclose(to_host(B), ref, rtol=4 * np.finfo(np.float64).eps, atol=0)


def _batch(ns, seed, singular=()):
    rng = np.random.default_rng(seed)
    mats, rhs = [], []
    for i, n in enumerate(ns):
        M = rng.uniform(-1, 1, (n, n)) + 1.2 * np.sqrt(n) * np.eye(n)[rng.permutation(n)]
        if i in singular:
            M[:, n // 2] = 0.0
        mats.append(M)
        rhs.append(rng.uniform(-1, 1, n))
    A = torch.from_numpy(np.concatenate([m.T.ravel() for m in mats])).cuda()
    B = torch.from_numpy(np.concatenate(rhs)).cuda()
    return mats, rhs, A, B, torch.zeros_like(B)


@pytest.mark.parametrize("ns", [[1] * 5, list(range(1, 66)), [64, 65, 63, 1024, 48, 47, 33, 500],
                                [(7 * i) % 24 + 1 for i in range(2300)], [96, 97, 127, 128, 129, 160]])
@pytest.mark.parametrize("prec", [slate_amd.PREC_FP32, slate_amd.PREC_FP64])
def test_batched_wave_and_workgroup_sizes(gpu, ns, prec):
    """Systems that one wave solves (up to 64 rows), alone, in full groups and
    beside workgroup systems.  Solutions against numpy's to 1e-11 relative:
    the condition numbers stay below about 1e4, and the backward errors below
    the refinement's tolerance, sqrt(n) eps."""
    say("batched %d systems up to %d, precision %d" % (len(ns), max(ns), prec))
    mats, rhs, A, B, X = _batch(ns, 5)
    iters, info, berr = slate_amd.gesv_batched(ns, A, B, X, prec)
    assert (info == 0).all() and (iters >= 0).all()
    assert (berr <= np.sqrt(np.asarray(ns)) * np.finfo(np.float64).eps * (1 if prec == slate_amd.PREC_FP32 else 32)).all()
    x = X.cpu().numpy()
    o = 0
    for M, b, n in zip(mats, rhs, ns):
        ref = np.linalg.solve(M, b)
        np.testing.assert_allclose(x[o:o + n], ref, rtol=0, atol=1e-11 * np.abs(ref).max())
        o += n


def test_batched_singular_small_and_large(gpu):
    """A zero column: info names it after the FP64 fallback, iters = -3, and
    the other systems are solved."""
    ns = [20, 64, 3, 100, 50]
    bad = (0, 1, 3)
    mats, rhs, A, B, X = _batch(ns, 6, bad)
    iters, info, _ = slate_amd.gesv_batched(ns, A, B, X, slate_amd.PREC_FP32)
    x = X.cpu().numpy()
    o = 0
    for i, (M, b, n) in enumerate(zip(mats, rhs, ns)):
        if i in bad:
            assert info[i] == n // 2 + 1 and iters[i] == -3
        else:
            assert info[i] == 0 and iters[i] >= 0
            np.testing.assert_allclose(x[o:o + n], np.linalg.solve(M, b), rtol=0, atol=1e-11)
        o += n


def test_batched_no_iterations(gpu):
    """max_iterations 0 and -1: only a first solve that already meets the
    tolerance counts, and none does with -1."""
    ns = [30, 200]
    mats, rhs, A, B, X = _batch(ns, 7)
    for most, want in ((0, -1), (-1, 0)):
        iters, info, _ = slate_amd.gesv_batched(ns, A, B, X, slate_amd.PREC_FP32,
                                                opts=slate_amd.Options(max_iterations=most))
        assert (info == 0).all() and (iters == want).all()


def _kernel_matrix(n, shift):
    """A Gaussian kernel on n points plus a small diagonal: symmetric positive
    definite, its diagonal blocks as ill conditioned as the whole."""
    t = np.sort(np.random.default_rng(n).uniform(0, 1, n))
    return np.exp(-((t[:, None] - t[None, :]) / 0.3) ** 2) + shift * np.eye(n)


@pytest.mark.parametrize("n", [96, 256, 700])
@pytest.mark.parametrize("nrhs", [2, 3, 4, 5])
@pytest.mark.parametrize("kind", ["lu", "lu_t", "lu_float", "lower", "upper"])
def test_few_right_hand_sides_backward_error(gpu, n, nrhs, kind):
    """Solves of several right-hand sides substitute: the residual against the
    computed factors stays below gamma_n for each triangle, entry by entry
    (Higham, Accuracy and Stability, theorem 8.5), with no condition number.
    |b - L U x| <= 2 n eps |L| |U| |x| holds both and the checking product."""
    say("right-hand sides n=%d nrhs=%d %s" % (n, nrhs, kind))
    dtype = torch.float32 if kind == "lu_float" else torch.float64
    A = to_dev(_kernel_matrix(n, 1e-4 if kind == "lu_float" else 1e-10), dtype)
    B = dev_rands(17, n, nrhs, dtype)
    b = to_host(B)
    if kind.startswith("lu"):
        info, ipiv = slate_amd.getrf(A)
        slate_amd.getrs(A, ipiv, B, trans=kind == "lu_t")
        F = to_host(A)
        L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
        perm = np.arange(n)
        for i, p in enumerate(ipiv):
            perm[i], perm[p - 1] = perm[p - 1], perm[i]
    else:
        uplo = slate_amd.LOWER if kind == "lower" else slate_amd.UPPER
        info = slate_amd.potrf(A, uplo=uplo)
        slate_amd.potrs(A, B, uplo=uplo)
        F = to_host(A)
        L = np.tril(F) if kind == "lower" else np.triu(F).T
        U, perm = L.T, np.arange(n)
    assert info == 0
    x = to_host(B)
    if kind == "lu_t":
        r, bound = b - U.T @ (L.T @ x[perm]), np.abs(U.T) @ (np.abs(L.T) @ np.abs(x[perm]))
    else:
        r, bound = b[perm] - L @ (U @ x), np.abs(L) @ (np.abs(U) @ np.abs(x))
    assert (np.abs(r) <= 2 * n * float(torch.finfo(dtype).eps) * bound).all()


@pytest.mark.parametrize("prec", [slate_amd.PREC_FP32, slate_amd.PREC_BF16])
def test_batched_float_overflow_falls_back(gpu, prec):
    """Entries above float's range make the float factor infinite or NaN: its
    norms are not finite, so it does not count as converged, and the FP64
    factor solves the system, on the one-wave and the workgroup path.  Scaling
    a system by a number leaves its relative errors as they are, so the bound
    is the one of the other batched tests."""
    ns = [2, 40, 64, 65, 100, 300]
    mats, rhs, A, B, X = _batch(ns, 8)
    A *= 1e40
    say("batched overflow, precision %d" % prec)
    iters, info, berr = slate_amd.gesv_batched(ns, A, B, X, prec)
    assert (info == 0).all() and (iters < 0).all()
    assert (berr <= 32 * np.sqrt(np.asarray(ns)) * np.finfo(np.float64).eps).all()
    x = X.cpu().numpy()
    o = 0
    for M, b, n in zip(mats, rhs, ns):
        ref = np.linalg.solve(M, b)
        np.testing.assert_allclose(1e40 * x[o:o + n], ref, rtol=0, atol=1e-11 * np.abs(ref).max())
        o += n


@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_batched_non_finite_is_reported(gpu, value):
    """A non-finite entry in the matrix or the right-hand side never counts as
    solved: no step count, and a backward error that is not finite."""
    ns = [40, 40, 40, 100, 100, 100]
    say("batched with %r" % value)
    mats, rhs, A, B, X = _batch(ns, 9)
    A[7] = value                       # systems 0 and 3: in the matrix
    A[3 * 1600 + 7] = value
    B[40 + 3] = value                  # systems 1 and 4: in the right-hand side
    B[120 + 100 + 3] = value
    iters, info, berr = slate_amd.gesv_batched(ns, A, B, X, slate_amd.PREC_FP32)
    bad = np.array([True, True, False, True, True, False])
    np.testing.assert_array_equal(iters < 0, bad)
    np.testing.assert_array_equal(~np.isfinite(berr), bad)


# numerators and quotients near both ends of the range, subnormal ones among
# them, where a product with the reciprocal and one correction would lose bits
_EXTREME = {np.float64: [1e-290, 1e-300, 5e-308, 1e-310, 3e-320, 1e306, 1.0, 0.0],
            np.float32: [1e-30, 1e-36, 3e-38, 1e-40, 3e-44, 1e37, 1.0, 0.0]}


def _extreme_quotients(n, T, seed):
    rng = np.random.default_rng(seed)
    d = rng.uniform(1, 16, n).astype(T)
    b = np.stack([(rng.uniform(1, 2, n) * s).astype(T) for s in _EXTREME[T]], axis=1)
    return d, b, b / d[:, None]


@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("trans", [False, True])
def test_getrs_extreme_numerators(gpu, T, trans):
    """A diagonal factor: every entry is one division, correctly rounded (the
    other terms of the substitution are exact zeros)."""
    say("getrs extreme numerators %s trans=%s" % (T.__name__, trans))
    n = 70
    dtype = torch.float64 if T is np.float64 else torch.float32
    d, b, ref = _extreme_quotients(n, T, 3)
    B = slate_amd.colmajor(torch.from_numpy(np.asfortranarray(b)).to(dtype).cuda())
    slate_amd.getrs(slate_amd.colmajor(torch.from_numpy(np.diag(d)).cuda()), np.arange(1, n + 1), B, trans=trans)
    np.testing.assert_array_equal(B.cpu().numpy(), ref)


def test_batched_extreme_numerators(gpu):
    """The same for the FP64 solves of the batch, one wave and a workgroup."""
    say("batched extreme numerators")
    ns, mats, rhs, refs = [], [], [], []
    for n in (33, 64, 100):
        d, b, ref = _extreme_quotients(n, np.float64, n)
        for j in range(b.shape[1]):
            ns.append(n)
            mats.append(np.diag(d).ravel())
            rhs.append(b[:, j])
            refs.append(ref[:, j])
    X = torch.zeros(sum(ns), dtype=torch.float64, device="cuda")
    slate_amd.gesv_batched(ns, torch.from_numpy(np.concatenate(mats)).cuda(), torch.from_numpy(np.concatenate(rhs)).cuda(),
                           X, slate_amd.PREC_FP64)
    np.testing.assert_array_equal(X.cpu().numpy(), np.concatenate(refs))


def _lu_error(A, F, ipiv, rows=None):
    """(|L| below the diagonal by column, whether |P A - L U| <= 2 n eps |L| |U|
    on the rows): n eps for the factorization, as much for the product here.
    A: the matrix, F: its factors, on the device."""
    n = A.shape[0]
    perm = np.arange(n)
    for i, p in enumerate(ipiv):
        perm[i], perm[p - 1] = perm[p - 1], perm[i]
    rows = torch.arange(n, device="cuda") if rows is None else torch.from_numpy(rows).cuda()
    L = torch.where(rows[:, None] > torch.arange(n, device="cuda")[None, :], F[rows], 0)
    most = L.abs().amax(0)
    L[torch.arange(len(rows), device="cuda"), rows] = 1.0
    U = F.triu()
    r = A[torch.from_numpy(perm).cuda()[rows]] - L @ U
    return most, bool((r.abs() <= 2 * n * torch.finfo(F.dtype).eps * (L.abs() @ U.abs())).all())


@pytest.mark.parametrize("n,ld", [(700, 700), (700, 701), (1500, 1504)])
@pytest.mark.parametrize("ib", [5, 16, 20, 32])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_panel_leaf_exchange_widths(gpu, n, ld, ib, dtype):
    """Leaves across workgroups in both register forms (16 and 32 columns) and
    narrower than them, rows aligned and not: pivoted strictly, the oracle's
    pivots in FP64, P A = L U."""
    say("panel leaf exchange n=%d ld=%d ib=%d %s" % (n, ld, ib, dtype))
    A = dev_rands(12, n, n, dtype)
    F = slate_amd.empty_colmajor(n, n, dtype, ld=ld)
    F.copy_(A)
    info, ipiv = slate_amd.getrf(F, slate_amd.Options(block_size=128, inner_blocking=ib))
    assert info == 0
    most, close = _lu_error(A, F, ipiv)
    assert float(most.max()) <= 1.0 and close
    if dtype == torch.float64:
        np.testing.assert_array_equal(ipiv, oracle.getrf(oracle.rands(12, n, n), nb=128, ib=16)[1])


@pytest.mark.parametrize("n,ib", [(33001, 0), (57400, 32)])
def test_panel_leaf_tall(gpu, n, ib):
    """FP64 panels above 32768 rows, where leaves of 16 columns keep two rows
    per thread, and above 57344 rows with 32 columns and two rows per thread:
    pivoted strictly, P A = L U on rows from the top, the middle and the end."""
    say("panel leaf n=%d ib=%d" % (n, ib))
    g = torch.Generator("cuda").manual_seed(n)
    A = torch.empty(n, n, dtype=torch.float64, device="cuda").uniform_(-1, 1, generator=g).t()
    F = A.t().clone().t()
    info, ipiv = slate_amd.getrf(F, slate_amd.Options(inner_blocking=ib))
    assert info == 0
    most, close = _lu_error(A, F, ipiv, np.r_[0:100, n // 2:n // 2 + 50, n - 100:n])
    assert float(most.max()) <= 1.0 and close


@pytest.mark.parametrize("n", [300, 700, 1500])
def test_panel_leaf_threshold_factors(gpu, n):
    """With a threshold of 0.5 a column whose diagonal was kept has |L| <= 2 up
    to the rounding of the scaling, one that was interchanged |L| <= 1 (both
    kinds occur), and P A = L U with the pivots taken, whatever they are."""
    say("panel leaf threshold factors n=%d" % n)
    A = dev_rands(77, n, n)
    F = A.t().clone().t()
    info, ipiv = slate_amd.getrf(F, slate_amd.Options(pivot_threshold=0.5, block_size=128))
    assert info == 0
    most, close = _lu_error(A, F, ipiv)
    kept = torch.from_numpy(ipiv == np.arange(1, n + 1)).cuda()
    assert 0 < int(kept.sum()) < n
    assert float(most[kept].max()) <= 2 * (1 + 4 * np.finfo(np.float64).eps)
    assert float(most[~kept].max()) <= 1.0 and close


@pytest.mark.parametrize("cfg", [(16, 256), (32, 256), (16, 512)])
@pytest.mark.parametrize("prec", [slate_amd.PREC_FP32, slate_amd.PREC_FP64])
def test_batched_update_order(gpu, cfg, prec):
    """The trailing update sums its products in the order of k.  Here the first
    two cancel, 2^23 - 2^23 (2^52 in FP64), before products of 1/4 arrive, so
    the factor is exact in that order and in others loses the small ones; an
    exact factor solves the system without a refinement step, bit for bit."""
    say("batched update order %s precision %d" % (cfg, prec))
    n, big = 80, 2.0 ** (23 if prec == slate_amd.PREC_FP32 else 52)
    M = np.eye(n)
    M[0, 32:], M[1, 32:], M[4, 32:], M[8, 32:] = big, -big, 0.25, 0.25
    M[32:, [0, 1, 4, 8]] = 1.0
    M[32:, 32:] = 0.5 + 4.0 * np.eye(n - 32)
    x = np.r_[np.arange(1.0, 33.0), np.tile([1.0, -1.0], (n - 32) // 2)]
    A = torch.from_numpy(M.T.ravel().copy()).cuda()
    B = torch.tensor([math.fsum(row * x) for row in M], dtype=torch.float64, device="cuda")
    X = torch.zeros_like(B)
    saved = slate_amd.tune_get_batched()[:3]
    try:
        slate_amd.tune_set_batched(*cfg, 1)
        iters, info, _ = slate_amd.gesv_batched([n], A, B, X, prec)
    finally:
        slate_amd.tune_set_batched(*saved)
    assert info[0] == 0 and iters[0] == 0
    np.testing.assert_array_equal(X.cpu().numpy(), x)
