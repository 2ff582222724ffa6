"""GPU tests of the one-workgroup leaf kernels at the edges of their ranges:
the Cholesky leaf (64 x 64, four register stages of 16 rows) and the inverted
diagonal blocks of the look-back solves (64 rows FP64, 128 rows FP32, four
stages)."""
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
