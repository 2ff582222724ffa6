"""GPU tests of the one-workgroup leaf kernels at the edges of their ranges:
the Cholesky leaf (64 x 64, four register stages of 16 rows)."""
import numpy as np
import pytest
import torch

import slate_amd
from helpers import say, spd, to_dev, to_host

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
