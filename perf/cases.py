"""Performance cases of the factor-and-solve library.

Each case is one call that a user's program makes, through the public entry
points of ``slate_amd``: plain LU and Cholesky solves in FP64, solves with
factors kept from an earlier call, the mixed-precision drivers with their
refinement, and batches of small uneven systems.  ``listed`` gives the fixed
cases, ``draw`` more of the same ranges, ``prepare`` the inputs on the GPU,
``run`` one call, ``work`` the bytes and flops the call cannot do without, and
``exact`` the results in 64 bits from plain torch.

Right-hand sides are made from a chosen solution (b = A x), so the exact
solution is known for every size to within the rounding of b.
"""
import math

import numpy as np
import torch

import slate_amd as S

# factorization precisions of the mixed drivers, by name
PRECISIONS = {"fp32": S.PREC_FP32, "bf16x2": S.PREC_BF16X2, "bf16x3": S.PREC_BF16X3}
# above this size a 64-bit factorization by torch takes too long to serve as a reference
FACTOR_MAX = 10000


def listed():
    return [
        # a small dense system inside a larger program (a local solve, a
        # coupling block): all launches and latency
        {"name": "gesv_100", "op": "gesv", "n": 100, "nrhs": 1, "kind": "rands"},
        # the size of the reference configuration of SLATE's CPU path
        {"name": "gesv_2000", "op": "gesv", "n": 2000, "nrhs": 1, "kind": "rands"},
        # an ordinary dense solve with a block of right-hand sides
        {"name": "gesv_8192_64", "op": "gesv", "n": 8192, "nrhs": 64, "kind": "rands"},
        # the full-size FP64 solve
        {"name": "gesv_32768", "op": "gesv", "n": 32768, "nrhs": 1, "kind": "svd", "cond": 1e4},
        # factored once, then one transposed solve per call (adjoint systems);
        # an odd size
        {"name": "getrs_t_10001", "op": "getrs", "n": 10001, "nrhs": 1, "trans": True},
        # a small SPD system given by its upper triangle (a normal-equation or
        # covariance matrix); a ragged size
        {"name": "posv_1500_upper", "op": "posv", "n": 1500, "nrhs": 3, "upper": True},
        # the full-size Cholesky factorization
        {"name": "potrf_32768", "op": "potrf", "n": 32768, "upper": False},
        # SLATE's own mixed solver: float factor, classic refinement; an odd size
        {"name": "mixed_fp32_6001", "op": "mixed", "n": 6001, "precision": "fp32", "gmres": False, "cond": 1e3},
        # the headline size: float factor with split-BF16 updates, GMRES refinement
        {"name": "mixed_gmres_65536", "op": "mixed", "n": 65536, "precision": "bf16x2", "gmres": True, "cond": 1e2},
        # the SPD mixed solver with float-accurate split-BF16 updates
        {"name": "posv_mixed_16384", "op": "posv_mixed", "n": 16384, "precision": "bf16x3", "gmres": False,
         "cond": 1e3},
        # a few hundred tiny systems (element or cell matrices)
        {"name": "batch_300_tiny", "op": "batched", "count": 300, "lo": 8, "hi": 64},
        # the batched workload: 4096 systems, half general, half SPD
        {"name": "batch_4096", "op": "batched", "count": 4096, "lo": 32, "hi": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gesv", "gesv", "getrs", "posv", "potrf", "mixed", "mixed", "posv_mixed", "batched"])
    if op == "gesv":
        n = _log_int(rng, 32, 32768)
        return {"op": op, "n": n, "nrhs": rng.choice([1, 1, 1, rng.randint(2, 64)]),
                "kind": "rands" if n <= 8192 else "svd", "cond": 1e4}
    if op == "getrs":
        return {"op": op, "n": _log_int(rng, 100, 16384), "nrhs": rng.choice([1, 1, rng.randint(2, 64)]),
                "trans": rng.random() < 0.5}
    if op == "posv":
        return {"op": op, "n": _log_int(rng, 32, 32768), "nrhs": rng.choice([1, rng.randint(2, 64)]),
                "upper": rng.random() < 0.5}
    if op == "potrf":
        return {"op": op, "n": _log_int(rng, 32, 32768), "upper": rng.random() < 0.5}
    if op in ("mixed", "posv_mixed"):
        n = _log_int(rng, 500, 40000)
        return {"op": op, "n": n, "precision": rng.choice(sorted(PRECISIONS)), "gmres": rng.random() < 0.5,
                "cond": 1e3 if n <= 16384 else 1e2}
    lo = _log_int(rng, 4, 64)
    hi = _log_int(rng, 64, 1024)
    # the sizes' third powers bounded by those of the full batch
    most = min(4096, int(4096 * (1024 / hi) ** 2))
    return {"op": op, "count": _log_int(rng, 50, most), "lo": lo, "hi": hi}


# ---- inputs -----------------------------------------------------------------
def _uniform(g, *shape):
    return torch.empty(*shape, dtype=torch.float64, device="cuda").uniform_(-1.0, 1.0, generator=g)


def _mixer(n, rng):
    """A sparse recipe for an n x n orthogonal matrix: three rounds of a random
    signed permutation followed by one orthogonal block on every group of (up
    to) 64 rows."""
    b = min(64, n)
    W = torch.from_numpy(np.linalg.qr(rng.standard_normal((b, b)))[0]).cuda()
    rounds = []
    for _ in range(3):
        p = torch.from_numpy(rng.permutation(n)).cuda()
        s = torch.from_numpy(rng.choice([-1.0, 1.0], n)).cuda()
        rounds.append((p, s))
    return b, W, rounds


def _mix_rows(Q, M):
    """Q M for the recipe Q."""
    b, W, rounds = Q
    n = M.shape[0]
    full = n // b * b
    for p, s in rounds:
        M = M[p]
        M *= s[:, None]
        out = torch.matmul(W, M[:full].view(full // b, b, -1)).view(full, -1)
        if full < n:
            out = torch.cat([out, M[full:]])
        M = out
    return M


def _mix_cols(Q, M):
    """M Q^T for the recipe Q."""
    b, W, rounds = Q
    m, n = M.shape
    full = n // b * b
    for p, s in rounds:
        M = M[:, p]
        M *= s[None, :]
        M[:, :full] = torch.matmul(M[:, :full].reshape(m * (full // b), b), W.t()).view(m, full)
    return M


def _spectrum(n, cond, seed, sym):
    """Column-major U diag(s) V^T (V = U when sym), s geometric from 1 to 1/cond."""
    rng = np.random.default_rng(seed)
    d = torch.from_numpy(cond ** (-np.arange(n) / max(n - 1, 1))).cuda()
    U = _mixer(n, rng)
    V = U if sym else _mixer(n, rng)
    M = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    M.diagonal().copy_(d)
    M = _mix_rows(U, M)
    M = _mix_cols(V, M)
    if sym:
        # exactly symmetric, in blocks of rows to bound the memory
        for i in range(0, n, 8192):
            j = min(n, i + 8192)
            up = 0.5 * (M[i:j, i:] + M[i:, i:j].t())
            M[i:j, i:] = up
            M[i:, i:j] = up.t()
    return M.t()


def _shifted(n, g):
    """SPD: a symmetric uniform matrix over sqrt(n), shifted past its spectrum
    (|eigenvalues| < 0.83); condition number about 10."""
    A = _uniform(g, n, n)
    for i in range(0, n, 8192):                        # blocks of rows bound the memory
        j = min(n, i + 8192)
        up = (0.5 / math.sqrt(n)) * (A[i:j, i:] + A[i:, i:j].t())
        A[i:j, i:] = up
        A[i:, i:j] = up.t()
    A.diagonal().add_(1.0)
    return A.t()


def _times(A, X):
    """A X by torch, column-major."""
    return torch.matmul(X.t(), A.t()).t() if X.dim() == 2 else torch.mv(A, X)


def _solution(n, nrhs, g):
    return _uniform(g, n) if nrhs == 1 else _uniform(g, nrhs, n).t()


def _sizes(case):
    return np.random.default_rng(1).integers(case["lo"], case["hi"] + 1, case["count"]).astype(np.int32)


def _prepare_batch(case, seed):
    """Packed systems: even ones general, R + t sqrt(n) P with R uniform and P
    a permutation (its rows have to be interchanged), odd ones SPD, the
    symmetric part of R shifted past its spectrum.  The shift varies per
    system: condition numbers from a few to a few hundred."""
    ns = _sizes(case)
    g = torch.Generator("cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    n64 = ns.astype(np.int64)
    offA = np.concatenate([[0], np.cumsum(n64 * n64)])
    offB = np.concatenate([[0], np.cumsum(n64)])
    A = _uniform(g, int(offA[-1]))
    X = _uniform(g, int(offB[-1]))
    B = torch.empty_like(X)
    where, shift = [], []
    for i, n in enumerate(n64):
        if i % 2:
            a = A[offA[i]:offA[i + 1]].view(n, n)
            a.copy_(0.5 * (a + a.t()))
            rows, t = np.arange(n), 0.817 * rng.uniform(1.05, 1.6)
        else:
            rows, t = rng.permutation(n), 0.578 * rng.uniform(1.1, 1.8)
        where.append(offA[i] + rows + n * np.arange(n))
        shift.append(np.full(n, t * math.sqrt(n)))
    A.index_add_(0, torch.from_numpy(np.concatenate(where)).cuda(), torch.from_numpy(np.concatenate(shift)).cuda())
    for i, n in enumerate(n64):
        a = A[offA[i]:offA[i + 1]].view(n, n)          # row j holds column j
        torch.mv(a.t(), X[offB[i]:offB[i + 1]], out=B[offB[i]:offB[i + 1]])
    return ns, A, B, X


def _factors(n, g, rng):
    """LU factors and pivots as a getrf call leaves them: well conditioned, the
    pivot of step i anywhere below."""
    F = _uniform(g, n, n)
    F *= 0.5 / math.sqrt(n)
    d = F.diagonal()
    d.copy_(torch.where(d < 0, -1.0, 1.0) * (1.0 + d.abs() * math.sqrt(n)))
    ipiv = np.arange(1, n + 1) + (rng.random(n) * (n - np.arange(n))).astype(np.int64)
    return F.t(), ipiv.astype(np.int64)


def _permuted(X, ipiv, back):
    """P X, or P^T X, for getrf's interchanges."""
    p = np.arange(len(ipiv))
    for i, k in enumerate(ipiv - 1):
        p[i], p[k] = p[k], p[i]
    p = torch.from_numpy(p).cuda()
    if not back:
        return X[p]
    out = torch.empty_like(X)
    out[p] = X
    return out


def _inputs(case, seed):
    """(A, X, B, more) of one case; X is the solution B was made from."""
    g = torch.Generator("cuda").manual_seed(seed)
    n, nrhs = case["n"], case.get("nrhs", 1)
    if case["op"] == "getrs":
        F, ipiv = _factors(n, g, np.random.default_rng(seed))
        X = _solution(n, nrhs, g)
        Xm = X if X.dim() == 2 else X[:, None]
        U = F.triu()
        L = F.tril(-1)
        L.diagonal().fill_(1.0)
        if case["trans"]:
            Y = torch.matmul(U.t(), torch.matmul(L.t(), _permuted(Xm, ipiv, False)))
        else:
            Y = _permuted(torch.matmul(L, torch.matmul(U, Xm)), ipiv, True)
        B = Y[:, 0].contiguous() if X.dim() == 1 else Y.t().contiguous().t()
        return F, X, B, ipiv
    if case["op"] in ("posv", "potrf"):
        A = _shifted(n, g)
    elif case["op"] == "gesv" and case["kind"] == "rands":
        A = _uniform(g, n, n).t()
    else:
        A = _spectrum(n, case["cond"], seed, case["op"] == "posv_mixed")
    if case["op"] == "potrf":
        return A, None, None, None
    X = _solution(n, nrhs, g)
    return A, X, _times(A, X), None


def prepare(case, seed):
    if case["op"] == "batched":
        ns, A, B, X = _prepare_batch(case, seed)
        return {"case": case, "ns": ns, "A": A, "B": B, "X": torch.zeros_like(X)}
    A, X, B, more = _inputs(case, seed)
    del X
    s = {"case": case, "A": A, "B": B, "ipiv": more}
    if case["op"] in ("gesv", "posv", "potrf"):
        s["F"] = torch.empty_like(A)                   # the call overwrites its matrix
    if B is not None:
        s["X"] = torch.empty_like(B)
    if case["op"] in ("mixed", "posv_mixed"):
        s["opts"] = S.Options(factor_precision=PRECISIONS[case["precision"]])
    return s


# ---- one call ---------------------------------------------------------------
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "gesv":
        s["F"].copy_(s["A"])
        s["X"].copy_(s["B"])
        info, ipiv = S.gesv(s["F"], s["X"])
        return {"info": info, "ipiv": ipiv, "LU": s["F"], "X": s["X"]}
    if op == "getrs":
        s["X"].copy_(s["B"])
        S.getrs(s["A"], s["ipiv"], s["X"], trans=c["trans"])
        return {"X": s["X"]}
    if op == "posv":
        s["F"].copy_(s["A"])
        s["X"].copy_(s["B"])
        info = S.posv(s["F"], s["X"], uplo=S.UPPER if c["upper"] else S.LOWER)
        return {"info": info, "L": s["F"], "X": s["X"]}
    if op == "potrf":
        s["F"].copy_(s["A"])
        info = S.potrf(s["F"], uplo=S.UPPER if c["upper"] else S.LOWER)
        return {"info": info, "L": s["F"]}
    # The mixed drivers and the batch also report how they got there (iteration
    # counts, the float factor's pivots, the last backward error, which are
    # matters of rounding); what a program goes on with is the solution, and
    # whether refinement reached it.
    if op == "mixed":
        f = S.gesv_mixed_gmres if c["gmres"] else S.gesv_mixed
        info, it, _ = f(s["A"], s["B"], s["X"], s["opts"])
        return {"info": info, "refined": it >= 0, "X": s["X"]}
    if op == "posv_mixed":
        f = S.posv_mixed_gmres if c["gmres"] else S.posv_mixed
        info, it = f(s["A"], s["B"], s["X"], S.LOWER, s["opts"])
        return {"info": info, "refined": it >= 0, "X": s["X"]}
    _, info, _, _, _, _ = S.gesv_batched_auto(s["ns"], s["A"], s["B"], s["X"])
    return {"info": info, "X": s["X"]}


def work(case):
    if case["op"] == "batched":
        n = _sizes(case).astype(np.float64)
        return {"bytes": float(np.sum(8 * n * n + 16 * n)), "flops": float(np.sum(2 / 3 * n ** 3 + 2 * n * n))}
    n, nrhs = float(case["n"]), case.get("nrhs", 1)
    rhs, solve = 16 * n * nrhs, 2 * n * n * nrhs
    return {
        "gesv": {"bytes": 16 * n * n + rhs, "flops": 2 / 3 * n ** 3 + solve},
        "getrs": {"bytes": 8 * n * n + rhs, "flops": solve},
        "posv": {"bytes": 8 * n * n + rhs, "flops": n ** 3 / 3 + solve},
        "potrf": {"bytes": 8 * n * n, "flops": n ** 3 / 3},
        "mixed": {"bytes": 8 * n * n + rhs, "flops": 2 / 3 * n ** 3 + solve},
        "posv_mixed": {"bytes": 4 * n * n + rhs, "flops": n ** 3 / 3 + solve},
    }[case["op"]]


def exact(case, seed):
    if case["op"] == "batched":
        _, _, _, X = _prepare_batch(case, seed)
        return {"info": None, "X": X}
    A, X, _, _ = _inputs(case, seed)
    small = case["n"] <= FACTOR_MAX
    if case["op"] == "potrf" and not small:
        return None
    if case["op"] == "gesv":
        LU = torch.linalg.lu_factor(A.cpu())[0] if small else None      # LAPACK: strict partial pivoting
        return {"info": None, "ipiv": None, "LU": LU, "X": X}
    if case["op"] in ("posv", "potrf"):
        L = None
        if small:
            # the other triangle stays as it was given
            C = torch.linalg.cholesky(A, upper=case["upper"])
            L = C + (A.tril(-1) if case["upper"] else A.triu(1))
        out = {"info": None, "L": L}
        if case["op"] == "posv":
            out["X"] = X
        return out
    if case["op"] == "getrs":
        return {"X": X}
    return {"info": None, "refined": None, "X": X}
