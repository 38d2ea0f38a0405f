"""Sizes at which the exact LU's kernels and their dispatch can go wrong:
edges of panels, of 256-column blocks and of the rule that chooses how many
columns a workgroup of the block-row substitution takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = {"complex128": 2.0 ** -53, "float64": 2.0 ** -53, "complex64": 2.0 ** -24}


def matrix(n, dtype, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n))
    if dtype != "float64":
        A = A + 1j * rng.standard_normal((n, n))
    return A.astype(dtype)


def backward_error(A, F, piv):
    """|P A - L U| / |A| in the Frobenius norm"""
    n = A.shape[0]
    wide = np.complex128 if np.iscomplexobj(A) else np.float64
    L = np.tril(F, -1).astype(wide) + np.eye(n)
    U = np.triu(F).astype(wide)
    perm = np.arange(n)
    for i in range(n):
        p = piv[i] - 1
        perm[[i, p]] = perm[[p, i]]
    assert np.abs(np.tril(F, -1)).max(initial=0.0) <= np.sqrt(2.0) * (1 + 8 * EPS[str(A.dtype)])
    return np.linalg.norm(A.astype(wide)[perm] - L @ U) / np.linalg.norm(A)


# 1024: 512 columns right of the next block (one per workgroup), 1025: 513
# (four per workgroup, one in the last); 1283: ragged last block and panel
@pytest.mark.parametrize("dtype", ["complex128", "float64", "complex64"])
@pytest.mark.parametrize("n", [31, 33, 289, 1024, 1025, 1283])
def test_block_rows(sx, n, dtype):
    print(f"block rows n={n} {dtype}", flush=True)
    A = matrix(n, dtype, 31 * n)
    M = sx.HMatrix.from_numpy(A, dtype=dtype)
    assert M.LUFactorize() == 0
    # |L| |U| of a random matrix under partial pivoting grows like n^(1/2)
    # to n^(2/3) relative to |A|, and rounding adds up as n^(1/2): 4 n eps
    # covers both with room (seen: below n eps)
    berr = backward_error(A, M.numpy(), M.ipiv.cpu().numpy())
    assert berr <= 4 * max(n, 32) * EPS[dtype], berr


# order 2^k Hadamard matrices: every entry of every remaining column ties with
# the largest (+-2^j), and elimination is exact, so the interchanges are
# LAPACK's only if each tie goes to the first row by its current position,
# within a workgroup and across workgroups (256 rows each)
@pytest.mark.parametrize("dtype", ["complex128", "float64", "complex64"])
@pytest.mark.parametrize("n", [64, 512, 1024])
def test_pivot_ties(sx, n, dtype):
    import scipy.linalg as sl
    print(f"pivot ties n={n} {dtype}", flush=True)
    H = sl.hadamard(n).astype("float64")
    rng = np.random.default_rng(n)
    H = H[rng.permutation(n)]
    LU, piv = sl.lu_factor(H)
    A = H.astype(dtype)
    M = sx.HMatrix.from_numpy(A, dtype=dtype)
    assert M.LUFactorize() == 0
    assert np.array_equal(M.ipiv.cpu().numpy(), piv + 1)
    assert np.array_equal(M.numpy(), LU.astype(dtype))


# past 15 workgroups (3840 rows) the panel polls keys first and reads the
# winner's row after them; the last panels of the same matrix read all
# candidates at once
def test_panel_both_exchanges(sx):
    import scipy.linalg as sl
    n = 4100
    print(f"both panel exchanges n={n}", flush=True)
    A = matrix(n, "float64", 5)
    M = sx.HMatrix.from_numpy(A)
    assert M.LUFactorize() == 0
    LU, piv = sl.lu_factor(A)
    assert np.array_equal(M.ipiv.cpu().numpy(), piv + 1)
    # same pivots: the factors differ by rounding carried through n steps
    assert np.max(np.abs(M.numpy() - LU)) <= 4 * n * EPS["float64"] * np.max(np.abs(LU)) * 10


# the same with the complex slots (66 and 34 words).  complex128: LAPACK's
# pivots; complex64, where roundings decide near-ties: P A v = L (U v) for
# vectors v, and multipliers of at most sqrt(2)
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_panel_both_exchanges_complex(sx, dtype):
    import scipy.linalg as sl
    n = 4100
    print(f"both panel exchanges n={n} {dtype}", flush=True)
    A = matrix(n, dtype, 5)
    M = sx.HMatrix.from_numpy(A, dtype=dtype)
    assert M.LUFactorize() == 0
    F, piv = M.numpy(), M.ipiv.cpu().numpy()
    if dtype == "complex128":
        assert np.array_equal(piv, sl.lu_factor(A)[1] + 1)
    assert np.abs(np.tril(F, -1)).max() <= np.sqrt(2.0) * (1 + 8 * EPS[dtype])
    perm = np.arange(n)
    for i in range(n):
        perm[[i, piv[i] - 1]] = perm[[piv[i] - 1, i]]
    V = matrix(n, "complex128", 8)[:, :4]
    UV = np.triu(F).astype("complex128") @ V
    LUV = np.tril(F, -1).astype("complex128") @ UV + UV
    res = np.linalg.norm(A.astype("complex128")[perm] @ V - LUV) / (np.linalg.norm(A) * np.linalg.norm(V) / np.sqrt(n))
    assert res <= 4 * n * EPS[dtype], res        # (as for the smaller orders)


# solves by blocks of 64 rows and tiles of 16 columns: one row, the edges of
# a block and of a tile, one and several blocks, a ragged last block; 1100
# columns take two sets
@pytest.mark.parametrize("dtype", ["complex128", "float64", "complex64"])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (1, 3), (63, 2), (64, 16), (65, 17), (300, 1), (300, 40), (1030, 5),
                                    (300, 600), (130, 1100)])
def test_solve_blocks(sx, n, nrhs, dtype):
    A = matrix(n, dtype, 7 * n + nrhs)
    B = matrix(max(n, nrhs), dtype, n + nrhs)[:n, :nrhs].copy()
    M = sx.HMatrix.from_numpy(A, dtype=dtype)
    assert M.LUFactorize() == 0
    wide = np.complex128 if np.iscomplexobj(A) else np.float64
    for trans in "NTC":
        print(f"solve n={n} nrhs={nrhs} {trans} {dtype}", flush=True)
        X = sx.HMatrix.from_numpy(B, dtype=dtype)
        M.LUSolve(X, Trans=trans)
        x = X.numpy().astype(wide)
        op = {"N": A, "T": A.T, "C": A.conj().T}[trans].astype(wide)
        # columnwise |b - op(A) x| against |A| |x|: the factorization's
        # backward error (4 n eps, as above) and two triangles of inner
        # products, with the 64-row blocks' inverses, of the same order
        res = np.linalg.norm(B - op @ x, axis=0) / (np.linalg.norm(A) * np.linalg.norm(x, axis=0))
        assert res.max() <= 8 * max(n, 32) * EPS[dtype], res.max()


# the batch's complex64 solves multiply by inverses of the 64x64 diagonal
# blocks; near the low-frequency limit of a Drude sphere the refinement stays
# within its fixed steps only if U times the inverse, not the inverse times U,
# is the identity to rounding (the other way five of these sixteen instances
# or their like had to be solved again, at residuals up to 1e-11)
def test_block_inverses_low_frequency(sx, O):
    V0, T = O.icosphere(3)
    Gs = []
    for seed in range(4):
        V = V0 + np.random.default_rng(seed).uniform(-0.02, 0.02, V0.shape) / 8
        G = sx.RWGGeometry()
        G.AddMesh(V, T, "DRUDE_10_0.1")
        Gs.append(G)
    print("low-frequency batch", flush=True)
    pw = sx.PlaneWave([1.0, 0.0, 0.0], [0.0, 0.0, 1.0])
    _, rel, info = sx.SweepBatched(Gs, np.array([0.049, 0.058, 0.067, 0.079]), pw)
    assert info[0] == 0
    assert np.max(rel) <= 2e-12, rel


# the mixed factorization's block rows on the matrix units: past 4096 columns
# right of the next block, a number of columns that is no multiple of 16 and an
# odd leading dimension
def test_mixed_wide_block_rows(sx):
    import torch
    n = 4699
    print(f"mixed block rows n={n}", flush=True)
    A = matrix(n, "complex64", 11)
    M = sx.HMatrix.from_numpy(A.astype("complex128"))
    LU32 = torch.zeros((n, n), dtype=torch.complex64, device="cuda")
    ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
    assert sx.lib().scuffx_lu32_from_c128(sx._ptr(M.t), n, n, sx._ptr(LU32), n, sx._ptr(ipiv)) == 0
    F, piv = LU32.cpu().numpy().T, ipiv.cpu().numpy()
    perm = np.arange(n)
    for i in range(n):
        perm[[i, piv[i] - 1]] = perm[[piv[i] - 1, i]]
    # P A v = L (U v) for a few vectors, against |L| |U| of a random matrix
    # (2e-5 sqrt(n / 40) relative to |A|, as for the smaller orders)
    v = matrix(8, "complex128", 3)[0][:4]
    V = np.outer(np.ones(n), v) * np.random.default_rng(4).standard_normal((n, 4))
    UV = np.triu(F).astype("complex128") @ V
    LUV = np.tril(F, -1).astype("complex128") @ UV + UV
    res = np.linalg.norm(A.astype("complex128")[perm] @ V - LUV) / (np.linalg.norm(A) * np.linalg.norm(V) / np.sqrt(n))
    assert res <= 2e-5 * np.sqrt(n / 40), res


# solves with one right-hand side near the low-frequency limit, where a
# dielectric's electric and magnetic rows differ by 1e6: products with the
# inverses of the 64x64 diagonal blocks lost seven digits.  Substitution solves
# (T + dT) x = b with |dT| <= gamma_n |T| for each triangle (Higham, Accuracy
# and Stability, theorem 8.5), so |P b - L U x| <= 2 gamma_n |L| |U| |x| entry by
# entry; a complex product rounds 2 sqrt(2) times as much as a real one
@pytest.mark.parametrize("dtype,noalloc", [("complex128", False), ("float64", False), ("complex128", True),
                                           ("complex64", False), ("complex64", True)])
def test_badly_scaled_blocks(sx, O, dtype, noalloc):
    V, T = O.icosphere(2)
    G = sx.RWGGeometry()
    G.AddMesh(V, T, "CONST_EPS_10")
    print(f"badly scaled blocks {dtype} noalloc={noalloc}", flush=True)
    A = G.AssembleBEMMatrix(0.001j).numpy()
    if dtype == "float64":
        A = A.real.copy()
    A = A.astype(dtype)
    n = A.shape[0]
    M = sx.HMatrix.from_numpy(A, dtype=dtype)
    assert M.LUFactorize() == 0
    F, piv = M.numpy(), M.ipiv.cpu().numpy()
    wide = np.longdouble if dtype == "float64" else np.clongdouble
    L, U = np.tril(F, -1).astype(wide) + np.eye(n), np.triu(F).astype(wide)
    perm = np.arange(n)
    for i in range(n):
        perm[[i, piv[i] - 1]] = perm[[piv[i] - 1, i]]
    for rows in (np.arange(n) % 2, np.ones(n)):
        b = (matrix(n, dtype, 17)[0] * rows).astype(dtype)
        X = sx.HMatrix.from_numpy(b.reshape(n, 1), dtype=dtype)
        if noalloc:
            rc = sx.lib().scuffx_lu_solve_noalloc(sx._ptr(M.t), n, n, sx._ptr(M.ipiv), sx._ptr(X.t), M.prec)
            assert rc == 0
        else:
            M.LUSolve(X)
        x = X.numpy()[:, 0].astype(wide)
        res = np.abs(b[perm].astype(wide) - L @ (U @ x))
        bound = np.abs(L) @ (np.abs(U) @ np.abs(x))
        c = 1.0 if dtype == "float64" else 2.0 * np.sqrt(2.0)
        print(f"  {float(np.max(res / bound)):.2e}", flush=True)
        assert np.max(res / bound) <= 2 * c * n * EPS[dtype]


def triangular(F, piv, B, trans, dtype, partial):
    """op(P^T L U) X = B row by row in dtype; a row's products in `partial`
    strided partial sums (0: one sum)"""
    n = F.shape[0]
    F, X = F.astype(dtype), B.astype(dtype)
    pad = np.zeros((max(1, partial) * (-(-n // max(1, partial))), X.shape[1]), dtype=dtype)

    def dot(a, lo, hi):
        if not partial:
            return a @ X[lo:hi]
        v = pad[:partial * (-(-(hi - lo) // partial))]
        v[:hi - lo] = a[:, None] * X[lo:hi]
        v[hi - lo:] = 0
        s = np.zeros((partial, X.shape[1]), dtype=dtype)
        for part in v.reshape(-1, partial, X.shape[1]):
            s = s + part
        while len(s) > 1:
            s = s[:len(s) // 2] + s[len(s) // 2:]
        return s[0]

    if trans == "N":
        for i in range(n):
            X[[i, piv[i] - 1]] = X[[piv[i] - 1, i]]
        for i in range(1, n):
            X[i] = X[i] - dot(F[i, :i], 0, i)
        for i in range(n - 1, -1, -1):
            X[i] = (X[i] - dot(F[i, i + 1:], i + 1, n)) / F[i, i]
    else:
        for i in range(n):
            X[i] = (X[i] - dot(F[:i, i], 0, i)) / F[i, i]
        for i in range(n - 2, -1, -1):
            X[i] = X[i] - dot(F[i + 1:, i], i + 1, n)
        for i in range(n - 1, -1, -1):
            X[[i, piv[i] - 1]] = X[[piv[i] - 1, i]]
    return X


# rounding of the solves against the same factors in wider arithmetic.  The
# yardstick is substitution in the same type with a row's products in 256
# partial sums, as one workgroup a row would take them: transposed systems
# are to be no further off (they were 1.7 to 3.7 times as far), untransposed ones,
# which do not keep what their subtractions lose, within 1.5 times (they were 1.7
# to 3.5; seen 1.2 to 1.5).  A quarter more allows for the scatter of eight
# columns; 0 columns: the inverse
@pytest.mark.parametrize("dtype", ["complex128", "float64", "complex64"])
@pytest.mark.parametrize("n,nrhs", [(100, 8), (300, 8), (970, 8), (64, 0), (200, 0)])
def test_solve_rounding(sx, n, nrhs, dtype):
    print(f"solve rounding n={n} {dtype}", flush=True)
    scale = 1.0 if dtype == "float64" else np.sqrt(0.5)
    A = (matrix(n, "complex128" if dtype != "float64" else dtype, 5 * n) * scale + 1.2 * np.sqrt(n) * np.eye(n))
    M = sx.HMatrix.from_numpy(A.astype(dtype), dtype=dtype)
    assert M.LUFactorize() == 0
    F, piv = M.numpy(), M.ipiv.cpu().numpy()
    B = matrix(max(n, nrhs), dtype, n)[:n, :nrhs].copy() if nrhs else np.eye(n, dtype=dtype)
    wide = {"complex128": np.clongdouble, "float64": np.longdouble, "complex64": np.complex128}[dtype]
    for trans, allowed in (("N", 1.5), ("T", 1.0)):
        exact = triangular(F, piv, B, trans, wide, 0)

        def err(X):
            return float(np.linalg.norm(np.abs(X - exact)) / np.linalg.norm(np.abs(exact)))

        X = sx.HMatrix.from_numpy(B, dtype=dtype)
        M.LUSolve(X, Trans=trans)
        e, e0 = err(X.numpy()), err(triangular(F, piv, B, trans, dtype, 256))
        print(f"  {trans} {e:.2e}, yardstick {e0:.2e}", flush=True)
        assert e <= 1.25 * allowed * e0, (trans, e, e0)


def test_factorizations_side_by_side(sx):
    """Threads that factor at once, each on a stream of its own (both panel
    exchanges, a panel in one workgroup, tournament pivoting): the same bits as
    one after another."""
    import threading
    import torch
    work = [(4100, "complex128"), (1500, "float64"), (2600, "complex64"), (4000, "mixed"), (400, "complex128")]
    A = [matrix(n, "complex128" if d == "mixed" else d, n) for n, d in work]

    def factor(i):
        n, d = work[i]
        if d != "mixed":
            M = sx.HMatrix.from_numpy(A[i], dtype=d)
            assert M.LUFactorize() == 0
            return M.t, M.ipiv
        M = sx.HMatrix.from_numpy(A[i])
        LU32 = torch.zeros((n, n), dtype=torch.complex64, device="cuda")
        ipiv = torch.zeros(n, dtype=torch.int32, device="cuda")
        sx._sync_stream()
        assert sx.lib().scuffx_lu32_from_c128(sx._ptr(M.t), n, n, sx._ptr(LU32), n, sx._ptr(ipiv)) == 0
        return LU32, ipiv

    print("factorizations side by side", flush=True)
    alone = [[t.cpu() for t in factor(i)] for i in range(len(work))]
    together = [None] * len(work)

    def thread(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            out = factor(i)
            torch.cuda.current_stream().synchronize()
            together[i] = [t.cpu() for t in out]

    ts = [threading.Thread(target=thread, args=(i,)) for i in range(len(work))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for a, b in zip(alone, together):
        assert b is not None and all(torch.equal(x, y) for x, y in zip(a, b))
