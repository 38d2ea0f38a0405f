"""Solves that allocate nothing: the one-right-hand-side solve
(scuffx_lu_solve_noalloc; no counterpart in the reference, meant for
callers that cannot allocate device memory).  On the same factors its
result equals scuffx_lu_solve's (trans 'N', nrhs 1) bit for bit -- both
run the same kernels, only the buffers differ -- on two calls in a row,
the second with a smaller system; n beyond its maximum is an error."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve_both(sx, n, seed, prec):
    import torch
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    b = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    dtype = "complex128" if prec == 64 else "complex64"
    M = sx.HMatrix.from_numpy(A, dtype=dtype)
    assert M.LUFactorize() == 0
    L = sx.lib()
    sx._sync_stream()
    tdt = torch.complex128 if prec == 64 else torch.complex64
    b_ref = torch.tensor(b, dtype=tdt, device="cuda")
    b_na = b_ref.clone()
    print(f"  noalloc solve n={n} prec={prec}", flush=True)
    assert L.scuffx_lu_solve(sx._ptr(M.t), n, n, sx._ptr(M.ipiv), b"N", 1, sx._ptr(b_ref), n, prec) == 0
    rc = L.scuffx_lu_solve_noalloc(sx._ptr(M.t), n, n, sx._ptr(M.ipiv), sx._ptr(b_na), prec)
    assert rc == 0, L.scuffx_last_error()
    torch.cuda.synchronize()
    x_ref, x_na = b_ref.cpu().numpy(), b_na.cpu().numpy()
    assert np.array_equal(x_ref, x_na)
    x = x_na.astype(np.complex128)
    berr = np.linalg.norm(A @ x - b) / (np.linalg.norm(A) * np.linalg.norm(x))
    assert berr <= (1e-14 if prec == 64 else 1e-6), berr


@pytest.mark.parametrize("prec", [64, 32])
def test_noalloc_solve_matches_lu_solve(sx, prec):
    _solve_both(sx, 3000, 11 + prec, prec)
    _solve_both(sx, 1000, 12 + prec, prec)     # second call, smaller system


def test_noalloc_solve_rejects_large_n(sx):
    import torch
    L = sx.lib()
    sx._sync_stream()
    nmax = 16384
    assert L.scuffx_lu_solve_noalloc_bytes() >= 16 * nmax
    A = torch.zeros(4, dtype=torch.complex128, device="cuda")
    piv = torch.zeros(4, dtype=torch.int32, device="cuda")
    b = torch.zeros(4, dtype=torch.complex128, device="cuda")
    rc = L.scuffx_lu_solve_noalloc(sx._ptr(A), nmax + 1, nmax + 1, sx._ptr(piv), sx._ptr(b), 64)
    assert rc == -1
    assert "16384" in L.scuffx_last_error().decode()


def test_refinement_solve_allocates_nothing_past_residency(sx):
    """the refinement's triangular solves run on its own buffers whatever the
    number of their workgroups: with more 64-row blocks than workgroups fit on
    the GPU (three on each of 256 CUs) they take no further device memory.
    Identity matrix and factors, so that the solution is the right-hand side."""
    import ctypes as C
    import torch
    nmax = 784 * 64
    M = torch.zeros((nmax, nmax), dtype=torch.complex128, device="cuda")
    M.diagonal().fill_(1)
    LU = torch.zeros((nmax, nmax), dtype=torch.complex64, device="cuda")
    LU.diagonal().fill_(1)
    ipiv = torch.arange(1, nmax + 1, dtype=torch.int32, device="cuda")
    b = torch.randn(nmax, dtype=torch.complex128, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    x = torch.zeros_like(b)
    taken = []
    # the first size lets the refinement's own buffers grow to 9/8 of its need
    for n in (768 * 64 - 5, nmax):
        print(f"  refinement n={n}", flush=True)
        sx._sync_stream()
        torch.cuda.synchronize()
        it, rel = C.c_int(), C.c_double()
        free = torch.cuda.mem_get_info()[0]
        rc = sx.lib().scuffx_refine(sx._ptr(M), n, nmax, sx._ptr(LU), nmax, sx._ptr(ipiv), sx._ptr(b), sx._ptr(x),
                                    1e-13, 5, C.byref(it), C.byref(rel))
        assert rc == 0, sx.lib().scuffx_last_error()
        torch.cuda.synchronize()
        taken.append(free - torch.cuda.mem_get_info()[0])
        # (the residual's |re| + |im| is at most 1e-13 of the right-hand side's)
        assert (x[:n] - b[:n]).abs().max() <= 1e-13 * 2 ** 0.5 * b[:n].abs().max()
    assert taken[1] == 0, taken
