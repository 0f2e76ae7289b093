"""GPU parity of the CP-ALS mode updates at the sizes where their launches
change: the inverse per rank class, row solves that invert V themselves (up to
rank 16 and 32768 rows), lambda taken in the Gram launch (up to 128 row blocks
and row blocks x rank 2048) and Grams left in partials (up to 8 row blocks of
the Gram), with sizes on both sides of those lines."""
import ctypes

import numpy as np
import pytest
import scipy.linalg

import oracle
from tests._tensors import uniform_tensor

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def _A():
    import alto_amd
    return alto_amd


def _run(dims, R, iters, dup=False, prec=0):
    """(factors, lambda, fits) of the library and of the oracle."""
    cidx, vals = uniform_tensor(dims, 6000, 17)
    U, _ = oracle.random_init(dims, R, 3)
    if dup:  # equal columns: V is singular and its elimination meets a zero pivot
        for u in U:
            u[:, R - 1] = u[:, 0]
    g = _A().AltoTensor(dims, cidx, vals, nprtn=8)
    s = _A().CpdSession(g, U, precision=prec)
    fits, _ = s.iterate(iters)
    return s.get(), fits, (dims, cidx, vals, U)


def _als(dims, cidx, vals, U, iters):
    """CP-ALS in numpy with the largest condition number of a V on the way."""
    U = [u.copy() for u in U]
    N, R, cond = len(dims), U[0].shape[1], 1.0
    grams = [u.T @ u for u in U]
    fits = []
    for it in range(iters):
        for j in range(N):
            rows = np.prod([U[m][cidx[m].astype(np.int64)] for m in range(N) if m != j], axis=0) * vals[:, None]
            M = np.zeros((dims[j], R))
            np.add.at(M, cidx[j].astype(np.int64), rows)
            V = np.prod([grams[m] for m in range(N) if m != j], axis=0)
            cond = max(cond, np.linalg.cond(V))
            u = scipy.linalg.solve(V, M.T, assume_a="pos").T
            lam = np.sqrt((u * u).sum(0)) if it == 0 else np.maximum(u.max(0), 1.0)
            U[j] = u / lam
            grams[j] = U[j].T @ U[j]
        normX = (vals * vals).sum()
        inner = (M * U[-1] * lam).sum()
        normU = lam @ np.prod(grams, axis=0) @ lam
        fits.append(1 - np.sqrt(normX + normU - 2 * inner) / np.sqrt(normX))
    return U, lam, fits, cond


EDGES = [(1, 300), (15, 2048), (16, 2048), (16, 2049), (16, 8192), (16, 8193), (16, 32768), (16, 32769), (17, 512),
         (31, 3800), (32, 512), (32, 513), (32, 16384), (32, 16385), (33, 2048), (48, 2730), (63, 2049), (64, 2048),
         (64, 2049), (65, 500), (128, 300)]


@pytest.mark.parametrize("R,rows", EDGES)
def test_mode_updates_match_numpy(R, rows):
    """Three iterations.  Every solve may lose cond(V) rounding errors per
    term of its sums, and each update starts from the one before it."""
    dims = [rows, 2 * R + 7, 3 * R + 5]
    (U, lam, _, _), fits, args = _run(dims, R, 3)
    Uo, lo, fo, cond = _als(*args, 3)
    tol = 9 * 8 * R * EPS * cond
    np.testing.assert_allclose(fits, fo, rtol=0, atol=tol)
    np.testing.assert_allclose(lam, lo, rtol=tol)
    for a, b in zip(U, Uo):
        np.testing.assert_allclose(a, b, rtol=0, atol=tol * np.abs(b).max())


@pytest.mark.parametrize("R", [2, 15, 16, 17, 32, 33, 64])
def test_singular_v_takes_the_pseudo_inverse(R):
    """The first update of a model with two equal columns against LAPACK's
    minimum-norm solution (later updates see factors that differ from equal
    columns by rounding)."""
    dims = [70, 2 * R + 7, 3 * R + 5]
    (U, _, _, _), _, (_, cidx, vals, U0) = _run(dims, R, 1, dup=True)
    rows = U0[1][cidx[1].astype(np.int64)] * U0[2][cidx[2].astype(np.int64)] * vals[:, None]
    M = np.zeros((dims[0], R))
    np.add.at(M, cidx[0].astype(np.int64), rows)
    V = (U0[1].T @ U0[1]) * (U0[2].T @ U0[2])
    e = np.linalg.eigvalsh(V)
    want = M @ np.linalg.pinv(V, rcond=1e-12, hermitian=True)
    want /= np.sqrt((want * want).sum(0))
    np.testing.assert_allclose(U[0], want, rtol=0, atol=64 * R * EPS * e[-1] / e[1] * np.abs(want).max())


@pytest.mark.parametrize("prec,tol", [(1, 1e-4), (2, 1e-3)])
@pytest.mark.parametrize("R,rows", [(16, 2048), (16, 8193), (32, 513), (64, 2049)])
def test_mode_updates_reduced_precision(prec, tol, R, rows):
    """FP32 / BF16 models: the fit within the bounds the CP-ALS runs of these
    precisions keep elsewhere."""
    dims = [rows, 2 * R + 7, 3 * R + 5]
    _, fits, (_, cidx, vals, U) = _run(dims, R, 4, prec=prec)
    o = oracle.OracleAlto(dims, cidx, vals, nprtn=8)
    Uo, lo = oracle.random_init(dims, R, 3)
    _, fo = o.cpd_als(Uo, lo, 4, 0.0)
    assert abs(fits[-1] - fo[-1]) <= tol * max(1.0, abs(fo[-1]))


@pytest.mark.parametrize("R", [2, 3, 7, 16, 17, 31, 32, 33, 64, 65, 101, 127, 128])
def test_pseudo_inverse_of_half_rank(R):
    """V of rank about R / 2 with a zero row (its pivot is exactly zero), so that
    the rotations sweep many times, against LAPACK's minimum-norm solution."""
    A = _A()
    rng = np.random.default_rng(R)
    B = rng.random((R, (R + 1) // 2)) - 0.3
    B[R // 2] = 0
    V = B @ B.T
    M = rng.random((50, R))
    g, d = A.DeviceArray.from_numpy(np.stack([np.eye(R), V])), A.DeviceArray.from_numpy(M)
    fb = ctypes.c_int(0)
    A.check(A.lib().alto_pseudo_inverse(g.ptr, 2, 0, R, d.ptr, 50, ctypes.byref(fb), None), "pinv")
    e = np.linalg.eigvalsh(V)
    e = e[e > 1e-10 * e[-1]]
    want = M @ np.linalg.pinv(V, rcond=1e-10, hermitian=True)
    assert fb.value == 1
    np.testing.assert_allclose(d.numpy(), want, rtol=0, atol=64 * R * EPS * e[-1] / e[0] * np.abs(want).max())


@pytest.mark.parametrize("R,prec", [(3, 0), (16, 0), (16, 1), (9, 2)])
def test_many_row_solve_blocks_equal_one_model(R, prec):
    """Five models in lockstep, whose modes of 32768 rows together pass the number
    of blocks up to which row solves invert V themselves, against the same models
    one by one (512 blocks each, which do): the same bits, MTTKRPs in a fixed
    order."""
    A = _A()
    L = A.lib()
    dims = [32768, 60, 32768]
    tensors = [A.AltoTensor(dims, *uniform_tensor(dims, 5000, k)) for k in range(5)]
    U = [oracle.random_init(dims, R, 3 + k)[0] for k in range(5)]
    A.check(L.alto_tune_set(18, 1), "deterministic")
    try:
        one = [A.CpdSession(t, u, prec) for t, u in zip(tensors, U)]
        for s in one:
            s.iterate(3)
        many = [A.CpdSession(t, u, prec) for t, u in zip(tensors, U)]
        A.cpd_sessions_iterate(many, 3, 0.0)
    finally:
        A.check(L.alto_tune_set(18, 0), "deterministic")
    for a, b in zip(one, many):
        (Ua, la, fa, _), (Ub, lb, fb, _) = a.get(), b.get()
        assert fa == fb and np.array_equal(la, lb)
        for x, y in zip(Ua, Ub):
            np.testing.assert_array_equal(x, y)
