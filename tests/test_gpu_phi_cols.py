"""CP-APR Phi with one nonzero per lane: every rank it takes and the first it
does not, output rows that fill, cross or share its blocks of 64 nonzeros, last
blocks of every fill, 64- and 128-bit coordinates; gathered (alto_phi) against
the definition, stored and read back (CP-APR's product cache) against CP-APR
without the cache."""
import numpy as np
import pytest

from tests._tensors import mttkrp_numpy, uniform_tensor

pytestmark = pytest.mark.gpu

PI_CACHE, PHI_VARIANT = 19, 11


def _A():
    import alto_amd
    return alto_amd


def _phi_numpy(cidx, vals, U, mode, eps=1e-10):
    pi = np.ones((len(vals), U[0].shape[1]))
    for m, u in enumerate(U):
        if m != mode:
            pi *= u[cidx[m].astype(np.int64)]
    d = np.maximum((pi * U[mode][cidx[mode].astype(np.int64)]).sum(1), eps)
    return mttkrp_numpy(cidx, vals / d, U, mode)


ROWS = {
    "one row": [2] * 700,
    "every row once": list(range(300)),
    "runs of 64": [i // 64 for i in range(640)],
    "runs of 63": [i // 63 for i in range(630)],
    "runs of 16": [i // 16 for i in range(400)],
    "runs of 17": [i // 17 for i in range(400)],
    "mixed": [0] * 130 + [1, 2, 3] + [4] * 61 + [5] * 33 + [6] * 31 + list(range(7, 60)) + [60] * 200,
}


@pytest.mark.parametrize("R", [1, 2, 3, 4, 5, 7, 8, 9, 10, 11, 16, 17])
@pytest.mark.parametrize("name", sorted(ROWS))
def test_phi_rows(name, R):
    A = _A()
    rows = np.asarray(ROWS[name])
    n = len(rows)
    rng = np.random.default_rng(n)
    cell = rng.permutation(60 * 50)[:n]
    cidx = np.ascontiguousarray(np.stack([rows, cell // 50, cell % 50]).astype(np.uint64))
    vals = 1.0 + rng.integers(0, 5, n)
    dims = [int(rows.max()) + 1, 60, 50]
    U = [0.1 + rng.random((d, R)) for d in dims]
    t = A.AltoTensor(dims, cidx, vals)
    for m in range(3):
        want = _phi_numpy(cidx, vals, U, m)
        # positive terms: a sum of at most n of them, each with the roundings
        # of its products, of a dot product of R and of a division
        assert (np.abs(t.phi(m, U) - want) <= want * (n + R + 8) * 2.0 ** -52).all(), m


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 4097])
@pytest.mark.parametrize("bits", [64, 128])
def test_phi_sizes(n, bits):
    A = _A()
    dims = [50, 40, 30, 20] if bits == 64 else [1 << 14, 1 << 14, 1 << 14, 1 << 14, 1 << 10]
    cidx, vals = uniform_tensor(dims, n, n)
    rng = np.random.default_rng(1)
    U = [0.1 + rng.random((d, 10)) for d in dims]
    t = A.AltoTensor(dims, cidx, vals, lit_bits=bits)
    for m in range(len(dims)):
        want = _phi_numpy(cidx, vals, U, m)
        assert (np.abs(t.phi(m, U) - want) <= want * (n + 18) * 2.0 ** -52).all(), m


@pytest.mark.parametrize("R", [2, 3, 6, 10, 11, 13, 15, 16, 17])
@pytest.mark.parametrize("n", [65, 5000])
def test_cached_products(R, n):
    """The kept products change where pi comes from, not its value, so the two
    runs differ by the order of sums alone: n eps per Phi, carried through the
    18 multiplicative updates of the run (each can at most triple it)."""
    A = _A()
    dims = [40, 30, 20]
    cidx, vals = uniform_tensor(dims, n, 3)
    vals = np.ceil(vals * 4)
    t = A.AltoTensor(dims, cidx, vals)
    rng = np.random.default_rng(R)
    U0 = [0.1 + rng.random((d, R)) for d in dims]
    got = {}
    try:
        for cache in (1, 0):
            for variant in (1, 0):
                A.check(A.lib().alto_tune_set(PI_CACHE, cache), "tune_set")
                A.check(A.lib().alto_tune_set(PHI_VARIANT, variant), "tune_set")
                U, lam = [u.copy() for u in U0], np.ones(R)
                r = t.cp_apr(U, lam, 2, 3, dobench=True)
                got[cache, variant] = (U, lam, r["loglik"])
    finally:
        A.lib().alto_tune_set(PI_CACHE, 1)
        A.lib().alto_tune_set(PHI_VARIANT, 1)
    tol = n * 2.0 ** -52 * 3 ** 18
    for k in ((1, 1), (1, 0), (0, 1)):
        for a, b in zip(got[k][0] + [got[k][1]], got[0, 0][0] + [got[0, 0][1]]):
            assert np.abs(a - b).max() <= tol * np.abs(b).max()
        assert abs(got[k][2] - got[0, 0][2]) <= tol * abs(got[0, 0][2])
