"""The vector-lane MTTKRP kernels at ranks that no lane width divides, with and
without the fiber layout, and the combining of a workgroup's last rows: rows
that cover one group, several wavefronts, whole workgroups, and streams shorter
than one segment."""
import numpy as np
import pytest

from tests._tensors import mttkrp_numpy, uniform_tensor, zipf_tensor

pytestmark = pytest.mark.gpu

SEG, NARROW_RANK, NARROW_SMALL, FIBERS, FIBER_MIN_NNZ = 1, 10, 12, 13, 16


def _A():
    import alto_amd
    return alto_amd


@pytest.fixture
def tune():
    A = _A()
    yield lambda p, v: A.check(A.lib().alto_tune_set(p, v), "tune_set")
    for p, v in ((SEG, 0), (NARROW_RANK, 32), (NARROW_SMALL, 1), (FIBERS, 1), (FIBER_MIN_NNZ, 4 << 20)):
        A.check(A.lib().alto_tune_set(p, v), "tune_set")


def _bound(A, prec, cidx, vals, U, mode):
    """Entry-wise error bound: the sum of the terms' magnitudes (all terms are
    positive) times the roundings on a term's way -- its factors and products
    (N + 1), and a sum of at most nnz terms, which in the 32-bit modes runs
    over at most 4096 terms before it goes on in 64 bits."""
    N, n = len(U), len(vals)
    eps = 2.0 ** -52 if prec == A.PREC_F64 else 2.0 ** -23
    return mttkrp_numpy(cidx, vals, U, mode) * eps * (N + 1 + min(n, 4096 if prec else n))


@pytest.mark.parametrize("fibers", [0, 1])
@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("R", [2, 3, 5, 15, 17, 18, 31, 33, 50, 63, 66, 127, 128])
def test_ranks(tune, R, prec, fibers):
    A = _A()
    tune(FIBERS, fibers)
    tune(FIBER_MIN_NNZ, 0)
    dims = [40, 70, 30, 9]
    cidx, vals = zipf_tensor(dims, 12000, R, s=1.1)
    g = A.AltoTensor(dims, cidx, vals)
    rng = np.random.default_rng(R)
    U = [rng.random((d, R)) for d in dims]
    if prec == A.PREC_BF16:
        U = [A.from_bf16_bits(A.to_bf16_bits(u)).astype(np.float64) for u in U]
    elif prec == A.PREC_F32:
        U = [u.astype(np.float32).astype(np.float64) for u in U]
    for narrow in ([32] if prec == A.PREC_F64 else [0, 128]):
        tune(NARROW_RANK, narrow)
        tune(NARROW_SMALL, 0)
        for m in range(len(dims)):
            err = np.abs(g.mttkrp(m, U, prec) - mttkrp_numpy(cidx, vals, U, m))
            assert (err <= _bound(A, prec, cidx, vals, U, m)).all(), (m, narrow)


def _rows_tensor(rows, seed):
    """One nonzero per entry of `rows` (mode 0), other coordinates distinct."""
    n = len(rows)
    rng = np.random.default_rng(seed)
    cell = rng.permutation(200 * 300)[:n] if n <= 60000 else None
    cidx = np.stack([np.asarray(rows), cell // 300, cell % 300]).astype(np.uint64)
    return [int(max(rows)) + 1, 200, 300], np.ascontiguousarray(cidx), 0.5 + rng.random(n)


ROWS = {
    "one row": [3] * 20000,
    "a row in the middle": list(range(300)) + [300] * 9000 + list(range(301, 700)),
    "two heavy rows": [0] * 4097 + [5] * 4095 + [6],
    "every row once": list(range(3000)),
    "one nonzero": [0],
    "runs of three": [i // 3 for i in range(5000)],
    "runs of a segment": [i // 16 for i in range(5000)],
    "row 0 last": [1] * 700 + [0] * 1300,
}


@pytest.mark.parametrize("seg", [0, 1, 7, 16, 64])
@pytest.mark.parametrize("R", [2, 8, 16, 32, 64, 100])
@pytest.mark.parametrize("name", sorted(ROWS))
def test_last_rows_combined(tune, name, R, seg):
    A = _A()
    tune(SEG, seg)
    dims, cidx, vals = _rows_tensor(ROWS[name], 5)
    rng = np.random.default_rng(1)
    U = [rng.random((d, R)) for d in dims]
    for fibers in (0, 1):
        tune(FIBERS, fibers)
        tune(FIBER_MIN_NNZ, 0)
        g = A.AltoTensor(dims, cidx, vals)
        for m in range(3):
            err = np.abs(g.mttkrp(m, U) - mttkrp_numpy(cidx, vals, U, m))
            assert (err <= _bound(A, 0, cidx, vals, U, m)).all(), (m, fibers)


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_batched_odd_ranks(prec):
    A = _A()
    rng = np.random.default_rng(7)
    ts, Us, co = [], [], []
    for k, (dims, n) in enumerate([([30, 40, 50], 900), ([9, 300, 20, 7], 5000), ([64, 64, 64], 1)]):
        cidx, vals = uniform_tensor(dims, n, k)
        ts.append(A.AltoTensor(dims, cidx, vals))
        co.append((cidx, vals))
        U = [rng.random((d, 26)).astype(np.float32).astype(np.float64) for d in dims]
        Us.append([A.from_bf16_bits(A.to_bf16_bits(u)).astype(np.float64) for u in U] if prec == A.PREC_BF16 else U)
    for mode in range(3):
        got = A.mttkrp_batched(ts, [mode] * 3, Us, prec)
        for o, (cidx, vals), U in zip(got, co, Us):
            err = np.abs(o - mttkrp_numpy(cidx, vals, U, mode))
            assert (err <= _bound(A, prec, cidx, vals, U, mode)).all()


@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("R", [34, 40, 64, 66, 128])
def test_batched_wide_lanes(tune, R, prec):
    """Four (FP32) and eight (BF16) columns per lane in the batched launch."""
    A = _A()
    tune(NARROW_RANK, 0)
    tune(NARROW_SMALL, 0)
    rng = np.random.default_rng(R)
    ts, Us, co = [], [], []
    for k, (dims, n) in enumerate([([30, 40, 50], 900), ([9, 300, 20, 7], 5000), ([64, 64, 64], 1)]):
        cidx, vals = uniform_tensor(dims, n, k)
        ts.append(A.AltoTensor(dims, cidx, vals))
        co.append((cidx, vals))
        U = [rng.random((d, R)).astype(np.float32).astype(np.float64) for d in dims]
        Us.append([A.from_bf16_bits(A.to_bf16_bits(u)).astype(np.float64) for u in U] if prec == A.PREC_BF16 else U)
    for mode in range(3):
        got = A.mttkrp_batched(ts, [mode] * 3, Us, prec)
        for o, (cidx, vals), U in zip(got, co, Us):
            err = np.abs(o - mttkrp_numpy(cidx, vals, U, mode))
            assert (err <= _bound(A, prec, cidx, vals, U, mode)).all()


@pytest.mark.parametrize("prec", [0, 1, 2])
def test_infinite_and_nan_entries_stay_where_they_are(tune, prec):
    """Non-finite factor entries reach the rows of their own nonzeros and no
    others: lanes past a segment's end read row 0 of every mode."""
    A = _A()
    tune(FIBER_MIN_NNZ, 0)
    tune(NARROW_SMALL, 0)
    dims, R = [50, 60, 40], 40
    cidx, vals = zipf_tensor(dims, 4001, 2, s=1.1)
    keep = (cidx[1] != 0) | (cidx[0] % 2 == 1)
    cidx, vals = np.ascontiguousarray(cidx[:, keep]), vals[keep]
    rng = np.random.default_rng(4)
    U = [rng.integers(1, 9, (d, R)).astype(np.float64) for d in dims]
    U[1][0, ::3] = np.inf
    U[1][0, 1::3] = np.nan
    for fibers in (0, 1):
        tune(FIBERS, fibers)
        got = A.AltoTensor(dims, cidx, vals).mttkrp(0, U, prec)
        hit = np.zeros(dims[0], bool)
        hit[cidx[0][cidx[1] == 0].astype(np.int64)] = True
        assert np.isinf(got[hit][:, ::3]).all() and np.isnan(got[hit][:, 1::3]).all()
        assert np.isfinite(got[~hit]).all() and np.isfinite(got[:, 2::3]).all()
