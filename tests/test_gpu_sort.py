"""The radix sort and the orderings built on it at the sizes where they can go
wrong: around its tiles (1024 and 4096 pairs), the switch of the tile size at
2^20, 64- and 128-bit keys, key bits that a digit width does not divide, and
equal keys (the order must stay that of the input)."""
import numpy as np
import pytest

import oracle
from tests._tensors import uniform_tensor

pytestmark = pytest.mark.gpu


def _A():
    import alto_amd
    return alto_amd


def _check(dims, cidx, vals, W, nprtn):
    A = _A()
    g = A.AltoTensor(dims, cidx, vals, nprtn=nprtn, lit_bits=64 * W)
    o = oracle.OracleAlto(dims, cidx, vals, W=W, nprtn=nprtn)
    gs, os_ = g.export(), o.state()
    for k in ("idx", "vals", "prtn_ptr", "intervals", "cr_masks"):
        assert np.array_equal(gs[k], os_[k]), k
    return g


@pytest.mark.parametrize("W", [1, 2])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 4095, 4097, 20481])
def test_create_sizes(n, W):
    cidx, vals = uniform_tensor([700, 90, 41], n, n)
    _check([700, 90, 41], cidx, vals, W, 3)


@pytest.mark.parametrize("n", [(1 << 20) - 1, 1 << 20, (1 << 20) + 1, 4096 * 300 + 5])
def test_create_around_the_tile_switch(n):
    dims = [5000, 1201, 333]
    cidx, vals = uniform_tensor(dims, n, 4)
    g = _check(dims, cidx, vals, 1, 16)
    # a stream of every mode: the first MTTKRP against a row sum
    ones = [np.ones((d, 2)) for d in dims]
    for m, d in enumerate(dims):
        want = np.bincount(cidx[m].astype(np.int64), weights=vals, minlength=d)
        # at most n additions of values in (0, 1]
        assert np.abs(g.mttkrp(m, ones)[:, 1] - want).max() <= n * 2.0 ** -52 * max(want.max(), 1.0)


@pytest.mark.parametrize("dims", [[2, 2, 2], [3, 1, 5], [1 << 20, 1 << 17, 3], [1 << 30, 1 << 30, 1 << 30, 7]])
def test_equal_keys_keep_their_order(dims):
    """Duplicate coordinates: values of one cell come out in input order."""
    A = _A()
    rng = np.random.default_rng(9)
    n = 9000
    cidx = np.stack([rng.integers(0, min(d, 3), n).astype(np.uint64) for d in dims])
    vals = np.arange(1, n + 1, dtype=np.float64)
    g = A.AltoTensor(dims, cidx, vals, nprtn=4)
    s = g.export()
    c = g.delinearize()
    assert np.array_equal(np.sort(s["vals"]), vals)
    at = (s["vals"] - 1).astype(np.int64)
    assert np.array_equal(c, cidx[:, at])
    same = (c[:, 1:] == c[:, :-1]).all(0)
    assert (np.diff(at)[same] > 0).all()
    for m in range(len(dims)):
        o = g.oidx(m).astype(np.int64)
        r = c[m][o].astype(np.int64)
        assert (np.diff(r) >= 0).all() and (np.diff(o)[np.diff(r) == 0] > 0).all()


@pytest.mark.parametrize("nprtn", [1, 7, 16, 999, 5000])
def test_intervals_of_many_partitions(nprtn):
    """More partitions than nonzeros included (empty ones)."""
    dims = [300, 200, 100]
    cidx, vals = uniform_tensor(dims, 4000, 2)
    _check(dims, cidx, vals, 1, nprtn)


def test_coordinate_outside_is_refused():
    A = _A()
    cidx, vals = uniform_tensor([30, 20, 10], 500, 1)
    cidx[1, 123] = 20
    with pytest.raises(A.AltoError):
        A.AltoTensor([30, 20, 10], cidx, vals)
