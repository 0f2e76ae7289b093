"""Mode streams of one tensor sorted by keys of different widths: 32-bit keys
with an odd number of digit passes next to 64-bit ones, in every order of the
modes, and two fiber tiers of different widths inside one mode."""
import itertools

import numpy as np
import pytest

from tests._tensors import mttkrp_numpy, zipf_tensor

pytestmark = pytest.mark.gpu

CHUNK_LOG2, FIBERS, FIBER_CHUNK_LOG2, FIBER_MIN_NNZ = 2, 13, 15, 16


def _A():
    import alto_amd
    return alto_amd


@pytest.fixture
def tune():
    A = _A()
    yield lambda p, v: A.check(A.lib().alto_tune_set(p, v), "tune_set")
    for p, v in ((CHUNK_LOG2, 0), (FIBERS, 1), (FIBER_CHUNK_LOG2, 30), (FIBER_MIN_NNZ, 4 << 20)):
        A.check(A.lib().alto_tune_set(p, v), "tune_set")


@pytest.mark.parametrize("dims,nnz,knobs", [
    # row + fiber row: 24 bits (3 passes) for the small modes, 34 for the large
    *((d, 300_000, {FIBER_MIN_NNZ: 0}) for d in itertools.permutations([3000, 3_000_000, 4000])),
    # three modes of 22 bits, one of 33
    *((d, 200_000, {FIBER_MIN_NNZ: 0}) for d in itertools.permutations([900, 4000, 3000, 6_000_000])
      if d.index(6_000_000) in (1, 3)),
    # mode 0: 22 bits in the first tier, 33 in the second
    *((d, 300_000, {FIBER_MIN_NNZ: 0, FIBERS: 2, FIBER_CHUNK_LOG2: 10})
      for d in itertools.permutations([200, 30, 60_000])),
    # chunk + row: 22 bits, then 33
    *((d, 2_200_000, {FIBERS: 0, CHUNK_LOG2: 10}) for d in ([900, 1 << 21, 700], [1 << 21, 900, 700])),
], ids=lambda x: "x".join(map(str, x)) if isinstance(x, (list, tuple)) else None)
def test_mixed_key_widths(tune, dims, nnz, knobs):
    A = _A()
    for p, v in knobs.items():
        tune(p, v)
    cidx, vals = zipf_tensor(list(dims), nnz, 5, s=1.1)
    g = A.AltoTensor(list(dims), cidx, vals)
    rng = np.random.default_rng(1)
    U = [rng.random((d, 2)) for d in dims]
    for m in range(len(dims)):
        want = mttkrp_numpy(cidx, vals, U, m)
        # positive terms: N + 1 roundings on each one's way, at most nnz additions
        bound = want * 2.0 ** -52 * (len(dims) + 1 + len(vals))
        assert (np.abs(g.mttkrp(m, U) - want) <= bound).all(), m
