"""The library's host code without a GPU (tests/_host_hip.py): sizes of the
buffers that launches are given, what is in flight when a call gives up, which
kernels a call takes."""
import itertools

import pytest

from tests import _host_hip


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = _host_hip.build(tmp_path_factory.mktemp("host_hip"))
    return lambda body: _host_hip.run(so, body)


# every buffer of keys and positions that a sorting kernel is given holds what
# the kernel reads or writes
_BOUNDS = r'''
import re
bad, widths = [], set()
def check(x):
    m = re.search(r"k_(stream_key|rs_hist|rs_scatter|fiber_count|fiber_place)I(j|m|N\w*?6Key128E)", x.name)
    if not m:
        return
    kind, size = m.group(1), {"j": 4, "m": 8}.get(m.group(2), 16)
    n = x.arg({"stream_key": 5, "rs_hist": 1, "rs_scatter": 2, "fiber_count": 1, "fiber_place": 2}[kind])
    if kind == "stream_key":
        widths.add(size)
    keys, pos = {"stream_key": ([7], [6, 8]), "rs_hist": ([0], []), "rs_scatter": ([0, 8], [1, 9]),
                 "fiber_count": ([0], []), "fiber_place": ([0], [1])}[kind]
    for args, each in ((keys, size), (pos, 4)):
        for k in args:
            p = x.arg(k)
            if p and H.host_hip_room(p) < n * each:
                bad.append([kind, k, n * each, H.host_hip_room(p)])
seen.append(check)
'''


@pytest.mark.parametrize("dims,nnz,knobs", [
    *((list(d), 5_000_000, {}) for d in itertools.permutations([3000, 3_000_000, 4000])),
    ([20000, 20_000_000, 300], 4_500_000, {}),
    *((list(d), 20_000_000, {}) for d in itertools.permutations([900, 4000, 3000, 6_000_000])),
    ([8192, 200_000_000], 20_000_000, {}),
    ([200_000_000, 8192], 20_000_000, {}),
    ([1000, 300, 1 << 24], 6_000_000, {"FIBERS": 2}),
    ([1 << 24, 1000, 300], 6_000_000, {"FIBERS": 2}),
    ([900, 1 << 24, 700], 5_000_000, {"FIBERS": 0, "CHUNK_LOG2": 10}),
], ids=str)
def test_stream_sort_buffers_hold_their_keys(host, dims, nnz, knobs):
    """Modes whose stream keys are of different widths (32 and 64 bits), with an
    odd number of sort passes for the narrower ones."""
    num = {"FIBERS": 13, "CHUNK_LOG2": 2}
    out = host(_BOUNDS + f'''
for p, v in {[(num[k], v) for k, v in knobs.items()]}:
    A.check(L.alto_tune_set(p, v), "tune")
t = tensor({dims}, {nnz})
out.update(status=mttkrp(t, {dims}, 2), widths=sorted(widths), bad=bad[:4])
''')
    assert out["status"] == 0 and out["widths"] == [4, 8]
    assert not out["bad"]
