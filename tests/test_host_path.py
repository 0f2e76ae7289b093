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


# out["runs"][k]: status of call() when its k-th allocation and all later ones
# fail, and what it left in flight; up to the first k that it does not reach
_FAILING = r'''
def failing(setup, call):
    runs = []
    for k in range(64):
        x = setup()
        A.check(L.alto_device_synchronize(), "sync")
        A.check(L.alto_device_trim(), "trim")
        H.host_hip_fail_from(k)
        status = call(x)
        H.host_hip_fail_from(-1)
        runs.append([status, H.host_hip_in_flight()])
        after(x)
        if status == 0:
            return runs
after = lambda x: None
'''

_CREATE = r'''
idx = np.zeros((3, 4000), np.uint64)
vals = np.ones(4000)
def create(_):
    h = C.c_void_p()
    d = np.array([70, 50, 40], np.uint64)
    st = L.alto_tensor_create(3, d.ctypes.data, 4000, A._ptr_array([r.ctypes.data for r in idx]), vals.ctypes.data,
                              0, 0, 0, 4, None, C.byref(h))
    if st == 0:
        L.alto_tensor_destroy(h)
    return st
out["runs"] = failing(lambda: None, create)
'''
_STREAMS = r'''
A.check(L.alto_tune_set(7, HOT), "hot rows")
out["runs"] = failing(lambda: tensor([70, 50, 40], 200_000), lambda t: mttkrp(t, [1] * 3, 16))
'''
_OIDX = r'''
o = np.zeros(200_000, np.uint64)
out["runs"] = failing(lambda: tensor([70, 50, 40], 200_000), lambda t: L.alto_tensor_export_oidx(t.h, 1, o.ctypes.data))
'''

_SEEDED = r'''
def seeded(t):
    h = C.c_void_p()
    st = L.alto_cpd_session_create_seeded(t.h, 16, A.PREC_BF16, 3, None, C.byref(h))
    if st == 0:
        L.alto_cpd_session_destroy(h)
    return st
out["runs"] = failing(lambda: tensor([70, 50, 40], 200_000), seeded)
'''
_HOST = r'''
dims = np.array([70, 50, 40], np.uint64)
U, lam, res = [np.ones((d, 10)) for d in dims], np.ones(10), A.AprResult()
up = A._ptr_array([u.ctypes.data for u in U])
idx, vals = [np.zeros(4000, np.uint64) for d in dims], np.ones(4000)
calls = dict(
    apr=lambda t: L.alto_cp_apr(t.h, 10, 2, 3, 1e-5, 1e-10, 1e-10, 1e-2, 0, up, lam.ctypes.data, C.byref(res), 0, None),
    coo=lambda t: L.alto_coo_mttkrp(3, dims.ctypes.data, 4000, A._ptr_array([i.ctypes.data for i in idx]),
                                    vals.ctypes.data, 0, 10, up, U[0].ctypes.data, 1, 0, None),
    kruskal=lambda t: L.alto_kruskal_normalize(3, dims.ctypes.data, 10, up, lam.ctypes.data, -1, 0, 0, None))
out["runs"] = failing(lambda: tensor([70, 50, 40], 200_000), calls["CALL"])
'''


@pytest.mark.parametrize("body", [_CREATE, _STREAMS.replace("HOT", "0"), _STREAMS.replace("HOT", "1"), _OIDX, _SEEDED,
                                  *(_HOST.replace("CALL", x) for x in ("apr", "coo", "kruskal"))],
                         ids=["create", "streams", "hot rows", "oidx", "seeded", "apr", "coo", "kruskal"])
def test_nothing_in_flight_when_an_allocation_fails(host, body):
    """A call that gives up hands its buffers back to the cache shared by all
    streams, so nothing that it enqueued may still be running."""
    runs = host(_FAILING + body)["runs"]
    assert len(runs) > 3 and runs[-1][0] == 0
    assert all(status != 0 and left == 0 for status, left in runs[:-1]), runs


# values and rank tables that kernels read: each must have been written by a
# kernel since the set-up
_WRITTEN = r'''
written, unwritten = set(), []
def watch(x):
    if "k_mode_gather" in x.name or "k_fiber_place" in x.name:
        o = x.arg(3 if "k_mode_gather" in x.name else 9, C.c_uint64 * 3)
        written.update(o[1:])
    elif "k_rank_scatter" in x.name:
        written.update((x.arg(2), x.arg(3)))
    elif "k_permute_rows" in x.name and x.arg(1) not in written:
        unwritten.append(x.name)
    elif "k_mttkrp" in x.name and x.arg(0, C.c_uint64 * 2)[1] not in written:
        unwritten.append(x.name)
seen.append(watch)
'''


@pytest.mark.parametrize("hot", [0, 1])
def test_a_failed_preparation_is_not_taken_for_a_finished_one(host, hot):
    """FP32 streams of a tensor prepared for FP64 (and, with hot rows, its rank
    tables): the call after a failed one builds what the failed one did not."""
    runs = host(_FAILING + _WRITTEN + f'''
dims = [70, 50, 40]
def setup():
    A.check(L.alto_tune_set(7, 0), "hot rows")
    t = tensor(dims, 200_000)
    A.check(mttkrp(t, dims, 16), "fp64")
    A.check(L.alto_tune_set(7, {hot}), "hot rows")
    written.clear()
    return t
def again(t):
    for m in range(3):
        A.check(mttkrp(t, dims, 16, m, A.PREC_F32), "fp32")
after = again
out["runs"] = failing(setup, lambda t: mttkrp(t, dims, 16, 0, A.PREC_F32))
out["unwritten"] = unwritten
''')
    assert len(runs["runs"]) > 3
    assert not runs["unwritten"]


@pytest.mark.parametrize("dims,bits,per", [
    ([4000, 3000], 64, 24), ([4000, 1 << 30], 128, 24),
    # fibers; the last one's coordinates take two words
    ([4000, 3000, 5000], 64, 24), ([1 << 30, 1 << 30, 1 << 30], 128, 24),
], ids=str)
def test_streams_need_no_room_for_records(host, dims, bits, per):
    """A preparation in memory that holds the streams and 24 bytes per nonzero
    succeeds, and takes the records up where there is room for them too."""
    n = 1 << 22  # (allocations are powers of two)
    words = 2 if sum((d - 1).bit_length() for d in dims) > 64 else 1
    out = host(_BOUNDS + _WRITTEN + f'''
records = []
seen.append(lambda x: records.append(x.name) if "k_records" in x.name else None)
t = tensor({dims}, {n}, lit_bits={bits})
A.check(L.alto_device_trim(), "trim")
stream = {len(dims)} * ({words} * 8 + 8) * {n}
H.host_hip_limit(H.host_hip_live() + stream + {per} * {n} + (8 << 20))
out["scarce"] = [mttkrp(t, {dims}, 2), len(records)]
H.host_hip_limit(1 << 60)
t = tensor({dims}, {n}, lit_bits={bits})
out["ample"] = [mttkrp(t, {dims}, 2), len(records)]
out["bad"] = bad
''')
    assert out["scarce"] == [0, 0] and not out["bad"]
    assert out["ample"] == [0, 1]


def test_narrow_rank_goes_back_to_its_default(host):
    """ALTO_TUNE_NARROW_RANK: -1 restores the rule per element type."""
    out = host(r'''
dims, lanes = [300, 200, 100], []
seen.append(lambda x: lanes.append(x.name) if "k_mttkrp" in x.name else None)
t = tensor(dims, 500_000)
for value in (None, 64, -1):
    if value is not None:
        A.check(L.alto_tune_set(10, value), "narrow rank")
    for prec in (A.PREC_F32, A.PREC_BF16):
        for R in (16, 24, 32, 64):
            A.check(mttkrp(t, dims, R, 0, prec), "mttkrp")
out["lanes"], out["refused"] = lanes, [L.alto_tune_set(10, v) for v in (-2, 129)]
''')
    shipped, narrow, restored = out["lanes"][:8], out["lanes"][8:16], out["lanes"][16:]
    assert len(out["lanes"]) == 24 and shipped == restored != narrow
    assert all(v != 0 for v in out["refused"])


@pytest.mark.parametrize("R,prec,nnz,kernel", [(1, 0, 20_000_000, "k_mttkrp<"), (25, 2, 20_000_000, "k_mttkrp<"),
                                               (16, 0, 20_000_000, "k_mttkrp<"), (16, 0, 10_000, "k_mttkrp16<"),
                                               (64, 2, 20_000_000, "k_mttkrp16<")])
def test_autotune_tries_each_mapping_around_its_own_rule(host, R, prec, nnz, kernel):
    """Segment lengths from a quarter to four times the length each kernel takes
    by itself are among the ones tried (the first two launches are the default's)."""
    strided = kernel == "k_mttkrp<"
    out = host(f'''
dims, tried = [3000, 2000, 1000], []
seen.append(lambda x: tried.append(x.arg(0, C.c_uint64 * 15)[14]) if "{'8k_mttkrpI' if strided else '10k_mttkrp16I'}" in x.name
            else None)
A.check(L.alto_tune_set(13, 0), "no fibers")
A.check(L.alto_tune_set(4, {0 if strided else -1}), "variant")
t = tensor(dims, {nnz})
A.check(mttkrp(t, dims, {R}, 0, {prec}), "mttkrp")
A.check(L.alto_tune_set(4, -1), "variant")
out["own"] = tried.pop()
tried.clear()
A.check(L.alto_mttkrp_autotune(t.h, {R}, {prec}, A._ptr_array([1 << 20] * 3), 1 << 20, 1, None, None), "autotune")
out["tried"] = sorted(set(tried))
''')
    window = [s for s in (16 << k for k in range(9)) if out["own"] <= 4 * s and s <= 4 * out["own"]]
    assert set(window) <= set(out["tried"]), out


@pytest.mark.parametrize("R", [3, 5, 8, 13])
def test_cp_apr_keeps_products_where_they_fit_unpadded(host, R):
    """The one-nonzero-per-lane Phi pads odd ranks and the last nonzeros in its
    product cache; where only nnz x rank doubles fit half the free memory, the
    products are kept all the same."""
    out = host(f'''
n, dims = 1_000_003, [300, 200, 100]
launched = []
seen.append(lambda x: launched.append(x.name) if "k_phi_" in x.name else None)
t = tensor(dims, n)
for key, room in (("tight", n * {R}), ("ample", (n + 64) * {R + 1}), ("none", n * {R} - 1)):
    H.host_hip_say_free(2 * 8 * room)
    launched.clear()
    t.cp_apr([np.ones((d, {R})) for d in dims], np.ones({R}), 1, 10)
    out[key] = sorted(set(launched))
''')
    # (the last template argument: 0 = no products, 1 = stored)
    assert len(out["tight"]) == 1 and "k_phi_b" in out["tight"][0] and "ELi1EEEv" in out["tight"][0]
    assert len(out["ample"]) == 1 and "k_phi_cols" in out["ample"][0] and "ELi1EEEv" in out["ample"][0]
    assert len(out["none"]) == 1 and "ELi0EEEv" in out["none"][0]


@pytest.mark.parametrize("R,prec,n,nnz,knob,segs", [
    (48, 0, 4, 100_000, 0, 16), (48, 0, 16, 100_000, 0, 32), (48, 0, 16, 200_000, 0, 64), (48, 0, 16, 3_000_000, 0, 128),
    (48, 0, 16, 100_000, 24, 24), (16, 0, 16, 100_000, 0, 8), (32, 0, 16, 100_000, 0, 16), (64, 1, 16, 200_000, 0, 32),
    (64, 2, 16, 200_000, 0, 16), (64, 0, 16, 5_000, 0, 16)])
def test_batched_segments(host, R, prec, n, nnz, knob, segs):
    """Segment lengths of a launch of many tensors: each tensor's own rule until
    the launch has more wavefronts than it needs, then longer ones."""
    out = host(f'''
dims, found, left = [300, 200, 100], [], []
def look(x):
    if "k_mttkrp16_batch" in x.name:
        a = x.arg(0, C.c_uint64 * (22 * 16 + 9))
        found.extend(a[22 * j + 14] for j in range({n}))
        # every nonzero has a lane group
        G = int(x.name.split("Li")[1].split("E")[0])
        left.extend(-(-a[22 * j + 13] // a[22 * j + 14]) * G > a[22 * j + 15] * 256 for j in range({n}))
seen.append(look)
A.check(L.alto_tune_set(1, {knob}), "segments")
ts = [tensor(dims, {nnz}) for _ in range({n})]
f = A._ptr_array([1 << 20] * 3)
st = L.alto_mttkrp_batched({n}, A._ptr_array([t.h for t in ts]), (C.c_int * {n})(*([0] * {n})), {R},
                           A._ptr_array([C.addressof(f)] * {n}), A._ptr_array([1 << 20] * {n}), {prec}, 0, None)
out.update(status=st, segs=sorted(set(found)), count=len(found), left=sum(left))
''')
    assert out == dict(status=0, segs=[segs], count=n, left=0)
