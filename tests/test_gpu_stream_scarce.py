"""Mode streams gathered from the keys and values, as where the memory for
records is not there: a process of its own whose large allocations are
refused once the tensor is built."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# hipMalloc that refuses more than `most` bytes and else calls the runtime's
_REFUSING = r'''
#include <stddef.h>
typedef int (*malloc_fn)(void**, size_t);
malloc_fn runtime_malloc;
size_t most = (size_t)-1;
int refused;
int hipMalloc(void** p, size_t n)
{
    if (n > most) {
        ++refused;
        return 2;
    }
    return runtime_malloc(p, n);
}
'''
_BODY = r'''
import ctypes as C, json, sys
sys.path.insert(0, sys.argv[2])
H = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # ahead of the runtime
import importlib.util, os
torch = importlib.util.find_spec("torch")
path = os.path.join(list(torch.submodule_search_locations)[0], "lib", "libamdhip64.so")
real = C.CDLL(path, mode=C.RTLD_GLOBAL)
C.c_void_p.in_dll(H, "runtime_malloc").value = C.cast(real.hipMalloc, C.c_void_p).value
most, refused = C.c_size_t.in_dll(H, "most"), C.c_int.in_dll(H, "refused")
import numpy as np
import alto_amd as A
from tests._tensors import mttkrp_numpy, zipf_tensor
L = A.lib()
out = []
A.check(L.alto_tune_set(16, 0), "fibers of small tensors")
for dims, bits in (([300, 4000, 500], 64), ([300, 4000, 500], 128), ([70, 1 << 20, 1 << 21, 1 << 22], 128)):
    n = 60_000
    cidx, vals = zipf_tensor(dims, n, 3, s=1.1)
    U = [np.random.default_rng(m).random((d, 2)) for m, d in enumerate(dims)]
    want = [mttkrp_numpy(cidx, vals, U, m) for m in range(len(dims))]
    for fibers in (0, 1, 2):
        A.check(L.alto_tune_set(13, fibers), "fibers")
        for prec in (A.PREC_F64, A.PREC_F32):
            V = U if prec == A.PREC_F64 else [u.astype(np.float32).astype(np.float64) for u in U]
            w = want if prec == A.PREC_F64 else [mttkrp_numpy(cidx, vals, V, m) for m in range(len(dims))]
            g = A.AltoTensor(dims, cidx, vals, lit_bits=bits)
            dev = [A.DeviceArray.from_numpy(v.astype(np.float64 if prec == A.PREC_F64 else np.float32)) for v in V]
            o = A.DeviceArray((dims[0], 2), np.float64)
            A.check(L.alto_device_trim(), "trim")
            words = 2 if sum((d - 1).bit_length() for d in dims) > 64 else 1
            most.value = n * 8 * (words + 1) - 1  # the records alone are larger
            before = refused.value
            g.mttkrp_device(0, dev, o, prec)
            most.value = 2 ** 64 - 1
            eps = 2.0 ** -52 if prec == A.PREC_F64 else 2.0 ** -23
            bad = 0
            for m in range(len(dims)):
                got = g.mttkrp(m, V, prec)
                # positive terms: value, factors and products (N + 2) rounded on
                # each one's way, at most n additions (32-bit runs: 4096)
                bound = w[m] * eps * (len(dims) + 2 + (n if prec == A.PREC_F64 else 4096))
                bad += int((np.abs(got - w[m]) > bound).sum())
            out.append([refused.value - before, bad])
print(json.dumps(out))
'''


def test_streams_without_records(tmp_path):
    src, so = tmp_path / "refusing.c", tmp_path / "librefusing.so"
    src.write_text(_REFUSING)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", _BODY, str(so), ROOT], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout.splitlines()[-1])
    assert len(out) == 18
    assert all(refused >= 1 and bad == 0 for refused, bad in out), out
