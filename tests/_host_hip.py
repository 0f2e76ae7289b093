"""The library on tests/_host_hip.c, in a process of its own: run(body) runs
the Python text `body` there, with `A` (the package), `H` (the runtime's side
for tests), `launches` (every launch: kernel name, grid, arguments through
arg(k, type)) and tensor(dims, nnz) at hand, and returns what it put into
`out`."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_PRELUDE = r'''
import ctypes as C, json, sys
sys.path.insert(0, sys.argv[2])
H = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # ahead of the real runtime for every later library
H.host_hip_room.restype = H.host_hip_live.restype = C.c_uint64
H.host_hip_room.argtypes = H.host_hip_limit.argtypes = H.host_hip_say_free.argtypes = [C.c_uint64]
import numpy as np
import alto_amd as A
L = A.lib()

class Launch:
    def __init__(self, name, grid, args):
        self.name, self.grid, self.args = name, grid, args
    def arg(self, k, typ=C.c_uint64):
        return C.cast(self.args[k], C.POINTER(typ))[0]

launches, seen = [], []
def _on_launch(name, grid, block, args):
    x = Launch(name.decode(), grid, args)
    launches.append((x.name, grid))
    for f in seen:
        f(x)
_cb = C.CFUNCTYPE(None, C.c_char_p, C.c_uint32, C.c_uint32, C.POINTER(C.c_void_p))(_on_launch)
H.host_hip_on_launch(_cb)

class Ptr:
    """a device array that is only an address"""
    def __init__(self, shape=(1, 1)):
        self.ptr, self.shape = 1 << 20, shape
def tensor(dims, nnz, **kw):
    return A.AltoTensor.from_device(dims, [1 << 20] * len(dims), 1 << 20, nnz, **kw)
def mttkrp(t, dims, R, mode=0, prec=A.PREC_F64):
    return L.alto_mttkrp(t.h, mode, R, A._ptr_array([1 << 20] * len(dims)), 1 << 20, prec, 0, None)
out = {}
'''


def build(folder):
    so = os.path.join(str(folder), "libhost_hip.so")
    src = os.path.join(ROOT, "tests", "_host_hip.c")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, src], check=True, capture_output=True, text=True)
    return so


def run(so, body):
    r = subprocess.run([sys.executable, "-c", _PRELUDE + body + "\nprint(json.dumps(out))", so, ROOT],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads(r.stdout.splitlines()[-1])
