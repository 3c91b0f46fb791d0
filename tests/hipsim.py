"""Runs a snippet on libflutas_amd.so over the host stand-in for the HIP runtime
(hipsim.c) in a process of its own.  The snippet finds `api`, `np`, `C`, `sim`
(the stand-in), and the helpers below."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
sim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
from flutas_amd import api
sim.sim_limit.argtypes = [C.c_size_t]
sim.sim_used.restype = sim.sim_peak.restype = C.c_size_t
sim.sim_count.restype = C.c_longlong
sim.sim_launch.restype = C.c_char_p
UNLIMITED = 1 << 62

def launches():
    # (kernel, grid, block, LDS bytes, stream) of every launch since sim_reset
    out = []
    for i in range(sim.sim_launches()):
        gb, lds, s = (C.c_uint * 6)(), C.c_size_t(), C.c_void_p()
        name = sim.sim_launch(i, gb, C.byref(lds), C.byref(s)).decode()
        out.append((name, tuple(gb[:3]), tuple(gb[3:]), lds.value, s.value))
    return out

def plan(ng, cbc="PPDDNN", **kw):
    dz = np.full(ng[2] + 2, float(ng[2]))
    return api.PoissonPlan(ng, tuple(float(n) for n in ng), dz, dz, cbc, **kw)

def field(ng, dtype=np.float64):
    return api.DeviceArray(tuple(n + 2 for n in ng), dtype)

def solve32(p, d):
    return api.lib.flutas_psolve_solve_f32(C.c_void_p(p._h), C.cast(C.c_void_p(d.ptr), C.POINTER(C.c_float)))
"""


def run(snippet, tmp_path):
    lib = os.path.join(str(tmp_path), "libhipsim.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-I/opt/rocm/include",
                    os.path.join(HERE, "hipsim.c"), "-o", lib], check=True)
    r = subprocess.run([sys.executable, "-c", PRELUDE + snippet, lib, ROOT], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout
