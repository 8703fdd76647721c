"""The library's host code on a machine without a GPU: run(tmp_path, code)
builds fake_hip/fake_hip.c, a stand-in for the HIP runtime that runs no kernel,
and executes `code` in a process of its own with these names:

    F    the stand-in (fake_limit, fake_used, hipSetDevice, ...)
    L    libatsim.so on it, with the argument types of _lib
    log()   the allocations, streams, events and launches since the last log(),
            as (what, demangled kernel name or "-", device, grid, threads)
    ctx(device)  a context; ptr(nbytes, ctx) device memory of one
    sim(c, N, ...)  a simulation (see the code below)

The code prints what it asserts; a failed assertion fails the test."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_HEAD = r'''
import ctypes as C, subprocess, sys
import numpy as np
sys.path.insert(0, %(root)r)
F = C.CDLL(%(fake)r, mode=C.RTLD_GLOBAL)
F.fake_log.restype = C.c_char_p
F.fake_used.restype = C.c_size_t
F.fake_limit.argtypes = [C.c_size_t]
from atmosphericturbulencesimul_amd import _lib
L = _lib.lib()
OK, EINVAL, EHIP, ENOMEM, EUNSUPPORTED = 0, -1, -2, -3, -4
_names = {}

def log():
    rows = [l.split() for l in F.fake_log().decode().splitlines()]
    F.fake_reset()
    new = sorted({r[1] for r in rows if r[1] not in _names and r[1] != "-"})
    if new:
        out = subprocess.run(["c++filt"] + new, capture_output=True, text=True, check=True).stdout.splitlines()
        for a, b in zip(new, out):
            _names[a] = b.replace("void ", "").replace("atsim::", "").split("(")[0]
    return [(r[0], _names.get(r[1], r[1]), int(r[2]), tuple(map(int, r[3:6])), int(r[6])) for r in rows]

def kernels():
    return [r[1] for r in log() if r[0] == "launch"]

def ctx(device=0):
    h = C.c_void_p()
    assert L.atsim_ctx_create(device, C.byref(h)) == OK
    return h

def err(c):
    return L.atsim_error(c).decode()

def ptr(nbytes, c):
    p = C.c_void_p()
    assert L.atsim_malloc(c, C.byref(p), nbytes) == OK, err(c)
    return p

def tune(c, **keys):
    for k, v in keys.items():
        assert L.atsim_set_tuning(c, k.encode(), v) == OK, err(c)

def sim_try(c, N, sli, W=2, D=1, M=None, factored=True, rule=1):
    """(return code, simulation): layers in the super-layers sli"""
    Lc, S = len(sli), max(sli) + 1
    d = _lib.SimDesc()
    lam = np.linspace(0.6e-6, 2.0e-6, W)
    a = dict(slayer_alt=np.arange(S) * 4000.0, lambda_=lam,
             scoeff=np.array([[0.5e-6 / m * (1.0 if factored else 1.0 + 1e-3 * l * w) for l in range(Lc)]
                              for w, m in enumerate(lam)]),
             xpos0=np.zeros((D, Lc)), ypos0=np.zeros((D, Lc)), vx=np.ones(Lc), vy=np.ones(Lc))
    d.N = d.Nout = N
    d.M, d.L, d.W, d.D = M or N, Lc, W, D
    d.dx, d.dt, d.zangle, d.bicubic, d.fresnel, d.amplitude = 0.02, 0.001, 0.0, 1, 1, 1
    keep = [np.ascontiguousarray(v, np.float64) for v in a.values()]
    for k, v in zip(a, keep):
        setattr(d, k, v.ctypes.data_as(C.POINTER(C.c_double)))
    s8 = np.array(sli, np.int64)
    uw = np.full(W, rule, np.int32)
    d.super_layer_index = s8.ctypes.data_as(C.POINTER(C.c_long))
    d.unwrap_mode = uw.ctypes.data_as(C.POINTER(C.c_int))
    h = C.c_void_p()
    return L.atsim_sim_create(c, C.byref(d), C.byref(h)), h

def sim(c, *a, **k):
    rc, h = sim_try(c, *a, **k)
    assert rc == OK, err(c)
    return h
'''


def run(tmp_path, code):
    gcc = shutil.which("gcc")
    if gcc is None or shutil.which("c++filt") is None:
        pytest.skip("gcc not available")
    fake = tmp_path / "libfakehip.so"
    src = os.path.join(ROOT, "tests", "fake_hip", "fake_hip.c")
    b = subprocess.run([gcc, "-std=gnu11", "-O1", "-Wall", "-shared", "-fPIC", "-o", str(fake), src],
                       capture_output=True, text=True)
    assert b.returncode == 0, b.stderr[-2000:]
    r = subprocess.run([sys.executable, "-c", _HEAD % dict(root=ROOT, fake=str(fake)) + code], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, (r.stdout + r.stderr)[-3000:]
    return r.stdout
