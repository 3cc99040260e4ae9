"""Runs a program over the library with the HIP runtime's host stand-in
(tests/host/hip_host.cpp): the real host code of libocr.so, kernels logged
instead of run."""
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, os, sys
import numpy as np
H = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
H.host_log.restype = C.c_char_p
H.host_device_bytes.restype = C.c_size_t
H.host_limit_device.argtypes = [C.c_size_t]
for f in ("host_hold", "host_capture"):
    getattr(H, f).argtypes = [C.c_void_p, C.c_int]
H.host_stream_id.argtypes = [C.c_void_p]
H.hipStreamCreateWithFlags.argtypes = [C.POINTER(C.c_void_p), C.c_uint]
H.hipStreamDestroy.argtypes = [C.c_void_p]
from openclrenderer_amd import abi, runtime, scenes

def stream():
    s = C.c_void_p()
    H.hipStreamCreateWithFlags(C.byref(s), 1)
    return s

def log():
    lines = [l.split() for l in H.host_log().decode().splitlines()]
    H.host_clear()
    return lines

def kernels(lines):
    return [l[1] for l in lines if l[0] == "launch"]
"""


def run(tmp_path, code):
    """Runs `code` after the prelude; returns what it printed."""
    from openclrenderer_amd import build as b
    if not os.path.exists(b.LIB):
        b.build()
    lib = str(tmp_path / "libhip_host.so")
    if not os.path.exists(lib):
        subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        os.path.join(HERE, "host", "hip_host.cpp"), "-o", lib], check=True)
    env = dict(os.environ, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), lib], capture_output=True, text=True, env=env,
                       cwd=ROOT, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    return r.stdout
