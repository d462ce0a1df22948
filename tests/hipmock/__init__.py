"""Runs a piece of Python in a child process in which libsssi.so's HIP calls go
to the test double hipmock.cpp: host paths (what is allocated, copied and
launched, and what happens when an allocation fails) without a GPU.  Kernels do
not run there, so results are zeros; `M` is the double's steering interface."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
LIB = os.path.join(HERE, "_build", "libhipmock.so")

_HEAD = f"""
import ctypes
M = ctypes.CDLL({LIB!r}, mode=ctypes.RTLD_GLOBAL)
for f in ("hipmock_mallocs", "hipmock_host_mallocs", "hipmock_count", "hipmock_arg",
          "hipmock_new_left"):
    getattr(M, f).restype = ctypes.c_long
for f in ("hipmock_fail_malloc", "hipmock_sync_us", "hipmock_copy_limit",
          "hipmock_fail_new"):
    getattr(M, f).argtypes = [ctypes.c_long]
M.hipmock_size.restype = ctypes.c_size_t
M.hipmock_mem_free.argtypes = [ctypes.c_size_t]
def watch(name, *sizes):
    M.hipmock_watch(name.encode(), (ctypes.c_size_t * len(sizes))(*sizes), len(sizes))
def arg(k, a, ctype):
    out = ctype()
    assert M.hipmock_arg(ctypes.c_long(k), a, ctypes.byref(out)) == ctypes.sizeof(out)
    return out
def count(name):
    return M.hipmock_count(name.encode())
def dims(name, k=0):
    d = (ctypes.c_uint * 6)()
    assert M.hipmock_dims(name.encode(), ctypes.c_long(k), d) == 0
    return tuple(d)
import numpy as np
import sssi_amd
from sssi_amd import synth
"""


def build():
    src = os.path.join(HERE, "hipmock.cpp")
    if os.path.exists(LIB) and os.path.getmtime(LIB) > os.path.getmtime(src):
        return
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", LIB, src, "-lpthread"], check=True)


def run(code, timeout=120, **env):
    """Run `code` in a child; its standard output.  Fails with the child."""
    build()
    r = subprocess.run([sys.executable, "-c", _HEAD + code], capture_output=True, text=True,
                       timeout=timeout, cwd=ROOT, env=dict(os.environ, **env))
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-2000:]}\n{r.stderr[-3000:]}"
    return r.stdout
