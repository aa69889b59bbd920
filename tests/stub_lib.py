"""Runs a piece of Python in a process whose HIP runtime is tests/hip_stub.c:
no device, no kernels, but the engine's host code, its streams and its
allocations.  The piece finds `ag`, `np`, `cases`, `state(name)` and the stub's
functions (`stub`) in place and prints what the test looks at."""
from __future__ import annotations

import functools
import os
import subprocess
import sys
import tempfile
import textwrap

import autogrid_amd

HERE = os.path.dirname(os.path.abspath(__file__))
SYMBOLS = {"hip_4.2": "*;", "hip_4.3": "hipStreamBeginCapture; hipStreamEndCapture; hipGraphDestroy; "
                                       "hipGraphExecDestroy; hipGraphInstantiate; hipGraphLaunch;"}

PRELUDE = """
import ctypes as C, os, sys, tempfile, dataclasses
sys.path[:0] = [{root!r}, {here!r}]
import numpy as np
import autogrid_amd as ag
import cases
stub = C.CDLL("libamdhip64.so.7")
for f in ("stub_pending", "stub_mallocs", "stub_largest", "stub_launches", "stub_launch_stream", "stub_malloc_size"):
    getattr(stub, f).restype = C.c_longlong
stub.stub_launch_name.restype = C.c_char_p
for f in ("stub_fail_from", "stub_fail_above", "stub_launch_stream", "stub_launch_name", "stub_malloc_size"):
    getattr(stub, f).argtypes = [C.c_longlong]


def state(name="small"):
    d = tempfile.mkdtemp()
    gpf = cases.materialize(name, d)
    cwd = os.getcwd()
    os.chdir(d)
    try:
        return ag.Job(gpf).prepare().state()
    finally:
        os.chdir(cwd)


def device(nbytes):
    p = C.c_void_p()
    assert stub.hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
    return p.value


def launched(first=0):
    return [(stub.stub_launch_name(i).decode(), stub.stub_launch_stream(i)) for i in range(first, stub.stub_launches())]
"""


@functools.lru_cache(maxsize=None)
def _library() -> str:
    d = tempfile.mkdtemp(prefix="hipstub_")
    script = os.path.join(d, "versions")
    with open(script, "w") as f:
        f.write("hip_4.2 { global: *; };\nhip_4.3 { global: " + SYMBOLS["hip_4.3"] + " } hip_4.2;\n")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wl,--version-script=" + script,
                    "-Wl,-soname,libamdhip64.so.7", os.path.join(HERE, "hip_stub.c"), "-o",
                    os.path.join(d, "libamdhip64.so.7")], check=True)
    return d


def run(code: str) -> str:
    """The piece's output."""
    env = dict(os.environ, LD_LIBRARY_PATH=_library())
    text = PRELUDE.format(root=os.path.dirname(os.path.dirname(autogrid_amd.__file__)), here=HERE) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", text], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout
