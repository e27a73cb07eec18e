"""Runs a piece of Python in a process of its own in which hip_calls.c stands
between libsevc.so and the HIP runtime."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "se-grain-growth-gpu_amd")

HEAD = """
import ctypes as C, sys
hip = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
hip.calls_what.restype = C.c_void_p
sys.path[:0] = [{pkg!r}, {here!r}]
import numpy as np
import sevc

def calls():
    return [(chr(hip.calls_kind(k)), hip.calls_what(k)) for k in range(hip.calls_count())]
"""


def run(body, tmp_path, timeout=90):
    """The child's output; its failure is the test's."""
    shim = str(tmp_path / "hip_calls.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", shim, os.path.join(HERE, "hip_calls.c"), "-ldl"], check=True)
    src = HEAD.format(shim=shim, pkg=PKG, here=HERE) + body
    r = subprocess.run([sys.executable, "-u", "-c", src], capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
