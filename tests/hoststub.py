"""libshockx.so's host code on the CPU, over the stand-in runtime of hip_stub.cpp."""
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, json, sys
stub = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
stub.stub_pinned.restype = ctypes.c_long
import numpy as np
from shock_amd import shockx

def case(n, **kw):
    c = shockx.Case(dims=2 if n[2] == 1 else 3, n=n, **kw)
    c.upload_metric([np.full(c.shape, float(m in (0, 4, 8, 9))) for m in range(10)])
    c.upload_state([np.ones(c.shape)] * 5)
    return c
"""


def build(tmp):
    out = os.path.join(str(tmp), "libhip_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "hip_stub.cpp"),
                    "-ldl", "-pthread"], check=True)
    return out


def run(stub, body):
    """body (Python source) in a process of its own, after PRELUDE; what it assigns to `result`."""
    src = PRELUDE.format(stub=stub) + body + "\nprint('RESULT ' + json.dumps(result), flush=True)\n"
    env = dict(os.environ, PYTHONPATH=os.path.dirname(HERE))
    p = subprocess.run([sys.executable, "-c", src], env=env, capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stderr[-3000:]
    return json.loads([l for l in p.stdout.splitlines() if l.startswith("RESULT ")][-1][7:])
