"""Runs host code of libemerge_amd.so on the CPU against tests/hip_recorder.c (no GPU, no HIP runtime):
`run(snippet, tmp_path)` executes a snippet in its own process with `L` (the library), `rec` (the recorder)
and `log()` (the calls since the last look), and returns what it printed as JSON lines."""
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PROLOGUE = """
import ctypes, json, sys
import numpy as np
rec = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
rec.rec_log.restype = ctypes.c_char_p
rec.rec_used.restype = ctypes.c_size_t
rec.rec_budget.argtypes = rec.rec_host_block.argtypes = [ctypes.c_size_t]
ctypes.CDLL("libstdc++.so.6", mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, {root!r})
from emerge_amd import _lib
L = _lib.load()
P = ctypes.c_void_p
def at(a): return P(a.ctypes.data)
def out(v): print(json.dumps(v), flush=True)
def log():
    lines = rec.rec_log().decode().splitlines()
    rec.rec_clear()
    return lines
"""


def run(snippet, tmp_path, env=None):
    stub = os.path.join(tmp_path, "libhip_recorder.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-fexceptions", "-o", stub, os.path.join(HERE, "hip_recorder.c"), "-ldl"], check=True)
    code = PROLOGUE.format(stub=stub, root=ROOT) + snippet
    got = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env={**os.environ, **(env or {})}, capture_output=True,
                         text=True, timeout=120)
    assert got.returncode == 0, got.stderr[-2000:]
    return [json.loads(line) for line in got.stdout.splitlines() if line.startswith(("{", "["))]
