"""Runs a piece of Python against libsplashtank_hip.so on a HIP runtime of host
memory (tests/c/host_hip.hip): no kernel runs, and `launches()` tells what the
host code would have launched.  In a process of its own, as the library's HIP
calls are bound once."""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes, re
import numpy as np
hip = ctypes.CDLL("tests/c/libhost_hip.so", mode=ctypes.RTLD_GLOBAL)
hip.host_hip_log.restype = ctypes.c_char_p
hip.host_hip_live.restype = ctypes.c_int64
hip.host_hip_set.argtypes = [ctypes.c_char_p, ctypes.c_int]
from splashtank_amd import capi, scenes
from tests.helpers import opts_for

def log():
    text = hip.host_hip_log().decode()
    hip.host_hip_clear()
    return text.splitlines()

def launches():
    '''[(launch / coop / refused, kernel, workgroups, threads)] since the last call'''
    out = []
    for line in log():
        p = line.split()
        if p[0] in ("launch", "coop", "refused"):
            m = re.match(r"_Z(\\d+)", p[1])  # the name's length, then the name
            out.append((p[0], p[1][m.end():m.end() + int(m.group(1))], int(p[2]), int(p[3])))
    return out
"""


def run(code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code)], cwd=ROOT, text=True, capture_output=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
