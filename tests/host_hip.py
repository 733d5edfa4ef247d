"""Runs a piece of test code in a child process on the library with the HIP runtime replaced by
host_hip.c (no GPU: memory calls and kernel launches are recorded, allocations can fail)."""
import os
import shutil
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "wormlike-chain-triblock_amd")

# loaded under the runtime's own name, so that the library's dependency on it is met by this one
PRELUDE = """
import ctypes, sys
import numpy as np
H = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
H.host_hip_alloc_bytes.restype = ctypes.c_longlong
H.host_hip_kernel.restype = ctypes.c_char_p
sys.path.insert(0, {pkg!r})
import wlc_mde as W
W.load()
def launches():
    return [H.host_hip_kernel(i).decode() for i in range(H.host_hip_launches())]
"""


def build(folder):
    so = os.path.join(str(folder), "libhosthip.so")
    cmd = [shutil.which("gcc") or "gcc", "-O1", "-shared", "-fPIC", "-Wl,-soname,libamdhip64.so.7",
           "-Wl,--version-script," + os.path.join(HERE, "host_hip.map"),
           os.path.join(HERE, "host_hip.c"), "-o", so]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return so


def run(so, code, env=None):
    """Output lines of `code` (after PRELUDE) in a child process."""
    r = subprocess.run([sys.executable, "-c", PRELUDE.format(so=so, pkg=PKG) + textwrap.dedent(code)],
                       capture_output=True, text=True, timeout=120, env=dict(os.environ, **(env or {})))
    assert r.returncode == 0, f"status {r.returncode}\n{r.stdout[-2000:]}\n{r.stderr[-4000:]}"
    return r.stdout.splitlines()
