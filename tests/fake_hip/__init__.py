"""libemgpu.so's host logic without a GPU: a child process loads a stand-in for
the HIP runtime (fake_hip.cpp) before the library and runs a test's code there,
with `fake` (the stand-in's own entry points) and `emg` at hand."""
import functools
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_log.restype = ctypes.c_char_p
for f in (fake.fake_used, fake.fake_peak):
    f.restype = ctypes.c_size_t
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_fail_in.argtypes = [ctypes.c_long] * 2
import numpy as np
import pytest
from ctca_amd import emg

def launches(f, *a):
    "what f launches"
    fake.fake_log_clear()
    f(*a)
    return fake.fake_log().decode().split("\\n")[:-1]

def records(total, n, pid=False):
    r = np.zeros(total, dtype=emg.PARTICLE)
    for c, m in zip("xyz", n):
        r[c] = np.arange(total) % m + 0.5
    if pid:
        r["pid"] = np.arange(total)
    return r
"""


@functools.lru_cache(None)
def library(folder):
    so = os.path.join(folder, "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    os.path.join(HERE, "fake_hip.cpp"), "-o", so],
                   check=True, capture_output=True, text=True)
    return so


def run(tmp_path, code):
    """Run `code` in a child process; the test fails where it does."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    so = library(str(tmp_path.parent))      # one for the session
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), so], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
    return r.stdout
