"""Runs a piece of Python against the library on fake_hip.cpp's runtime: two
devices, no GPU.  In a process of its own, where the fake's symbols come before
libamdhip64's."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
_PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(%r, mode=C.RTLD_GLOBAL)
fake.fake_fail_rho.argtypes = [C.c_double]
fake.fake_capacity.argtypes = [C.c_size_t]
fake.fake_fail_launch.argtypes = [C.c_char_p, C.c_int]
for f in (fake.fake_used, fake.fake_peak):
    f.restype = C.c_size_t
fake.fake_count.restype = fake.fake_launches.restype = C.c_long
MALLOCS, FREES, WAITS, FOREIGN = range(4)
sys.path.insert(0, %r)
import numpy as np
import phylocsf_amd as P
from phylocsf_amd import _lib
L = _lib.lib()


def launches(name):
    return fake.fake_launches(name.encode())


def batch(model, regions, cols):
    codes = np.zeros((regions * cols, model.tree.nl), np.uint8)
    return P.Batch(model, codes, np.arange(regions + 1) * cols)
"""


@pytest.fixture(scope="session")
def on_fake(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", lib, os.path.join(HERE, "fake_hip.cpp")], check=True)

    def run(body, env=None):
        code = _PRELUDE % (lib, ROOT) + textwrap.dedent(body)
        r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, **(env or {})),
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
        assert r.returncode == 0, r.stdout[-4000:]

    return run
