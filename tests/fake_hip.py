"""Runs a snippet against the library's host code on the CPU, with
tests/native/fake_hip.c preloaded in place of the HIP runtime: `lib` is the
library with its C signatures, `fake` the recorder, `launches()` what was
launched since the last reset as (kernel, grid, block), `ctx` a context."""
import json
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(os.path.dirname(HERE), "era-boojum-cuda_amd")

PRELUDE = """
import ctypes, json, re, sys
sys.path.insert(0, {pkg!r})
from boojum_cuda_amd import _lib
lib = _lib.lib()
fake = ctypes.CDLL({so!r})
fake.fake_kernel.restype = ctypes.c_char_p
fake.fake_arg_word.restype = ctypes.c_uint64
ctx = ctypes.c_void_p()
assert lib.bc_context_create(12, 12, ctypes.byref(ctx)) == 0
def launches():
    out = []
    for i in range(fake.fake_launches()):
        s = (ctypes.c_uint32 * 6)()
        fake.fake_shape(i, s)
        out.append((fake.fake_kernel(i).decode(), list(s[:3]), list(s[3:])))
    return out
def kernels():
    return [re.search(r"(ntt|bary|poseidon)_[a-z0-9_]*_kernel", k).group(0) for k, _, _ in launches()]
def done(value):
    print("RESULT", json.dumps(value))
fake.fake_reset()
"""


def run(tmp_path, code):
    """The value the snippet passes to done()."""
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    so = os.path.join(str(tmp_path), "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "native", "fake_hip.c")], check=True)
    env = dict(os.environ, LD_PRELOAD=so)
    out = subprocess.run([sys.executable, "-c", PRELUDE.format(pkg=PKG, so=so) + textwrap.dedent(code)], env=env,
                         capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    return json.loads(out.stdout.split("RESULT ", 1)[1])
