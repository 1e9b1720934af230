"""CPU check of gl::join_halves (csrc/gl_lazy.hpp, host form) against 128-bit
integer arithmetic (tests/native/join_check.cpp), to the edges of its range."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = shutil.which("clang++") or shutil.which("amdclang++") or "/opt/rocm/llvm/bin/clang++"


@pytest.mark.skipif(not os.path.exists(CLANG) and shutil.which(CLANG) is None, reason="clang++ not available")
@pytest.mark.parametrize("opt", ["-O0", "-O2"])
def test_halves_match_128bit_reference(tmp_path, opt):
    exe = tmp_path / "join_check"
    subprocess.run([CLANG, opt, "-std=c++17", "-o", str(exe), os.path.join(HERE, "native", "join_check.cpp")],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip().endswith("ok"), out.stdout + out.stderr
