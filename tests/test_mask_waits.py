"""Wait states in the compiled kernels (gfx950; compiled and disassembled on the
CPU): a lane mask that a vector instruction writes may be read as a carry or a
select two instructions later at the earliest, and so may a register by a
lane-rotating (DPP) operand.  Inside asm blocks and across them nobody but the
source takes care of that."""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "era-boojum-cuda_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
CARRY = ("v_mad_u64_u32", "v_mad_i64_i32", "v_add_co", "v_sub_co", "v_addc_co", "v_subb_co", "v_subrev_co",
         "v_subbrev_co")


def operands(text):
    """Comma-separated operands, each without trailing modifiers."""
    return [o.split()[0] for o in re.findall(r"(?:[^,\[]|\[[^\]]*\])+", text) if o.split()]


def registers(operand):
    if operand == "vcc":
        return ["vcc"]
    m = re.fullmatch(r"-?\|?([sv])(?:\[(\d+):(\d+)\]|(\d+))\|?", operand)
    if not m:
        return []
    lo = int(m[2] or m[4])
    return [f"{m[1]}{i}" for i in range(lo, int(m[3] or m[4]) + 1)]


def close_reads(lines):
    """(earlier instruction, reading instruction) with less than two wait
    states between, in program order."""
    written, at, bad = {}, 0, []
    for line in lines:
        if re.match(r"^[0-9a-f]+ <|^_Z\w+:", line):
            written = {}
        m = re.match(r"\s+([sv]_\w+)(?: (.*))?$", re.split(r"//|;", line)[0].rstrip())
        if not m:
            m = re.match(r"\s+([a-z]+_\w+)", line)
            at += 1 if m else 0
            continue
        name, ops = m[1], operands(m[2] or "")
        if name == "s_nop":
            at += int(ops[0], 0) + 1
            continue
        at += 1
        if name.startswith("s_"):
            for r in registers(ops[0]) if ops else []:  # scalar results are waited for by the hardware
                written.pop(r, None)
            continue
        outs = 2 if name.startswith(CARRY) else 1
        rotated = re.search(r"row_|quad_perm", m[2] or "")
        for k, o in enumerate(ops[outs:]):
            for r in registers(o):
                if r in written and at - written[r][0] < 3 and (r[0] != "v" or (rotated and k == 0)):
                    bad.append((written[r][1], line.strip()))
        for o in ops[:outs]:
            for r in registers(o):
                written[r] = (at, line.strip())
    return bad


def test_the_check_sees_close_reads():
    head = ["\tv_mad_u64_u32 v[0:1], s[4:5], v1, v6, v[2:3]"]
    read = ["\tv_subb_co_u32_e64 v6, s[6:7], v4, v3, s[4:5]"]
    other = ["\tv_mov_b32_e32 v9, -1"]
    assert len(close_reads(head + read)) == len(close_reads(head + other + read)) == 2  # both words of the mask
    assert not close_reads(head + other + other + read) and not close_reads(head + ["\ts_nop 1"] + read)
    assert close_reads(head + ["\ts_nop 0"] + read)
    assert not close_reads(head + ["\ts_or_b64 s[4:5], s[4:5], s[8:9]"] + read)
    turn = ["\tv_add_u32_dpp v2, v9, v2 row_ror:8 row_mask:0xf bank_mask:0xf bound_ctrl:1"]
    assert close_reads(other + turn) and not close_reads(other + ["\ts_nop 1"] + turn)
    assert not close_reads(["\tv_mov_b32_e32 v8, -1", "\tv_add_u32_e32 v2, v8, v2"])


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_products_with_half_known_factors(tmp_path):
    """The header's products take any factors, also ones whose high half the
    compiler knows: the instructions that then fall away also kept a carry and
    its reader apart."""
    src = tmp_path / "products.hip"
    cases = {"mul by a constant": "o[0] = gl::mul(a[0], 7);",
             "mul by a widened word": "o[0] = gl::mul(a[0], w[0]);",
             "mul of a widened word": "o[0] = gl::mul(w[0], a[0]);",
             "mul by a power of two": "o[0] = gl::mul(a[0], 1ull << 40);",
             "mul by a high bit": "o[0] = gl::mul(a[0], (uint64_t)(w[0] & 1) << 32);",
             "square of a widened word": "o[0] = gl::mul(w[0], w[0]);"}
    for n in (1, 2, 3, 4):
        for r in ("ANY", "CANON", "LAZY"):
            cases[f"row of {n} {r}"] = (f"uint64_t x[{n}], y[{n}]; int32_t e[{n}] = {{}};"
                                        f"for (int i = 0; i < {n}; ++i) x[i] = a[i], y[i] = w[i];"
                                        f"gl::mul_row<{n}, gl::{r}>(x, x, y, e);"
                                        f"for (int i = 0; i < {n}; ++i) o[i] = x[i] + e[i];")
    src.write_text('#include "gl_lazy.hpp"\n#include <hip/hip_runtime.h>\n' + "".join(
        f"__global__ void k{i}(uint64_t *o, const uint64_t *a, const uint32_t *w) {{\n"
        f"  o += 4 * threadIdx.x, a += 4 * threadIdx.x, w += 4 * threadIdx.x;\n  {c}\n}}\n"
        for i, c in enumerate(cases.values())))
    out = tmp_path / "products.s"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I" + CSRC, "--cuda-device-only", "-S", "-o", str(out), str(src)],
                   check=True, capture_output=True)
    bodies = re.split(r"^_Z2?k(\d+)\w*:", re.sub(r"^_Z\d+k", "_Zk", out.read_text(), flags=re.M), flags=re.M)[1:]
    assert len(bodies) == 2 * len(cases)
    for i, text in zip(bodies[::2], bodies[1::2]):
        assert not close_reads(text.split("s_endpgm")[0].splitlines()), list(cases)[int(i)]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump not available")
def test_built_kernels(tmp_path):
    so = shutil.copy(os.path.join(ROOT, "era-boojum-cuda_amd", "libboojum_ntt.so"), tmp_path)
    subprocess.run([OBJDUMP, "--offloading", so], check=True, capture_output=True, cwd=tmp_path)
    images = glob.glob(str(tmp_path / "*gfx950*"))
    assert images
    carries = 0
    for image in images:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", image], check=True, capture_output=True,
                              text=True).stdout
        lines = text.splitlines()
        carries += sum("v_mad_u64_u32" in line for line in lines)
        assert not close_reads(lines), image
    assert carries > 10000
