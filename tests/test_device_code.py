"""The gfx950 code that the compiler makes of the device sources: what inline code has to keep to by itself, since the compiler
does not look into it."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "wick_amd", "csrc")
LLVM = "/opt/rocm/llvm/bin"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w"]  # the Makefile's

# Sums of which the first is known last, and a source that a vector instruction writes right in front.
PROBE = """
#include "wick_rocm_device.h"
using namespace wick_rocm;
__global__ void probe(v16f* sums, const float* x, const v16f* v) {
    v16f s = sums[threadIdx.x];
    s[0] = sqrtf(1.0f / s[0]);
    fmac_row_lanes(s, x[threadIdx.x] * 3.0f, v[threadIdx.x]);
    sums[threadIdx.x] = s;
}
"""


def registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]$|v(\d+)$", operand)
    if not m:
        return range(0)
    return range(int(m[1]), int(m[2]) + 1) if m[1] else range(int(m[3]), int(m[3]) + 1)


def lane_reads(asm):
    """(how many multiply-adds that read another lane there are, those less than two wait states behind a vector write of what they read)"""
    before, found, early = [], 0, []
    for line in asm.splitlines():
        line = re.split(r";|//", line)[0].strip()
        if not line or line.startswith("."):
            continue
        if line.endswith(":"):  # a place that is jumped to: the jump itself is a wait state, what is in front of it stays
            continue
        op, _, rest = line.partition(" ")
        operands = [o.strip() for o in rest.split(",")]
        if op == "v_fmac_f32_dpp":
            found += 1
            states = 0
            for was, written, waits in reversed(before):
                if states >= 2:
                    break
                if set(written) & set(registers(operands[1].split()[0])):
                    early.append((was, line))
                states += waits
        written = registers(operands[0]) if op.startswith("v_") and not op.startswith("v_cmp") else range(0)
        before = (before + [(line, written, int(rest, 0) + 1 if op == "s_nop" else 1)])[-4:]
    return found, early


def test_the_lane_reads_of_a_run_wait_for_their_source(tmp_path):
    """A source of another lane is read two wait states after a vector instruction wrote it at the earliest, whatever order the
    compiler would like the sums in."""
    src = tmp_path / "probe.hip"
    src.write_text(PROBE)
    r = subprocess.run(["/opt/rocm/bin/hipcc", *FLAGS, "-I", CSRC, "--cuda-device-only", "-S", str(src), "-o", str(tmp_path / "probe.s")],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    found, early = lane_reads((tmp_path / "probe.s").read_text())
    assert found == 16 and not early, early


def test_the_lane_reads_of_the_built_gemm_wait_for_their_source(tmp_path):
    """The same of every such instruction in the library as it is built."""
    shutil.copy(os.path.join(ROOT, "wick_amd", "lib", "obj", "gemm.o"), tmp_path)
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "gemm.o"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    code, = [p for p in tmp_path.iterdir() if "gfx950" in p.name]
    asm = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", "--no-leading-addr", str(code)], check=True, capture_output=True, text=True).stdout
    found, early = lane_reads(asm)
    assert found > 0 and not early, early
