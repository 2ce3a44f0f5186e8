"""The DPP multiply-add groups (row_ops.hpp): no accumulator may share a register with a
factor that a later instruction of the group still reads, also where the compiler knows
the two to hold the same value."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from ultimateepm_amd import build as B

SOURCE = r"""
#include "row_ops.hpp"
template <typename R>
__device__ void dots(const R* p, R* o) {
    const R t = p[threadIdx.x];
    R acc[4] = {t, t, t, t}, A[16];
    for (int i = 0; i < 16; ++i) A[i] = t;
    uepm::rowop::dot16(acc, t, A);
    o[threadIdx.x] = acc[0] + acc[1] + acc[2] + acc[3];
}
template <typename R>
__device__ void axpys(const R* p, R* o) {
    const R t = p[threadIdx.x];
    R A[16];
    for (int i = 0; i < 16; ++i) A[i] = t;
    uepm::rowop::axpy16(A, t, t);
    for (int i = 0; i < 16; ++i) o[threadIdx.x + 64 * i] = A[i];
}
__global__ void d32(const float* p, float* o) { dots(p, o); }
__global__ void d64(const double* p, double* o) { dots(p, o); }
__global__ void a32(const float* p, float* o) { axpys(p, o); }
__global__ void a64(const double* p, double* o) { axpys(p, o); }
"""


def _registers(operand):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", operand)
    return set(range(int(m[1]), int(m[2]) + 1)) if m else {int(operand[1:])}


def test_accumulators_share_no_register_with_a_factor(tmp_path):
    if not (os.path.exists(B.HIPCC) or shutil.which(B.HIPCC)):
        pytest.skip("no hipcc here")
    src = tmp_path / "t.hip"
    src.write_text(SOURCE)
    out = tmp_path / "t.s"
    subprocess.run([B.HIPCC, "-x", "hip", *B.COMMON, *B.DEVICE_FLAGS, "--offload-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    groups = out.read_text().split("ASMSTART")[1:]
    assert len(groups) == 6  # one group a dot16, two an axpy16
    for g in groups:
        rows = [re.findall(r"v\[\d+:\d+\]|\bv\d+\b", line.split("row_newbcast")[0])
                for line in g.split("ASMEND")[0].splitlines() if "_dpp" in line]
        assert rows and all(len(r) == 3 for r in rows)
        written = set().union(*(_registers(r[0]) for r in rows))
        read = set().union(*(_registers(r[1]) | _registers(r[2]) for r in rows))
        assert not written & read, g
