"""The GEMM's stores to C declare the alignment C has: that of its elements."""

from __future__ import annotations

import re
import subprocess

import pytest

from vdn_h3_amd import _build

SOURCE = """
#define VDNH3_GEMM_KERNEL
#include "gemm_kernel.h"
namespace vdnh3 {
__global__ void probe_bf16(uint16_t *c, const uint16_t *o) { stream_store(stream_load(o), c); }
__global__ void probe_f32(float *c, const float *o) { stream_store(stream_load(o), c); }
__global__ void probe_i32(int32_t *c) { stream_store(u32x4_t{1, 2, 3, 4}, c); }
}  // namespace vdnh3
"""


def test_gemm_stores_declare_element_alignment(tmp_path):
    """Compiled to the compiler's own representation: every 16-byte access of C is marked with its elements' alignment."""
    try:
        hipcc = _build._hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    source = tmp_path / "probe.hip"
    source.write_text(SOURCE)
    proc = subprocess.run([hipcc, *_build.HIP_FLAGS, f"-I{_build.CSRC}", "--offload-device-only", "-S", "-emit-llvm",
                           str(source), "-o", "-"], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    accesses = {}
    for kernel, body in re.findall(r"define [^\n]*@\w*(probe_[a-z0-9]+)EP[^\n]*\{\n(.*?)\n\}", proc.stdout, re.S):
        accesses[kernel] = [int(a) for a in re.findall(r"<4 x (?:i32|float)>.*?align (\d+)[^\n]*!nontemporal", body)]
    assert accesses == {"probe_bf16": [2, 2], "probe_f32": [4, 4], "probe_i32": [4]}
