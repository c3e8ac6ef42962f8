"""Registers of the GGUF matrix-core kernel that decide how many of its workgroups share a compute unit."""
import os

import pytest

from oxydllm_amd import _lib, synth
from tests import gpu_code


def test_one_to_four_q6_k_rows_have_two_workgroups_a_compute_unit(tmp_path):
    """Eight waves each, two a SIMD: four of them fit up to 128 of the 512 registers.  Layers of more than 256 strips
    take 7 - 18 % longer with one workgroup a compute unit."""
    if not os.path.exists(gpu_code.LLVM + "llvm-readelf"):
        pytest.skip("no llvm-readelf")
    found = {}
    for co in gpu_code.code_objects(_lib.LIB_PATH, tmp_path):
        if b"ggm_kernel" in co.read_bytes():
            found.update(gpu_code.registers(co))
    for fmt in (synth.GGUF_Q6_K, synth.GGUF_Q4_0, synth.GGUF_Q4_K, synth.GGUF_Q8_0, synth.GGUF_Q5_K):
        (regs,) = [r for n, r in found.items() if f"10ggm_kernelILi{fmt}ELi1ELi1ELi8ELi1ELb0EE" in n]
        assert regs <= 128, (fmt, regs)
