"""The prompt quantizers' code arithmetic (iq_quantize.h), checked on the CPU.

A finite group's codes come from one multiplication by a reciprocal within one
fp32 ulp of 1/s in place of the reference's division by s (quant.py:69-71,
108-109), and its scale from a multiplication by 1/L.  tests/quant_reciprocal.c
compares the two over all pairs of finite fp16 operands and over all bf16
pairs with s in [2^-100, 2^100], for every level count and all three
reciprocals.  The GPU tests then compare the kernels' codes bit for bit with
the oracle (tests/test_gpu_quantize_edges.py) and the golden vectors.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("gcc") is None, reason="gcc is needed to build the checker")
def test_one_multiplication_gives_the_reference_codes_exhaustively(tmp_path):
    exe = str(tmp_path / "quant_reciprocal")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-fopenmp", "-o", exe,
                    os.path.join(HERE, "quant_reciprocal.c"), "-lm"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "fp16 0 bf16 0 scales 0"
