"""The quantizers' arithmetic (csrc/quant_math.h) equals the specification's plain operations:
tests/gpu_checks/quant_math_check.hip runs the kernels' own code over whole input domains on the
GPU. Needs a GPU and the binary that kvq_decode_amd.build compiles."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gpu_checks", "quant_math_check")


def test_quantizer_arithmetic_exhaustively():
    assert os.path.exists(BIN), f"{BIN} missing: build with python -m kvq_decode_amd.build"
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=100)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
