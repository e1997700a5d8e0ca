"""Host side of the GEMMs on a machine without a GPU: which calls are
refused (before anything is launched) and which get as far as their launch; launch rules."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(ROOT, "tests", "cpp", "bin", "test_gemm_host")


@pytest.mark.parametrize("mode", ["deep", "timing", "segments", "small"])
def test_gemm_host(mode):
    assert os.path.exists(BIN), "tests/cpp/bin/test_gemm_host missing: run __graft_entry__.build()"
    # no visible device, also where there is one: the operands are no memory
    env = {**os.environ, "HIP_VISIBLE_DEVICES": "", "ROCR_VISIBLE_DEVICES": ""}
    p = subprocess.run([BIN, mode], capture_output=True, text=True, timeout=120, env=env)
    assert p.returncode == 0, p.stdout + p.stderr
