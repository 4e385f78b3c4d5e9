"""The bounds of the prefill kernels' weight copies (Q4Piece in
metalops_amd/csrc/q4_common.h), run on the host: tests/q4_piece_check.cpp is compiled
with hipcc (host code only, no GPU call).  Widths below a wave's 64 columns leave
waves without a column of their own; their copies have to stay inside the row too."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_copies_stay_inside_the_row(tmp_path):
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "q4_piece_check")
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950",
                    "-I", os.path.join(ROOT, "metalops_amd", "csrc"), "-I", os.path.join(ROOT, "include"),
                    "-x", "hip", os.path.join(HERE, "q4_piece_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
