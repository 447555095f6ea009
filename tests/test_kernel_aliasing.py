"""The last PLOC passes' kernel writes its errors and logs into the block of words
that it reads back for the host, so no parameter of it may be declared free of
aliases: the compiler could then read the words before they are written."""
import re
import subprocess
from pathlib import Path

import pytest

from realtimeraytracing_amd import build

ROOT = Path(__file__).resolve().parents[1]


def test_ploc_tail_parameters(tmp_path):
    try:
        hipcc = build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc missing")
    ir = tmp_path / "build.ll"
    subprocess.run([hipcc, *build.compile_flags(), "-O1", "-Xclang", "-disable-llvm-passes", "--cuda-device-only", "-S",
                    "-emit-llvm", str(build.CSRC / "build.hip"), "-o", str(ir)], check=True, capture_output=True)
    heads = re.findall(r"^define amdgpu_kernel void @\S*k_ploc_tail\S*\((.*)\) #", ir.read_text(), re.M)
    assert len(heads) == 1
    assert "noalias" not in heads[0]
