"""Every kernel launcher that libimq's host C++ calls is an ordinary undefined
symbol of its object file, so that a translation unit left out of a link is a
link error and not a call of a null address (CPU: host-only compiles, no GPU)."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CLANG = Path("/opt/rocm/llvm/bin/clang++")


@pytest.mark.parametrize("src", ["capi", "step", "cond", "te"])
def test_launchers_are_strong_symbols(tmp_path, src):
    if not CLANG.exists() or shutil.which("nm") is None:
        pytest.skip("ROCm clang++ or nm not available")
    obj = tmp_path / f"{src}.o"
    subprocess.run([str(CLANG), "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{ROOT / 'aestrix_amd' / 'csrc'}", "-c",
                    str(ROOT / "aestrix_amd" / "csrc" / f"{src}.cpp"), "-o", str(obj)],
                   check=True, capture_output=True)
    lines = subprocess.run(["nm", "-uC", str(obj)], check=True, capture_output=True,
                           text=True).stdout.splitlines()
    ours = [line.split(None, 1) for line in lines if "imq::" in line]
    assert any("launch_" in name for _, name in ours)
    assert not [name for kind, name in ours if kind != "U"]
