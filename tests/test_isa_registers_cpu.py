"""Vector registers of built kernels whose speed hangs on how many waves a SIMD
holds, from the kernel descriptors in aestrix_amd/libimq.so (CPU only: the code
objects are taken out of the library with the ROCm LLVM tools).

A SIMD's 512 registers hold eight waves of up to 64 registers.
"""

from __future__ import annotations

import os
import re
import subprocess
from pathlib import Path

import pytest

from aestrix_amd import _lib

LLVM = Path(os.environ.get("ROCM_PATH", "/opt/rocm")) / "llvm" / "bin"
TOOLS = {n: LLVM / n for n in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")}
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _run(*args: str) -> str:
    return subprocess.run(args, check=True, capture_output=True, text=True).stdout


@pytest.fixture(scope="module")
def registers(tmp_path_factory) -> dict[str, int]:
    """{kernel symbol: vector registers}."""
    lib = Path(_lib.LIB_PATH)
    if not all(p.exists() for p in TOOLS.values()) or not lib.exists():
        pytest.skip("the ROCm LLVM tools or libimq.so are missing")
    d = tmp_path_factory.mktemp("co")
    fat = d / "fatbin.bin"
    _run(str(TOOLS["llvm-objcopy"]), f"--dump-section=.hip_fatbin={fat}", str(lib), str(d / "x.so"))
    data = fat.read_bytes()
    starts = [m.start() for m in re.finditer(re.escape(MAGIC), data)] + [len(data)]
    out: dict[str, int] = {}
    for a, b in zip(starts, starts[1:]):
        (d / "b").write_bytes(data[a:b])
        _run(str(TOOLS["clang-offload-bundler"]), "--unbundle", "--type=o", f"--input={d / 'b'}",
             "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={d / 'co'}")
        notes = _run(str(TOOLS["llvm-readelf"]), "--notes", str(d / "co"))
        for kernel in notes.split(".agpr_count:")[1:]:
            name, count = (re.search(rf"\.{key}:\s+(\S+)", kernel) for key in ("name", "vgpr_count"))
            out[name.group(1)] = int(count.group(1))
    return out


def test_split_sums_of_aligned_rows_hold_eight_waves(registers):
    """The sums with 16-byte loads pay nothing for the form with single floats:
    32 registers and under, a gate/up pair (two sums a thread) 64."""
    sums = {n: v for n, v in registers.items() if "reduce_ep_kernel" in n}
    aligned = {n: v for n, v in sums.items() if not re.search(r"Lb0E+v", n)}
    assert len(aligned) >= 11
    over = {n: v for n, v in aligned.items() if v > (64 if "EpSwiGLU" in n else 32)}
    assert not over, over
