"""The package imports with a torch that has no GPU names (CPU; in a process of
its own, with the name taken out of torch first)."""

from __future__ import annotations

import subprocess
import sys
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

CODE = """
import types
import torch
if hasattr(torch._C, "_cuda_getCurrentRawStream"):
    del torch._C._cuda_getCurrentRawStream
import aestrix_amd
from aestrix_amd import ops, weights
torch.cuda.current_stream = lambda idx: types.SimpleNamespace(cuda_stream=1000 + idx)
assert ops.raw_stream(3) == 1003
"""


def test_import_without_torch_gpu_names():
    r = subprocess.run([sys.executable, "-c", CODE], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
