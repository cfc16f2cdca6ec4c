"""Tile plans on the host: the planner of qgemm.hip compiled without a device (it
counts on 256 CUs then) and asked for the plans that a measurement decided."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "aestrix_amd", "csrc")
SOURCE = r"""
#include "qgemm.hip"
#include <cstdio>
int main() {
  int m, n, k, split, pair, resid;
  while (std::scanf("%d %d %d %d %d %d", &m, &n, &k, &split, &pair, &resid) == 6) {
    const imq::BigPlan p = imq::pick_big_plan(m, n, k, 256, split, pair, resid);
    std::printf("%d %d %d %d\n", 32 * p.mt, 128 * p.nt, p.splits,
                imq::qgemm_big_supported(k, n, m) ? 1 : 0);
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("plans")
    src, exe = d / "plans.hip", d / "plans"
    src.write_text(SOURCE)
    # The kernels' launches stay undefined: nothing here calls them.
    subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-O1", "-w", "-I", CSRC, "-I",
                    os.path.join(ROOT, "include"), str(src), "-o", str(exe),
                    "-Wl,--unresolved-symbols=ignore-all"], check=True, timeout=300)

    def ask(*shapes):
        text = "\n".join(" ".join(str(int(v)) for v in s) for s in shapes)
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True,
                             timeout=60, env={**os.environ, "HIP_VISIBLE_DEVICES": ""}).stdout
        rows = [tuple(int(v) for v in line.split()) for line in out.splitlines()]
        assert len(rows) == len(shapes)
        return rows

    return ask


def test_ragged_rows_of_partial_sums_split_less(plans):
    """N % 4 != 0: a split's partial sums are added float by float."""
    odd, even = plans((62, 12390, 8448, 1, 0, 0), (62, 12392, 8448, 1, 0, 0))
    assert odd[2] <= 2 < even[2], (odd, even)
    for s in ((391, 9998, 3712), (372, 6779, 5824)):
        assert plans((*s, 1, 0, 0))[0][2] == 1, s


PAIR_SPLITS = {33: 3, 48: 3, 64: 3, 112: 2, 128: 2, 129: 2, 136: 2, 144: 2, 160: 2, 170: 1}


@pytest.mark.parametrize("rows", sorted(PAIR_SPLITS))
def test_a_gate_up_pairs_third_split(plans, rows):
    """Four layers (19456 rows of weights, K = 2560) at 129-144 rows: 330-333 us with two
    splits, 338-343 with three; at 33-64 rows three are ahead."""
    assert plans((rows, 19456, 2560, 1, 1, 0))[0][2] == PAIR_SPLITS[rows]


# m, n, k, and whether the large-M kernel takes the shape (else the register-staged).
RAGGED = [(865, 16768, 704, 0), (865, 16768, 832, 0), (865, 16768, 1152, 0), (865, 16768, 1600, 0),
          (865, 16768, 2880, 1), (865, 16768, 1280, 1), (1948, 19724, 832, 0),
          (495, 26496, 1152, 1), (4608, 3072, 960, 1), (333, 5001, 2880, 1), (333, 5001, 704, 1),
          (2048, 2048, 832, 1), (1500, 12288, 832, 1), (700, 27648, 832, 1), (512, 2560, 320, 1),
          (512, 18432, 448, 0), (4608, 9216, 192, 0), (64, 512, 64, 0)]


@pytest.mark.parametrize("m,n,k,tile", RAGGED)
def test_kernel_of_a_ragged_k(plans, m, n, k, tile):
    assert plans((m, n, k, 0, 0, 0))[0][3] == tile
