"""The f32 qGEMV with two weight rows per lane (two to four rows of x, from
16384 weight rows and K = 768 on, in K tiles that fill the lanes, or over many
rows) and its neighbours on the one-row form.

Oracle: float64 sums of x with the bit-exact f32 weights.  An fp32 sum of K
products in any order is off by at most K 2^-23 of the sum of their magnitudes
(one rounding per product and per add, to first order).
"""

from __future__ import annotations

import pytest
import torch

import aestrix_amd as imq
from aestrix_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,k", [(16383, 768), (16384, 704), (16384, 768), (16385, 832),
                                 (16385, 960), (16500, 4160), (17000, 3072), (17000, 4032),
                                 (28671, 1536), (28672, 1536)])
def test_f32_wide_rows(m, n, k):
    print(f"f32 wide M={m} N={n} K={k}", flush=True)
    x, w, s, b = synth.to_device(synth.make_problem(m, n, k, seed=m + k))
    x, s, b = x.float() * 1.37, s.float(), b.float()
    y = imq.quantized_matmul(x, w, s, b).double()
    assert torch.equal(y, imq.quantized_matmul(x, w, s, b).double())
    deq = imq.dequantize(w, s, b).double()
    want = x.double() @ deq.T
    bound = k * 2.0 ** -23 * (x.double().abs() @ deq.abs().T)
    assert torch.all((y - want).abs() <= bound)
    one = torch.zeros_like(x)
    cols = torch.linspace(0, k - 1, m).long().cuda()
    one[torch.arange(m), cols] = 1.0
    assert torch.equal(imq.quantized_matmul(one, w, s, b), imq.dequantize(w, s, b)[:, cols].T)
