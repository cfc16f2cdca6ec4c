"""K that is not a multiple of 256 on the large-M tile kernel.

Its loop runs over K rounded up to 256, the surplus taking zero activations,
scales and biases.  The sizes sit at the edges of that rule: one to three
groups past a block, an even and an odd number of groups (rows of scales that
start inside a dword), scales from a row slice (a base inside a dword), and
non-finite values in the rows and groups that the surplus reads beside.

Oracle: RNE_T of the double-accumulated product with the bit-exact T dequant.
An fp32 sum of K products differs from it by at most about K 2^-24 of the sum
of their magnitudes, far below the rounding to T: MAE 1e-3, normwise 1e-2.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import aestrix_amd as imq
from aestrix_amd import synth
from oracle import cref, ref

pytestmark = pytest.mark.gpu

TDT = {"bf16": torch.bfloat16, "f16": torch.float16}


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def host_bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def values(bits, dtype):
    return ref.bf16_to_f32(bits).astype(np.float64) if dtype == "bf16" else \
        bits.view(np.float16).astype(np.float64)


def problem(m, n, k, dtype, seed):
    p = synth.make_problem(m, n, k, seed=seed)
    x, w, s, b = synth.to_device(p)
    if dtype == "f16":
        x, s, b = x.half(), s.half(), b.half()
    return x, w, s, b


def check(y, x, w, s, b, dtype, what):
    wh = w.cpu().numpy().view(np.uint32)
    want = cref.qmm_t_f64(host_bits(x), wh, host_bits(s), host_bits(b), dtype)
    t = torch.from_numpy(np.asarray(want, np.float64)).to(TDT[dtype])
    st = ref.error_stats_values(values(host_bits(y), dtype), values(host_bits(t), dtype))
    print(f"{what}: mae={st['mae']:.3g} normwise={st['max_rel_normwise']:.3g}", flush=True)
    assert st["mae"] <= 1e-3 and st["max_rel_normwise"] <= 1e-2, (what, st)


# (m, n, k): every tile height that is built, one to three groups past a block,
# partial row and column tiles, odd n.
SHAPES = [(5, 257, 320), (33, 130, 448), (17, 1000, 576), (64, 384, 640), (100, 515, 1984),
          (129, 301, 832), (200, 777, 2880), (333, 640, 1088), (700, 1111, 384), (1030, 260, 704),
          (512, 2560, 4544)]


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_ragged_k_matches_the_oracle(dtype, m, n, k):
    print(f"ragged {dtype} M={m} N={n} K={k} {imq.qmm_plan(m, n, k, TDT[dtype])}", flush=True)
    x, w, s, b = problem(m, n, k, dtype, seed=m + n + k)
    y = imq.quantized_matmul(x, w, s, b)
    g = imq.qgemm(x, w, s, b)
    torch.cuda.synchronize()
    assert torch.equal(y, imq.quantized_matmul(x, w, s, b))
    rows = np.unique(np.linspace(0, m - 1, 24).astype(int)) if m * n * k > 2 ** 28 else np.arange(m)
    r = torch.from_numpy(rows).cuda()
    check(y[r], x[r], w, s, b, dtype, "dispatcher")
    check(g[r], x[r], w, s, b, dtype, "tile kernel alone")


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k", [(40, 300, 320), (300, 515, 960), (130, 260, 2880)])
def test_ragged_k_one_hot_rows_are_single_weights(dtype, m, n, k):
    print(f"ragged one-hot {dtype} M={m} N={n} K={k}", flush=True)
    _, w, s, b = problem(1, n, k, dtype, seed=3)
    cols = np.linspace(0, k - 1, m).astype(int)
    x = torch.zeros((m, k), dtype=TDT[dtype], device="cuda")
    x[torch.arange(m), torch.from_numpy(cols).cuda()] = 1.0
    want = imq.dequantize(w, s, b)[:, torch.from_numpy(cols).cuda()].T
    assert torch.equal(imq.quantized_matmul(x, w, s, b), want)


@pytest.mark.parametrize("k", [320, 384, 448, 2880])
@pytest.mark.parametrize("m", [48, 300])
def test_ragged_k_neighbours_stay_out(m, k):
    """Rows of x, scales and biases that hold infinities and NaN change no other
    row's or column's outputs, and a row slice of a projection (its scales from
    the middle of a dword) gives the slice of the whole one's outputs."""
    n = 333
    print(f"ragged neighbours M={m} K={k}", flush=True)
    x, w, s, b = problem(m, n, k, "bf16", seed=11)
    y = imq.qgemm(x, w, s, b)
    x2, s2, b2 = x.clone(), s.clone(), b.clone()
    x2[1::3] = float("nan")
    x2[2::3] = float("inf")
    s2[1::2] = float("inf")
    b2[1::2] = float("nan")
    y2 = imq.qgemm(x2, w, s2, b2)
    assert torch.equal(y2[0::3, 0::2], y[0::3, 0::2])
    part = imq.qgemm(x, w[1:], s[1:], b[1:])
    assert torch.equal(part, y[:, 1:])


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_ragged_k_fused_stages_equal_the_tile_kernel_and_glue(dtype):
    m, n, k = 300, 512, 832
    print(f"ragged fused {dtype} M={m} N={n} K={k}", flush=True)
    x, w, s, b = problem(m, n, k, dtype, seed=21)
    y = imq.qgemm(x, w, s, b)
    g = torch.Generator(device="cuda").manual_seed(4)
    res = torch.randn((m, n), device="cuda", generator=g)
    gate = torch.randn(n, device="cuda", generator=g)
    assert torch.equal(imq.qmm_postscale(x, w, s, b, 16.0), y.float() * 16.0)
    assert np.array_equal(imq.qmm_gate_add(x, w, s, b, res, gate, 0.5).cpu().numpy(),
                          ref.glue_gate_add(y.float().cpu().numpy(), res.cpu().numpy(),
                                            gate.cpu().numpy(), 0.5))
    assert torch.equal(imq.qmm_add(x, w, s, b, y), (y.float() + y.float()).to(y.dtype))
    width = 200
    sw = imq.qmm_swiglu(x, w, s, b, width, 7, 260).float().cpu().numpy()
    yh = y.float().cpu().numpy()
    want = torch.from_numpy(ref.glue_swiglu(yh[:, 7:7 + width], yh[:, 260:260 + width], 1.0, 1.0)
                            .astype(np.float32)).to(y.dtype).float().numpy()
    st = ref.error_stats_values(sw.astype(np.float64), want.astype(np.float64))
    assert st["mae"] <= 1e-3 and st["max_rel_normwise"] <= 1e-2, st
