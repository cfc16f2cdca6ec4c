"""The fused output stages on the short and narrow tiles the planner gives them.

Each stage rounds the accumulator to T before its arithmetic and no C entry
point splits K, so a fused call equals imq_qgemm followed by the glue bit for
bit whatever tiles the two take.  The shapes cover 64- to 256-row tiles of 128
columns, partial row and column tiles and the split-sum kernel's unaligned rows.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import aestrix_amd as imq
from aestrix_amd import synth
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def problem(m, n, k, dtype, seed):
    x, w, s, b = synth.to_device(synth.make_problem(m, n, k, seed=seed))
    return (x, w, s, b) if dtype == "bf16" else (x.half(), w, s.half(), b.half())


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("m,n,k,rows", [(300, 1500, 768, 64), (512, 6144, 512, 128),
                                        (900, 4600, 512, 160), (1536, 4096, 512, 192)])
def test_fused_stages_on_narrow_tiles(dtype, m, n, k, rows):
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    plan = imq.qmm_plan(m, n, k, tdt, entry="fused")
    print(f"fused tiles {dtype} M={m} N={n} K={k} {plan}", flush=True)
    assert plan["kernel"] == "tile" and plan["splits"] == 1
    assert plan["tile_cols"] == 128 and plan["tile_rows"] == rows
    x, w, s, b = problem(m, n, k, dtype, seed=5)
    y = imq.qgemm(x, w, s, b)
    g = torch.Generator(device="cuda").manual_seed(6)
    res = torch.randn((m, n), device="cuda", generator=g)
    gate = torch.randn(n, device="cuda", generator=g)
    assert torch.equal(imq.qmm_postscale(x, w, s, b, 16.0), y.float() * 16.0)
    assert np.array_equal(imq.qmm_gate_add(x, w, s, b, res, gate, 0.25).cpu().numpy(),
                          ref.glue_gate_add(y.float().cpu().numpy(), res.cpu().numpy(),
                                            gate.cpu().numpy(), 0.25))
    assert torch.equal(imq.qmm_add(x, w, s, b, y), (y.float() + y.float()).to(tdt))
    if dtype == "f16":
        assert torch.equal(imq.qmm_postscale(x, w, s, b, 16.0, out_dtype=torch.float16),
                           (y.float() * 16.0).half())


@pytest.mark.parametrize("m,n,k", [(40, 700, 2560), (33, 1001, 4096), (64, 515, 2048)])
def test_split_sums_of_unaligned_rows(m, n, k):
    """Rows of partial sums that are not whole 16-byte pieces; one-hot rows of x
    pick single weights, exact whatever the split."""
    plan = imq.qmm_plan(m, n, k)
    print(f"split sums M={m} N={n} K={k} {plan}", flush=True)
    assert plan["kernel"] == "tile" and plan["splits"] > 1
    _, w, s, b = problem(1, n, k, "bf16", seed=9)
    cols = torch.linspace(0, k - 1, m).long().cuda()
    x = torch.zeros((m, k), dtype=torch.bfloat16, device="cuda")
    x[torch.arange(m), cols] = 1.0
    assert torch.equal(imq.quantized_matmul(x, w, s, b), imq.dequantize(w, s, b)[:, cols].T)


@pytest.mark.parametrize("rows", [33, 128, 129, 180, 511])
@pytest.mark.parametrize("hidden,nq", [(1024, 2048), (576, 3072), (704, 576)])
def test_layer_residual_add_around_its_plan_line(rows, hidden, nq):
    """The encoder layers' residual add: two planner models and, at 576, no K split.
    One-hot attention rows pick single weights of o and a zero down projection adds
    nothing, so the layer's output is T(x + weight) whatever tiles and splits."""
    from aestrix_amd.te import TeLayer, TextEncoderLayers
    print(f"layer residual add rows={rows} hidden={hidden} nq={nq}", flush=True)
    def proj(n, k, seed):
        _, w, s, b = problem(1, n, k, "bf16", seed)
        return imq.Q(w=w, s=s, b=b, n=n, k=k)
    o, down = proj(hidden, nq, 1), proj(hidden, 512, 2)
    down.s.zero_(), down.b.zero_()
    ones = torch.ones(hidden, device="cuda")
    te = TextEncoderLayers([TeLayer(qkv=proj(nq + 128, hidden, 3), o=o, gate_up=proj(1024, hidden, 4),
                                    down=down, norm_in=ones, norm_post=ones)], max_rows=512)
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn((rows, hidden), device="cuda", generator=g).bfloat16()
    cols = torch.linspace(0, nq - 1, rows).long().cuda()
    attn = torch.zeros((rows, nq), dtype=torch.bfloat16, device="cuda")
    attn[torch.arange(rows), cols] = 1.0
    want = (x.float() + imq.dequantize(o.w, o.s, o.b)[:, cols].T.float()).bfloat16()
    assert torch.equal(te.attn_out_mlp(0, x, attn), want)
    te.close()
