"""A double block's shared launches: the plans that real sizes get, their results
on those tiles and the kernels that a pass launches.

Each case names the tiles and K splits of its four launches, so that a change of
the planner's constants that drops a tile from these tests fails here first.
Row counts leave the last row tile of both parts part empty.  q, k and v equal
imq_qgemm bit for bit (no split, the same products); the residual after both
halves equals the single products and their glue within the reordering of fp32
sums: K of them differ by at most K 2^-24 of their magnitudes' sum, far below
one rounding of the product to T, 2^-9 (bf16) or 2^-12 (f16) of it (MAE 1e-3,
normwise 1e-2).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import aestrix_amd as imq
from aestrix_amd.step import DitDims, DitStep, random_projections
from oracle import ref

pytestmark = pytest.mark.gpu

# l_img, l_txt, dim, ff_inner; tile rows x columns / K splits of q/k/v, attention
# out, MLP in, MLP out on 256 compute units.
CASES = [
    ((1000, 490, 3072, 9216), "256x256/1 192x128/1 256x256/1 256x256/3"),
    ((799, 500, 1536, 4096), "256x128/1 128x128/1 192x256/1 128x128/1"),
    ((1000, 500, 2048, 6144), "192x256/1 128x128/1 192x256/1 128x128/1"),
    ((2300, 500, 3072, 9216), "224x256/1 160x256/1 224x256/1 160x256/1"),
    ((570, 300, 3072, 9216), "160x256/1 128x128/1 160x256/1 192x128/2"),
    ((700, 300, 1536, 1536), "192x128/1 128x128/1 128x256/1 128x128/1"),
    ((250, 16, 1536, 4096), "128x128/1 128x128/3 128x256/1 128x128/6"),
]
GROUPS = ("qkv", "attn_out", "mlp_in", "mlp_out")


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the plans named are those of 256 compute units")


def close(x, want, what):
    st = ref.error_stats_values(x.cpu().numpy().astype(np.float64),
                                want.cpu().numpy().astype(np.float64))
    print(f"  {what}: mae={st['mae']:.3g} normwise={st['max_rel_normwise']:.3g}", flush=True)
    assert st["mae"] <= 1e-3 and st["max_rel_normwise"] <= 1e-2, (what, st)


@pytest.mark.parametrize("tdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sizes,plans", CASES, ids=["x".join(map(str, c[0])) for c in CASES])
def test_shared_launches_by_plan(tdt, sizes, plans):
    l_img, l_txt, dim, ff = sizes
    print(f"shared launches {tdt} {sizes}", flush=True)
    d = DitDims(l_img=l_img, l_txt=l_txt, dim=dim, ff_inner=ff, n_double=1, n_single=0)
    projs = random_projections(d, tdt, seed=3)
    step = DitStep(d, projs)
    p = {g: step.group_plan(g) for g in GROUPS}
    assert all(p[g]["kernel"] == "tile" for g in GROUPS)
    assert " ".join("%(tile_rows)dx%(tile_cols)d/%(splits)d" % p[g] for g in GROUPS) == plans
    g = torch.Generator(device="cuda").manual_seed(1)

    def randn(*s):
        return torch.randn(s, device="cuda", generator=g)

    gates = randn(4, dim) * 0.5
    step.set_conditioning(torch.ones(dim, device="cuda"), gates.contiguous())
    nx, nx2, attn = (randn(d.joint, dim).to(tdt) for _ in range(3))
    t, i = slice(0, l_txt), slice(l_txt, d.joint)
    qkv = [torch.empty((d.joint, dim), dtype=tdt, device="cuda") for _ in range(3)]
    step.double_attn_in(0, None, *qkv, nx=nx)
    assert step.kernels == 1
    for j in range(3):
        for rows, q in ((i, projs[j]), (t, projs[3 + j])):
            assert torch.equal(qkv[j][rows], imq.qgemm(nx[rows], q.w, q.s, q.b))
    x = randn(d.joint, dim)
    want = x.clone()
    sums = {g: 2 if p[g]["splits"] > 1 else 0 for g in GROUPS}  # one per projection
    step.double_attn_out(0, attn, x)
    assert step.kernels == 1 + sums["attn_out"]
    for rows, q, k in ((i, projs[6], 0), (t, projs[7], 1)):
        want[rows] = imq.qmm_gate_add(attn[rows], q.w, q.s, q.b, want[rows].contiguous(),
                                      gates[k].contiguous(), 1.0)
    close(x, want, "attention out")
    want = x.clone()
    step.double_mlp(0, x, nx=nx2)
    assert step.kernels == 2 + sums["mlp_out"]
    for rows, up, down, k in ((i, projs[8], projs[9], 2), (t, projs[10], projs[11], 3)):
        m = imq.qmm_swiglu(nx2[rows], up.w, up.s, up.b, ff, 0, ff)
        want[rows] = imq.qmm_gate_add(m, down.w, down.s, down.b, want[rows].contiguous(),
                                      gates[k].contiguous(), 1.0)
    close(x, want, "MLP out")
    step.close()


def test_kernels_of_a_step():
    """Every kernel of a pass is counted: norms, shared and single products, split
    sums, the head's four operations."""
    d = DitDims(l_img=250, l_txt=16, dim=1536, ff_inner=4096, n_double=2, n_single=1)
    step = DitStep(d, random_projections(d, torch.float16, seed=4))
    h, e = torch.randn(250, 1536, device="cuda"), torch.randn(16, 1536, device="cuda")
    qkv = torch.empty((266, 3 * 1536), dtype=torch.float16, device="cuda")
    concat = torch.zeros((266, 1536 + 4096), dtype=torch.float16, device="cuda")
    x = torch.randn(266, 1536, device="cuda")
    step.single_attn_in(0, x, qkv, concat)
    single = step.kernels
    step.single_attn_out(0, concat, x)
    single += step.kernels
    assert 4 <= single <= 7  # a norm, three products, up to three sums
    for graph in (True, False):
        step.run(h, e, use_graph=graph)
        # Per double block two norms, four shared launches, two products' sums twice.
        assert step.kernels == 2 * (2 + 4 + 4) + single
        assert step.launches == 2 * 14 + 4
    step.close()


def test_operands_past_32_bit_offsets_run_one_by_one():
    """MLP-outs whose image activations reach 2 GiB: the image product on the kernel
    with 64-bit addresses, the text product on its own; sampled rows against the
    single entry points over those rows alone."""
    l_img, l_txt, dim, ff = 16384, 40, 256, 65536
    d = DitDims(l_img=l_img, l_txt=l_txt, dim=dim, ff_inner=ff, n_double=1, n_single=0)
    projs = random_projections(d, torch.float16, seed=5)
    step = DitStep(d, projs)
    assert step.group_plan("mlp_in")["kernel"] == "tile"
    assert step.group_plan("mlp_out")["kernel"] == "tile_reg"
    g = torch.Generator(device="cuda").manual_seed(2)
    gates = torch.randn((4, dim), device="cuda", generator=g) * 0.5
    step.set_conditioning(torch.ones(dim, device="cuda"), gates.contiguous())
    nx = torch.randn((d.joint, dim), device="cuda", generator=g).half()
    x0 = torch.randn((d.joint, dim), device="cuda", generator=g)
    x = x0.clone()
    step.double_mlp(0, x, nx=nx)
    assert 3 <= step.kernels <= 4  # the shared SwiGLU, two products, at most one sum
    for rows, up, down, k in (
            (torch.tensor([l_txt, l_txt + 127, l_txt + 8192, d.joint - 1]), projs[8], projs[9], 2),
            (torch.arange(l_txt), projs[10], projs[11], 3)):
        rows = rows.cuda()
        m = imq.qmm_swiglu(nx[rows], up.w, up.s, up.b, ff, 0, ff)
        want = imq.qmm_gate_add(m, down.w, down.s, down.b, x0[rows], gates[k].contiguous(), 1.0)
        close(x[rows], want, "sampled rows")
    step.close()
