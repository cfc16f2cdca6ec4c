"""The double block's grouped launches against the single ones.

Each product of a group keeps its own rows, weights and output stage, and no
stage but the gated residual add may split K: q, k and v equal imq_qgemm bit
for bit, and the residual after both halves equals the same products and glue
within the reordering of their fp32 sums (MAE 1e-3, normwise 1e-2).  Row counts
take the 128-row tiles (128 and 256 columns; the taller ones are in
test_gpu_group_plans.py) through their edges: one tile for both, a text part larger
than the image part, single rows, and a K long enough for the MLP-outs to split.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import aestrix_amd as imq
from aestrix_amd.step import DitDims, DitStep, random_projections
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("tdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("l_img,l_txt,dim,ff", [(1, 1, 256, 256), (33, 300, 512, 768),
                                                (257, 129, 768, 2560), (700, 77, 512, 256),
                                                (128, 128, 256, 6144)])
def test_double_block_groups(tdt, l_img, l_txt, dim, ff):
    print(f"grouped {tdt} {l_img}+{l_txt} dim={dim} ff={ff}", flush=True)
    d = DitDims(l_img=l_img, l_txt=l_txt, dim=dim, ff_inner=ff, n_double=1, n_single=0)
    projs = random_projections(d, tdt, seed=3)
    step = DitStep(d, projs)
    g = torch.Generator(device="cuda").manual_seed(1)

    def randn(*s):
        return torch.randn(s, device="cuda", generator=g)

    gates = randn(4, dim) * 0.5
    step.set_conditioning(torch.ones(dim, device="cuda"), gates.contiguous())
    nx, nx2, attn = (randn(d.joint, dim).to(tdt) for _ in range(3))
    x0 = randn(d.joint, dim)
    t, i = slice(0, l_txt), slice(l_txt, d.joint)
    qkv = [torch.empty((d.joint, dim), dtype=tdt, device="cuda") for _ in range(3)]
    step.double_attn_in(0, None, *qkv, nx=nx)
    for j in range(3):
        for rows, q in ((i, projs[j]), (t, projs[3 + j])):
            assert torch.equal(qkv[j][rows], imq.qgemm(nx[rows], q.w, q.s, q.b))
    x = x0.clone()
    step.double_attn_out(0, attn, x)
    step.double_mlp(0, x, nx=nx2)
    want = x0.clone()
    for rows, out, up, down, ga, gm in ((i, projs[6], projs[8], projs[9], 0, 2),
                                        (t, projs[7], projs[10], projs[11], 1, 3)):
        r = want[rows].contiguous()
        r = imq.qmm_gate_add(attn[rows], out.w, out.s, out.b, r, gates[ga].contiguous(), 1.0)
        m = imq.qmm_swiglu(nx2[rows], up.w, up.s, up.b, ff, 0, ff)
        want[rows] = imq.qmm_gate_add(m, down.w, down.s, down.b, r, gates[gm].contiguous(), 1.0)
    st = ref.error_stats_values(x.cpu().numpy().astype(np.float64), want.cpu().numpy().astype(np.float64))
    print(f"  mae={st['mae']:.3g} normwise={st['max_rel_normwise']:.3g}", flush=True)
    assert st["mae"] <= 1e-3 and st["max_rel_normwise"] <= 1e-2, st
    again = x0.clone()
    step.double_attn_out(0, attn, again)
    step.double_mlp(0, again, nx=nx2)
    assert torch.equal(again, x)
    step.close()
