"""The conditioning chain with the SiLU in the stores of its first two projections:
every pass height (each instantiation of the f32 qGEMV, its last rows repeated or
not, a second pass) and projections whose last workgroup is not full.

Oracle: ref.cond_chain.  Each output is a sum of K products in fp32, off by at
most K 2^-23 of its magnitudes' sum; over random signs the chained error stays
far under 1e-5 normwise (measured up to 3e-7), which is the bar here.  A SiLU
left out or taken twice, or a row in another's place, is off by more than 0.1.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from aestrix_amd.cond import Conditioner, random_conditioner
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("dim", [64, 832, 1024])
@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 8, 9, 15, 16, 17])
def test_chain_at_each_pass_height(dim, count):
    print(f"chain rows dim={dim} timesteps={count}", flush=True)
    l1, l2, heads = random_conditioner(dim, 192, seed=dim + count)
    host = lambda q: (q.w.cpu().numpy().view(np.uint32), q.s.cpu().numpy(), q.b.cpu().numpy())
    t = np.linspace(990.0, 10.0, count).astype(np.float32)
    cond = Conditioner(l1, l2, heads)
    temb, hd = cond.run(t)
    temb2, hd2 = cond.run(t)
    torch.cuda.synchronize()
    assert torch.equal(temb, temb2) and torch.equal(hd, hd2)
    rows = np.unique(np.linspace(0, heads.n - 1, 257).astype(int))
    wt, wh = ref.cond_chain(t, host(l1), host(l2), host(heads), head_rows=rows)
    for got, want in ((temb.cpu().numpy(), wt), (hd.cpu().numpy()[:, rows], wh)):
        d = np.abs(got.astype(np.float64) - want)
        assert np.all(d.max(axis=1) <= 1e-5 * np.abs(want).max(axis=1))
    cond.close()
