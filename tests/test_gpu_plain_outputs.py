"""Outputs are plain tensors, also where the inputs are of a torch.Tensor subclass."""

from __future__ import annotations

import pytest
import torch

import aestrix_amd as imq
from aestrix_amd import synth
from aestrix_amd.te import TeLayer, TextEncoderLayers

pytestmark = pytest.mark.gpu


class Tagged(torch.Tensor):
    pass


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def test_outputs_are_plain_tensors():
    x, w, s, b = synth.to_device(synth.make_problem(3, 256, 256, seed=1))
    xt, st, bt = (t.as_subclass(Tagged) for t in (x, s, b))
    y = imq.quantized_matmul(xt, w, st, bt)
    assert type(y) is torch.Tensor and torch.equal(y, imq.quantized_matmul(x, w, s, b))
    d = imq.dequantize(w, st, bt)
    assert type(d) is torch.Tensor and torch.equal(d, imq.dequantize(w, s, b))
    q = imq.Q(w=w, s=s, b=b, n=256, k=256)
    up = synth.to_device(synth.make_problem(1, 512, 256, seed=2))
    qkv = synth.to_device(synth.make_problem(1, 256 + 2 * 64, 256, seed=3))
    ones = torch.ones(256, device="cuda")
    te = TextEncoderLayers([TeLayer(qkv=imq.Q(*qkv[1:], n=384, k=256), o=q,
                                    gate_up=imq.Q(*up[1:], n=512, k=256), down=q, norm_in=ones,
                                    norm_post=ones)], max_rows=4)
    out = te.attn_in(0, xt)
    assert type(out) is torch.Tensor and torch.equal(out, te.attn_in(0, x))
    te.close()
