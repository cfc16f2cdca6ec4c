"""Embedding rows by ids on the host (imq_dequantize_rows_host): the ids travel as
kernel arguments, 768 a launch.  Bit-equal to the same rows of the whole
dequantize at one id, around a launch's capacity and past the Python layer's
limit, for every type, both integer types and a strided id tensor; ids outside
the table are refused before any launch, whatever the count."""

from __future__ import annotations

import pytest
import torch

import aestrix_amd as imq
from aestrix_amd import ops, synth

pytestmark = pytest.mark.gpu
TDT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("count", [1, 30, 767, 768, 769, 2000, ops.MAX_ARG_ROWS + 1])
def test_host_ids_equal_the_whole_dequantize(dtype, count):
    print(f"rows by host ids {dtype} count={count}", flush=True)
    n, k = 500, 192
    _, w, s, b = synth.to_device(synth.make_problem(1, n, k, seed=2))
    s, b = s.to(TDT[dtype]), b.to(TDT[dtype])
    ids = torch.randint(0, n, (count,), generator=torch.Generator().manual_seed(count))
    ids[-1], ids[0] = n - 1, 0
    want = imq.dequantize(w, s, b)[ids.cuda()]
    assert torch.equal(imq.dequantize_rows(w, s, b, ids), want)
    assert torch.equal(imq.dequantize_rows(w, s, b, ids.int()), want)
    assert torch.equal(imq.dequantize_rows(w, s, b, ids.repeat_interleave(2)[::2]), want)
    assert torch.equal(imq.dequantize_rows(w, s, b, ids.cuda()), want)


def test_host_ids_captured_and_out_of_range():
    n, k = 300, 256
    _, w, s, b = synth.to_device(synth.make_problem(1, n, k, seed=4))
    for bad in (n, -1, 1 << 40):
        ids = torch.tensor([0, bad, 1])
        with pytest.raises(ValueError, match="ids must lie"):
            imq.dequantize_rows(w, s, b, ids)
    assert imq.dequantize_rows(w, s, b, torch.zeros(0, dtype=torch.int64)).shape == (0, k)
    ids = torch.arange(20)
    out = torch.empty((20, k), dtype=s.dtype, device="cuda")
    want = imq.dequantize(w, s, b)[:20]
    imq.dequantize_rows(w, s, b, ids, out=out)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        imq.dequantize_rows(w, s, b, ids, out=out)
    ids.zero_()  # read at capture
    for _ in range(3):
        out.zero_()
        torch.randn(100, device="cuda").sum().item()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_host_ids_in_the_middle_of_a_byte_buffer():
    n, k = 300, 256
    _, w, s, b = synth.to_device(synth.make_problem(1, n, k, seed=6))
    want = imq.dequantize(w, s, b)
    for off in (1, 4):
        buf = bytearray(off) + bytearray(torch.arange(40).numpy().tobytes())
        ids = torch.frombuffer(buf, dtype=torch.int64, offset=off)
        print(f"rows by host ids {ids.data_ptr() % 8} bytes past a multiple of 8", flush=True)
        assert torch.equal(imq.dequantize_rows(w, s, b, ids), want[:40])


def test_more_host_ids_than_arguments_pay_for_are_captured():
    n, k, count = 300, 64, ops.MAX_ARG_ROWS + 900
    _, w, s, b = synth.to_device(synth.make_problem(1, n, k, seed=8))
    ids = torch.randint(0, n, (count,), generator=torch.Generator().manual_seed(3))
    want = imq.dequantize(w, s, b)[ids.cuda()]
    out = torch.empty_like(want)
    imq.dequantize_rows(w, s, b, ids, out=out)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        imq.dequantize_rows(w, s, b, ids, out=out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
