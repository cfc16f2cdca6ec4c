"""The work a program has this framework do, as cases that can be timed and checked.

Each case is a dict of plain values; ``kind`` names the public entry points it
goes through:

* ``layers``   -- the text encoder's layer halves (``aestrix_amd.te``);
* ``embed``    -- the embedding rows of a prompt's token ids (``dequantize_rows``);
* ``chain``    -- the denoiser's conditioning chain (``aestrix_amd.cond``), float32;
* ``double`` / ``single`` -- one transformer block of the denoiser through its
  halves around the caller's attention (``aestrix_amd.step``);
* ``denoise``  -- one whole denoise step, replayed as a graph;
* ``matmul``   -- ``quantized_matmul`` on one resident packed projection;
* ``linear``   -- ``apply_linear``: float32 in, float16 inside, float32 (or float16) out;
* ``dequant``  -- a whole packed projection expanded.

Weights are in the packed format (eight 4-bit codes a word, a scale and a bias
per 64 inputs) with the sizes of trained ones: a projection's outputs have the
scale of its inputs.  Everything is drawn on the device from the seed.
"""

import math

import torch

from aestrix_amd import cond as cond_mod
from aestrix_amd import ops
from aestrix_amd import step as step_mod
from aestrix_amd import te as te_mod

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# Layer widths: the text encoder's, and those of a smaller one.
WIDTHS = {"base": (2560, 4096, 1024, 9728), "small": (1024, 2048, 1024, 3072)}


def listed():
    return [
        # One token through four encoder layers: the latency of the smallest
        # calls, every projection a weight stream.
        {"name": "layers-1", "kind": "layers", "rows": 1, "layers": 4, "width": "base", "dtype": "bf16"},
        # A short prompt's 30 tokens: few rows against the whole weight stream.
        {"name": "layers-30", "kind": "layers", "rows": 30, "layers": 4, "width": "base", "dtype": "bf16"},
        # A full padded prompt window.
        {"name": "layers-512", "kind": "layers", "rows": 512, "layers": 4, "width": "base", "dtype": "bf16"},
        # The embedding rows of a 30-token prompt, ids on the host as a
        # tokenizer leaves them.
        {"name": "embed-30", "kind": "embed", "count": 30, "rows": 131072, "k": 2560, "dtype": "bf16"},
        # The modulation vectors of a four-step schedule, once per image.
        {"name": "chain-4", "kind": "chain", "count": 4, "dim": 3072},
        # A double block of a 512 x 512 image: 1024 image and 512 text rows.
        {"name": "double-512px", "kind": "double", "img": 1024, "txt": 512, "dim": 3072, "ff": 9216, "dtype": "f16"},
        # A single block of a 1024 x 1024 image: 4096 image and 512 text rows.
        {"name": "single-1024px", "kind": "single", "img": 4096, "txt": 512, "dim": 3072, "ff": 9216, "dtype": "f16"},
        # The whole denoise step of a 1024 x 1024 image, the program's inner loop.
        {"name": "denoise-1024px", "kind": "denoise", "img": 4096, "txt": 512, "dim": 3072, "ff": 9216, "double": 5, "single": 20, "dtype": "f16"},
        # The largest single projection that the denoiser calls on its own.
        {"name": "matmul-mlp-in", "kind": "matmul", "m": 4608, "n": 18432, "k": 3072, "dtype": "bf16"},
        # Ragged sizes, as other models and prompts bring them.
        {"name": "matmul-ragged", "kind": "matmul", "m": 333, "n": 5001, "k": 2880, "dtype": "bf16"},
        # An attention projection of the denoiser called from float32 activations.
        {"name": "linear-4096", "kind": "linear", "m": 4096, "n": 3072, "k": 3072, "dynamic": False, "out16": False},
        # The largest projection expanded, for a caller that keeps dense weights.
        {"name": "dequant-qkv-mlp", "kind": "dequant", "n": 27648, "k": 3072, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layers", "layers", "embed", "chain", "double", "single", "denoise", "matmul", "matmul", "matmul",
                       "linear", "dequant"])
    if kind == "layers":
        return {"kind": kind, "rows": _log(rng, 1, 512), "layers": 4, "width": rng.choice(["base", "base", "small"]),
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "embed":
        return {"kind": kind, "count": _log(rng, 1, 2048), "rows": _log(rng, 8192, 262144), "k": 64 * rng.randint(8, 80),
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "chain":
        return {"kind": kind, "count": _log(rng, 1, 32), "dim": 256 * rng.randint(4, 12)}
    if kind in ("double", "single", "denoise"):
        # Image sides in patches (16 pixels each): any aspect ratio.
        c = {"kind": kind, "img": rng.randint(16, 64) * rng.randint(16, 64), "txt": rng.choice([512, 512, rng.randint(16, 511)])}
        c["dim"], c["ff"] = rng.choice([(3072, 9216), (3072, 9216), (2048, 6144), (1536, 4096)])
        if kind == "denoise":
            c["double"], c["single"] = rng.randint(1, 5), rng.randint(1, 20)
        c["dtype"] = rng.choice(["f16", "f16", "bf16"])
        return c
    if kind == "matmul":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        return {"kind": kind, "m": _log(rng, 1, 16 if dtype == "f32" else 4608), "n": _log(rng, 256, 27648),
                "k": 64 * _log(rng, 2, 192), "dtype": dtype}
    if kind == "linear":
        return {"kind": kind, "m": _log(rng, 128, 4608), "n": 64 * _log(rng, 16, 288), "k": 64 * _log(rng, 16, 192),
                "dynamic": rng.random() < 0.3, "out16": rng.random() < 0.3}
    return {"kind": kind, "n": _log(rng, 512, 27648), "k": 64 * _log(rng, 8, 192), "dtype": rng.choice(["bf16", "bf16", "f16", "f32"])}


# ---- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _proj(g, n, k, dtype):
    """A packed projection whose outputs have the scale of its inputs."""
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), dtype=torch.int32, device="cuda", generator=g)
    unit = 1.0 / (4.0 * k ** 0.5)
    s = _randn(g, n, k // 64).abs() * unit
    b = -8.0 * s + _randn(g, n, k // 64) * (0.1 * unit)
    if dtype == torch.float32:  # float32 parameters hold the pack's bf16 values
        s, b = s.bfloat16(), b.bfloat16()
    return ops.Q(w=w, s=s.to(dtype), b=b.to(dtype), n=n, k=k)


def _layers_parts(case, seed):
    hidden, nq, nkv, inter = WIDTHS[case["width"]]
    t, g, m = DTYPES[case["dtype"]], _gen(seed), case["rows"]
    layers = []
    for _ in range(case["layers"]):
        layers.append(te_mod.TeLayer(
            qkv=_proj(g, nq + 2 * nkv, hidden, t), o=_proj(g, hidden, nq, t),
            gate_up=_proj(g, 2 * inter, hidden, t), down=_proj(g, hidden, inter, t),
            norm_in=1.0 + 0.1 * _randn(g, hidden), norm_post=1.0 + 0.1 * _randn(g, hidden)))
    # Each layer's own input and attention output, as its neighbours leave them.
    xs = [_randn(g, m, hidden).to(t) for _ in layers]
    attn = [_randn(g, m, nq).to(t) for _ in layers]
    return layers, xs, attn


def _block_dims(case):
    kind = case["kind"]
    return step_mod.DitDims(l_img=case["img"], l_txt=case["txt"], dim=case["dim"], ff_inner=case["ff"],
                            n_double=case.get("double", 1 if kind == "double" else 0),
                            n_single=case.get("single", 1 if kind == "single" else 0))


def _block_parts(case, seed):
    d, t, g = _block_dims(case), DTYPES[case["dtype"]], _gen(seed)
    projs = [_proj(g, n, k, t) for _, n, k in d.projection_shapes()]
    norm_w = 1.0 + 0.1 * _randn(g, d.dim)
    gates = 0.5 * _randn(g, 4 * d.n_double + d.n_single, d.dim)
    return d, t, g, projs, norm_w, gates


def _block_inputs(case, d, t, g):
    """The residual that reaches a block, its modulated norms and the attention output."""
    i = {"x0": _randn(g, d.joint, d.dim), "nx": _randn(g, d.joint, d.dim).to(t), "attn": _randn(g, d.joint, d.dim).to(t)}
    if case["kind"] == "double":
        i["nx2"] = _randn(g, d.joint, d.dim).to(t)
    return i


def _denoise_inputs(d, t, g):
    head = (_proj(g, d.dim, 128, t), _proj(g, 128, d.dim, t))
    return head, _randn(g, d.l_img, 128), _randn(g, d.l_txt, d.dim)


def _times(case, seed):
    """A schedule's timesteps, descending from 1000, moved a little by the seed."""
    n = case["count"]
    return [1000.0 * (n - i) / n - 0.5 * (seed % 97) / n for i in range(n)]


def _plain_parts(case, seed):
    """Packed projection and input of the kinds that run one projection."""
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        q = _proj(g, case["n"], case["k"], torch.float16)
        return q, 4.0 * _randn(g, case["m"], case["k"])
    t = DTYPES[case["dtype"]]
    if kind == "embed":
        q = _proj(g, case["rows"], case["k"], t)
        ids = torch.randint(0, case["rows"], (case["count"],), generator=torch.Generator().manual_seed(seed + 7))
        return q, ids
    q = _proj(g, case["n"], case["k"], t)
    return q, (_randn(g, case["m"], case["k"]).to(t) if kind == "matmul" else None)


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "layers":
        layers, st["x"], st["attn"] = _layers_parts(case, seed)
        st["plan"] = te_mod.TextEncoderLayers(layers, max_rows=512)
    elif kind == "chain":
        g, dim = _gen(seed), case["dim"]
        projs = [_proj(g, n, k, torch.float32) for n, k in ((dim, 256), (dim, dim), (17 * dim, dim))]
        st["plan"] = cond_mod.Conditioner(*projs)
        st["times"] = _times(case, seed)
    elif kind in ("double", "single", "denoise"):
        d, t, g, projs, norm_w, gates = _block_parts(case, seed)
        st["plan"] = step_mod.DitStep(d, projs)
        st["plan"].set_conditioning(norm_w, gates.contiguous())
        if kind == "denoise":
            head, st["lat"], st["e"] = _denoise_inputs(d, t, g)
            st["plan"].set_head(*head)
        else:
            st.update(_block_inputs(case, d, t, g))
            st["x"] = torch.empty_like(st["x0"])
            if kind == "double":
                st["qkv"] = [torch.empty((d.joint, d.dim), dtype=t, device="cuda") for _ in range(3)]
            else:
                st["qkv"] = torch.empty((d.joint, 3 * d.dim), dtype=t, device="cuda")
                st["concat"] = torch.cat([st.pop("attn"), torch.zeros((d.joint, d.ff_inner), dtype=t, device="cuda")], 1)
    else:
        q, st["in"] = _plain_parts(case, seed)
        st["q"] = q
        if kind == "linear":
            st["linear"] = ops.QuantizedLinear(q.w, q.s, q.b)
            st["target"] = 64.0 if case["dynamic"] else None
            st["out16"] = case["out16"]
    return st


def run(st):
    kind = st["kind"]
    if kind == "layers":
        out = []
        for i, (x, attn) in enumerate(zip(st["x"], st["attn"])):
            out.append({"qkv": st["plan"].attn_in(i, x), "y": st["plan"].attn_out_mlp(i, x, attn)})
        return out
    if kind == "embed":
        q = st["q"]
        return ops.dequantize_rows(q.w, q.s, q.b, st["in"])
    if kind == "chain":
        temb, heads = st["plan"].run(st["times"])
        return {"temb": temb, "heads": heads}
    if kind == "double":
        p, x = st["plan"], st["x"]
        x.copy_(st["x0"])  # the residual that the block before has left
        p.double_attn_in(0, None, *st["qkv"], nx=st["nx"])
        p.double_attn_out(0, st["attn"], x)
        p.double_mlp(0, x, nx=st["nx2"])
        return {"q": st["qkv"][0], "k": st["qkv"][1], "v": st["qkv"][2], "x": x}
    if kind == "single":
        p, x = st["plan"], st["x"]
        x.copy_(st["x0"])
        p.single_attn_in(0, None, st["qkv"], st["concat"], nx=st["nx"])
        p.single_attn_out(0, st["concat"], x)
        return {"qkv": st["qkv"], "concat": st["concat"], "x": x}
    if kind == "denoise":
        return st["plan"].denoise(st["lat"], st["e"], -0.25)
    q = st["q"]
    if kind == "matmul":
        return ops.quantized_matmul(st["in"], q.w, q.s, q.b)
    if kind == "linear":
        return ops.apply_linear(st["linear"], st["in"], output_f16=st["out16"], dynamic_target=st["target"])
    return ops.dequantize(q.w, q.s, q.b)


# ---- the same in 64 bits


def _codes(w):
    """[n, k] codes of packed words [n, k / 8], low nibble first."""
    shifts = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    return ((w.unsqueeze(-1) >> shifts) & 15).reshape(w.shape[0], -1)


def _wide(q, a=0, b=None):
    """Rows [a, b) of scale * code + bias in float64."""
    w, s, t = q.w[a:b], q.s[a:b].double(), q.b[a:b].double()
    c = _codes(w).double().reshape(w.shape[0], -1, 64)
    return (c.mul_(s.unsqueeze(-1)).add_(t.unsqueeze(-1))).reshape(w.shape[0], -1)


def _mm(x, q, a=0, b=None):
    """x . W^T in float64; the format holds a weight in its scales' type."""
    b = q.n if b is None else b
    cols = []
    for r in range(a, b, 8192):
        cols.append(x @ _wide(q, r, min(b, r + 8192)).to(q.s.dtype).double().T)
    return cols[0] if len(cols) == 1 else torch.cat(cols, 1)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _swiglu(x, q, width, gate, up):
    g = _mm(x, q, gate, gate + width)
    return g * torch.sigmoid(g) * _mm(x, q, up, up + width)


def _double_exact(d, w, g, x, attn, nx2):
    """The block's residual after attention and after its MLPs (nx2: the MLPs' input, or a function of x)."""
    t, i = slice(0, d.l_txt), slice(d.l_txt, d.joint)
    x[i] += g[0] * _mm(attn[i], w[6])
    x[t] += g[1] * _mm(attn[t], w[7])
    n = nx2(x)
    x[i] += g[2] * _mm(_swiglu(n[i], w[8], d.ff_inner, 0, d.ff_inner), w[9])
    x[t] += g[3] * _mm(_swiglu(n[t], w[10], d.ff_inner, 0, d.ff_inner), w[11])
    return x


def _qkv_exact(d, w, nx):
    return [torch.cat([_mm(nx[:d.l_txt], w[3 + j]), _mm(nx[d.l_txt:], w[j])]) for j in range(3)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "layers":
        out = []
        layers, xs, attn = _layers_parts(case, seed)
        inter = WIDTHS[case["width"]][3]
        for l, x, a in zip(layers, xs, attn):
            x = x.double()
            qkv = _mm(_rms(x, l.norm_in, te_mod.EPS), l.qkv)
            r = x + _mm(a.double(), l.o)
            m = _swiglu(_rms(r, l.norm_post, te_mod.EPS), l.gate_up, inter, 0, inter)
            out.append({"qkv": qkv, "y": r + _mm(m, l.down)})
        return out
    if kind == "chain":
        g, dim = _gen(seed), case["dim"]
        l1, l2, heads = [_proj(g, n, k, torch.float32) for n, k in ((dim, 256), (dim, dim), (17 * dim, dim))]
        # The sinusoid is float32 by definition: its largest angle, 1000, keeps
        # about 1e-5 of a turn.
        i = torch.arange(128, dtype=torch.float32)
        freq = torch.exp(-torch.log(torch.tensor(10000.0)) * i / 128.0)
        arg = (torch.tensor(_times(case, seed), dtype=torch.float32)[:, None] * freq).double()
        sin = torch.cat([arg.cos(), arg.sin()], 1).cuda()
        h = _mm(sin, l1)
        temb = _mm(h * torch.sigmoid(h), l2)
        return {"temb": temb, "heads": _mm(temb * torch.sigmoid(temb), heads)}
    if kind in ("double", "single", "denoise"):
        d, t, g, projs, norm_w, gates = _block_parts(case, seed)
        gates = gates.double()
        if kind == "double":
            i = _block_inputs(case, d, t, g)
            q, k, v = _qkv_exact(d, projs, i["nx"].double())
            x = _double_exact(d, projs, gates, i["x0"].double(), i["attn"].double(), lambda x: i["nx2"].double())
            return {"q": q, "k": k, "v": v, "x": x}
        if kind == "single":
            i = _block_inputs(case, d, t, g)
            nx = i["nx"].double()
            mlp = _swiglu(nx, projs[0], d.ff_inner, 3 * d.dim, 3 * d.dim + d.ff_inner)
            concat = torch.cat([i["attn"].double(), mlp], 1)
            return {"qkv": _mm(nx, projs[0], 0, 3 * d.dim), "concat": concat,
                    "x": i["x0"].double() + gates[0] * _mm(concat, projs[1])}
        head, lat, e = _denoise_inputs(d, t, g)
        x = torch.cat([e.double(), _mm(lat.double(), head[0])])
        # Without an attention core a step takes the values for the attention's
        # output in double blocks and zeros in single ones.
        for b in range(d.n_double):
            w = projs[12 * b:12 * b + 12]
            n = _rms(x, norm_w, 1e-5)
            v = torch.cat([_mm(n[:d.l_txt], w[5]), _mm(n[d.l_txt:], w[2])])
            x = _double_exact(d, w, gates[4 * b:4 * b + 4], x, v, lambda x: _rms(x, norm_w, 1e-5))
        for b in range(d.n_single):
            w = projs[12 * d.n_double + 2 * b:12 * d.n_double + 2 * b + 2]
            mlp = _swiglu(_rms(x, norm_w, 1e-5), w[0], d.ff_inner, 3 * d.dim, 3 * d.dim + d.ff_inner)
            concat = torch.cat([torch.zeros((d.joint, d.dim), dtype=torch.float64, device="cuda"), mlp], 1)
            x += gates[4 * d.n_double + b] * _mm(concat, w[1])
        return lat.double() - 0.25 * _mm(_rms(x[d.l_txt:], norm_w, 1e-5), head[1])
    q, x = _plain_parts(case, seed)
    if kind == "embed":
        rows = x.cuda()
        return _wide(ops.Q(w=q.w[rows], s=q.s[rows], b=q.b[rows], n=len(rows), k=q.k))
    if kind == "dequant":
        return _wide(q)
    return _mm(x.double(), q)


# ---- what a pass cannot do without


def _weight_bytes(n, k, size):
    """Codes, and a scale and a bias per 64 inputs."""
    return n * k // 2 + 2 * size * n * (k // 64)


def work(case):
    kind = case["kind"]
    size = {"bf16": 2, "f16": 2, "f32": 4}[case.get("dtype", "f32")]
    if kind == "layers":
        hidden, nq, nkv, inter = WIDTHS[case["width"]]
        m = case["rows"]
        shapes = [(nq + 2 * nkv, hidden), (hidden, nq), (2 * inter, hidden), (hidden, inter)]
        byts = sum(_weight_bytes(n, k, 2) for n, k in shapes) + 8 * hidden
        byts += 2 * m * (2 * hidden + 2 * nq + 2 * nkv)  # x and attention in, qkv and y out
        return {"bytes": case["layers"] * byts, "flops": case["layers"] * sum(2 * m * n * k for n, k in shapes)}
    if kind == "embed":
        return {"bytes": case["count"] * (_weight_bytes(1, case["k"], size) + case["k"] * size + 8),
                "flops": 2 * case["count"] * case["k"]}
    if kind == "chain":
        dim, m = case["dim"], case["count"]
        shapes = [(dim, 256), (dim, dim), (17 * dim, dim)]
        passes = sum(2 * m * n * k for n, k in shapes)
        return {"bytes": sum(_weight_bytes(n, k, 4) for n, k in shapes) + 4 * m * 18 * dim, "flops": passes}
    if kind in ("double", "single", "denoise"):
        d = _block_dims(case)
        shapes = d.projection_shapes()
        byts = sum(_weight_bytes(n, k, 2) for _, n, k in shapes)
        flops = sum(2 * d.rows_of(name) * n * k for name, n, k in shapes)
        j, dim = d.joint, d.dim
        if kind == "double":  # x in and out, nx, nx2 and attention in, q, k and v out
            byts += j * dim * (4 + 4 + 2 * 3 + 2 * 3)
        elif kind == "single":  # x in and out, nx and attention in, qkv and the MLP half out
            byts += j * (dim * (4 + 4 + 2 + 2 + 6) + 2 * d.ff_inner)
        else:
            byts += 2 * _weight_bytes(dim, 128, 2) + 4 * (2 * d.l_img * 128 + d.l_txt * dim)
            flops += 2 * 2 * d.l_img * dim * 128
        return {"bytes": byts, "flops": flops}
    n, k = case["n"], case["k"]
    if kind == "dequant":
        return {"bytes": _weight_bytes(n, k, size) + n * k * size, "flops": 2 * n * k}
    m = case["m"]
    if kind == "linear":
        return {"bytes": _weight_bytes(n, k, 2) + 4 * m * k + (2 if case["out16"] else 4) * m * n, "flops": 2 * m * n * k}
    return {"bytes": _weight_bytes(n, k, size) + size * m * (n + k), "flops": 2 * m * n * k}


def tolerance(case):
    """About four times the error against 64 bits that was measured, which is what
    rounding to the case's type gives (an output's own rounding alone is 1.7e-3
    in bf16, 2.1e-4 in f16); expanded weights have one right value."""
    kind, t = case["kind"], case.get("dtype")
    if kind in ("embed", "dequant"):
        return "exact"
    if kind == "chain":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "linear":
        return {"rel": 1.2e-3, "max": 1e-2}
    if kind == "layers":
        return {"rel": 1.2e-2, "max": 8e-2} if t == "bf16" else {"rel": 1.5e-3, "max": 1e-2}
    if kind in ("double", "single"):
        return {"rel": 1.2e-2, "max": 8e-2} if t == "bf16" else {"rel": 1.5e-3, "max": 1e-2}
    if kind == "denoise":
        return {"rel": 8e-3, "max": 6e-2} if t == "bf16" else {"rel": 1e-3, "max": 1e-2}
    return {"bf16": {"rel": 7e-3, "max": 4e-2}, "f16": {"rel": 1e-3, "max": 6e-3}, "f32": {"rel": 1e-5, "max": 1e-4}}[t]
