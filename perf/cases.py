"""The work that a program using this package has it do: one case per public entry point of the Q8_0 linear path and
of what sits between its products, and two whole calls (a Gaussian decoder, a denoiser step).

A case names its entry point in "op" and gives its sizes. listed() holds the sizes of the package's own configurations
and benchmark beside small and ragged ones; draw() spreads the same entry points over the ranges around them. Weights
are drawn N(0, std), inputs N(0, 1), everything on the GPU from the seed; the Q8_0 blocks are made here in plain torch,
so that exact() computes each result in 64 bits without the package.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "idol.cpp_amd"))

import idol_export as E  # noqa: E402
import idol_kernels as K  # noqa: E402
import idolq_lib as L  # noqa: E402
from decoder_mlp import FEAT, HIDDEN, MID, NFREQ, OUT  # noqa: E402
from decoders import Decoders  # noqa: E402
from denoiser import CTX_DIM, HEAD_DIM, DenoiserLayer, SyntheticDenoiser  # noqa: E402
from ggml_types import GGMLQuantizationType  # noqa: E402
from idol_packed import PackedLinear, enable_fused_packed  # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
KINDS = {"q8_0": GGMLQuantizationType.Q8_0, "q4_0": GGMLQuantizationType.Q4_0, "q4_k": GGMLQuantizationType.Q4_K}
BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144)}


def listed():
    return [
        # one token through a packed layer: the smallest call, weights read once, latency and launch counts
        dict(name="linear_token", op="linear", kind="q8_0", dtype="bf16", m=1, n=4096, k=4096, bias=True),
        # a short prompt through a packed layer in the other fused format and half type; rows fill no tile
        dict(name="linear_ragged", op="linear", kind="q4_k", dtype="fp16", m=333, n=4608, k=1536, bias=True),
        # the denoiser's MLP over one sequence: up projection with GELU, down projection with the residual
        dict(name="mlp_block", op="mlp", dtype="bf16", m=4096, dim=1536, hidden=6144),
        # the denoiser's self-attention, both guidance branches, on views of the fused projection
        dict(name="attention_self", op="attention", dtype="bf16", batch=2, heads=24, lq=4096, lk=4096),
        # the real decoders' cross-attention in fp32: anchors over latent tokens, a ragged number of anchors
        dict(name="attention_decoder", op="attention_f32", heads=16, hd=64, lq=1000, lk=8192),
        # the denoiser's modulated layer norm
        dict(name="norm", op="norm", dtype="bf16", form="ada", batch=2, rows=8192, dim=1536),
        # the decoders' up projection with the float kernel (erf-GELU epilogue)
        dict(name="packed_float", op="packed", kernel="float", m=1024, n=4096, k=1024, gelu=True, residual=False),
        # the decoders' down projection with the integer kernel, the package's default, residual added; ragged rows
        dict(name="packed_int8", op="packed", kernel="int8", m=1000, n=1024, k=4096, gelu=False, residual=True),
        # the per-point head over a whole grid of query points
        dict(name="points", op="points", m=262144),
        # writing a weight as Q8_0 blocks and expanding a packed layer (the route of layers that are not fused)
        dict(name="weights", op="weights", kind="q8_0", dtype="bf16", n=6144, k=1536),
        # a whole call: the Gaussian decoder at the real model's width and latent size, two blocks
        dict(name="decoder", op="decoder", part="gaussian", dim=1024, heads=16, blocks=2, rows=1024, tokens=8192),
        # a whole call: a denoiser step of two layers, both guidance branches at the full sequence length
        dict(name="denoiser", op="denoiser", layers=2, batch=2, seq=4096, ctx=1024, heads=24),
    ]


def draw(rng):
    def log(lo, hi, step=1):
        return max(step, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)

    op = rng.choice(("linear", "linear", "mlp", "attention", "attention_f32", "norm", "packed", "packed", "points",
                     "weights", "decoder", "denoiser"))
    if op == "linear":
        kind = rng.choice(("q8_0", "q8_0", "q4_0", "q4_k"))
        step = 256 if kind == "q4_k" else rng.choice((32, 64, 256))
        return dict(op=op, kind=kind, dtype=rng.choice(("bf16", "fp16")), m=log(1, 4096), n=log(200, 6144),
                    k=log(512, 4096, step), bias=rng.random() < 0.7)
    if op == "mlp":
        dim = rng.choice((768, 1024, 1536))
        return dict(op=op, dtype=rng.choice(("bf16", "bf16", "fp16")), m=log(64, 8192), dim=dim, hidden=4 * dim)
    if op == "attention":
        lq = log(64, 4096)
        return dict(op=op, dtype=rng.choice(("bf16", "fp16")), batch=rng.choice((1, 2)), heads=rng.choice((8, 12, 16, 24)),
                    lq=lq, lk=lq if rng.random() < 0.5 else log(64, 4096))
    if op == "attention_f32":
        hd = rng.choice((64, 64, 32))
        lq = log(32, 2048)
        return dict(op=op, heads=rng.choice((8, 16)), hd=hd, lq=lq, lk=lq if rng.random() < 0.3 else log(64, 8192))
    if op == "norm":
        batch = rng.choice((1, 2))
        return dict(op=op, dtype=rng.choice(("bf16", "fp16", "fp32")), form=rng.choice(("plain", "affine", "ada")),
                    batch=batch, rows=batch * log(64, 8192), dim=rng.choice((768, 1000, 1024, 1536, 2048)))
    if op == "packed":
        k = rng.choice((512, 1024, 2048, 4096))
        return dict(op=op, kernel=rng.choice(("float", "int8")), m=log(1, 4096), n=log(200, 4096), k=k,
                    gelu=rng.random() < 0.5, residual=rng.random() < 0.5)
    if op == "points":
        return dict(op=op, m=log(256, 262144))
    if op == "weights":
        kind = rng.choice(("q8_0", "q4_0", "q4_k"))
        return dict(op=op, kind=kind, dtype=rng.choice(("bf16", "fp16", "fp32")), n=log(256, 6144),
                    k=log(512, 4096, 256))
    if op == "decoder":
        return dict(op=op, part=rng.choice(("octree", "gaussian")), dim=rng.choice((512, 1024)), heads=16,
                    blocks=rng.choice((1, 2)), rows=log(64, 1024), tokens=log(256, 8192))
    return dict(op=op, layers=rng.choice((1, 2)), batch=rng.choice((1, 2)), seq=log(64, 4096), ctx=log(64, 1024),
                heads=rng.choice((8, 16, 24)))


# ---------------------------------------------------------------------------------------------- weights and inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(shape, device=DEV, generator=gen)


def _q8_0(w):
    """GGUF Q8_0 blocks (uint8 [n, k / 32, 34]) of an fp32 matrix: d = amax / 127, q = x / d rounded half away."""
    n, k = w.shape
    b = w.reshape(n, k // 32, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    x = b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    q = torch.trunc(x + torch.copysign(torch.full_like(x, 0.5), x)).to(torch.int8)
    return torch.cat([d.half().view(torch.uint8), q.view(torch.uint8)], dim=-1)


def _blocks(gen, kind, n, k, std):
    """Packed bytes [n, blocks, block bytes] of a random matrix of about this standard deviation."""
    if kind == "q8_0":
        return _q8_0(_randn(gen, n, k) * std)
    values, size = BLOCK[kind]
    b = torch.randint(0, 256, (n, k // values, size), device=DEV, generator=gen, dtype=torch.int32).to(torch.uint8)
    d = std * (0.5 + torch.rand((n, k // values, 1), device=DEV, generator=gen))
    if kind == "q4_0":  # 4-bit codes around 8: standard deviation 4.6
        b[:, :, :2] = (d / 4.6).half().view(torch.uint8)
    else:  # 6-bit scales about 31 times 4-bit codes about 7.5, less the minimums
        d = d / (31.0 * 4.6)
        b[:, :, :2] = d.half().view(torch.uint8)
        b[:, :, 2:4] = (7.5 * d).half().view(torch.uint8)
    return b


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _values(b, kind="q8_0"):
    """The fp64 matrix of packed bytes [n, blocks, block bytes]."""
    n = b.shape[0]
    if kind == "q8_0":
        return (_half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, -1)
    if kind == "q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], dim=-1).double() - 8.0
        return (_half(b[..., :2]) * q).reshape(n, -1)
    s = b[..., 4:16].to(torch.int32)
    lo, mid, hi = s[..., 0:4], s[..., 4:8], s[..., 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], dim=-1)
    mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], dim=-1)
    codes = b[..., 16:].reshape(*b.shape[:2], 4, 32)
    q = torch.stack([codes & 15, codes >> 4], dim=3).reshape(*b.shape[:2], 8, 32).double()
    d = _half(b[..., :2]) * sc.double()
    m = _half(b[..., 2:4]) * mn.double()
    return (d.unsqueeze(-1) * q - m.unsqueeze(-1)).reshape(n, -1)


class _Source:
    """A packed matrix as a GGUF reader hands it over."""

    def __init__(self, b, kind, n, k):
        self.shape, self.tensor_type, self.data = np.array([k, n]), KINDS[kind], b.cpu().numpy()


def _inputs(case, seed):
    """Everything of a case that is drawn, from the seed alone: what prepare() lays out and exact() computes with."""
    gen = _gen(seed)
    op = case["op"]
    if op == "linear":
        dt = DTYPES[case["dtype"]]
        return dict(b=_blocks(gen, case["kind"], case["n"], case["k"], 0.02),
                    x=_randn(gen, case["m"], case["k"]).to(dt),
                    bias=(_randn(gen, case["n"]) * 0.01).to(dt) if case["bias"] else None)
    if op == "mlp":
        d, h = case["dim"], case["hidden"]
        return dict(up=_blocks(gen, "q8_0", h, d, 0.02), down=_blocks(gen, "q8_0", d, h, 0.02),
                    up_b=_randn(gen, h) * 0.01, down_b=_randn(gen, d) * 0.01,
                    x=_randn(gen, case["m"], d).to(DTYPES[case["dtype"]]))
    if op == "attention":
        B, D, dt = case["batch"], case["heads"] * HEAD_DIM, DTYPES[case["dtype"]]
        if case["lq"] == case["lk"]:  # one fused projection
            qkv = _randn(gen, B * case["lq"], 3 * D).to(dt)
            return dict(q=qkv[:, :D], k=qkv[:, D:2 * D], v=qkv[:, 2 * D:])
        q = _randn(gen, B * case["lq"], D).to(dt)
        kv = _randn(gen, B * case["lk"], 2 * D).to(dt)
        return dict(q=q, k=kv[:, :D], v=kv[:, D:])
    if op == "attention_f32":
        D = case["heads"] * case["hd"]
        kv = _randn(gen, case["lk"], 2 * D)
        return dict(q=_randn(gen, case["lq"], D), k=kv[:, :D], v=kv[:, D:])
    if op == "norm":
        dim, form = case["dim"], case["form"]
        r = dict(x=_randn(gen, case["rows"], dim).to(DTYPES[case["dtype"]]))
        if form == "affine":
            r.update(gamma=1.0 + 0.1 * _randn(gen, dim), beta=0.1 * _randn(gen, dim))
        if form == "ada":
            r.update(shift=0.1 * _randn(gen, case["batch"], dim), scale=0.1 * _randn(gen, case["batch"], dim),
                     rows_per_batch=case["rows"] // case["batch"])
        return r
    if op == "packed":
        return dict(b=_blocks(gen, "q8_0", case["n"], case["k"], 0.02), bias=_randn(gen, case["n"]) * 0.01,
                    x=_randn(gen, case["m"], case["k"]),
                    residual=_randn(gen, case["m"], case["n"]) if case["residual"] else None)
    if op == "points":
        m = case["m"]
        k1 = FEAT + 6 * NFREQ
        w = [_values(_blocks(gen, "q8_0", n, k, 0.05)).bfloat16() for n, k in ((HIDDEN, k1), (HIDDEN, HIDDEN), (MID, HIDDEN))]
        return dict(w=w, b=[_randn(gen, n) * 0.01 for n in (HIDDEN, HIDDEN, MID)], wh=_randn(gen, OUT, MID) * 0.05,
                    bh=_randn(gen, OUT) * 0.01, freqs=torch.pow(2.0, torch.linspace(0.0, 10.0, NFREQ)).to(DEV),
                    feats=_randn(gen, m, FEAT), coords=torch.rand((m, 3), device=DEV, generator=gen) * 2.0 - 1.0)
    if op == "weights":
        return dict(w=_randn(gen, case["n"], case["k"]) * 0.02, b=_blocks(gen, case["kind"], case["n"], case["k"], 0.02))
    if op == "decoder":
        D, rows = case["dim"], case["rows"]
        r = {}

        def lin(name, out, in_):  # matrices as Q8_0 blocks, the narrow input projections in fp32
            w = _randn(gen, out, in_) / math.sqrt(in_)
            r[name] = (_q8_0(w) if in_ % 256 == 0 else w, 0.02 * _randn(gen, out))

        def attn(p, cross):
            if cross:
                lin(p + ".to_q", D, D)
                lin(p + ".to_kv", 2 * D, 16)
            else:
                lin(p + ".to_qkv", 3 * D, D)
            lin(p + ".to_out", D, D)
            for g in ("q", "k"):
                r[f"{p}.{g}_rms_norm.gamma"] = 1.0 + 0.1 * _randn(gen, D)

        octree = case["part"] == "octree"
        lin("oct.in_proj", D, 3)
        lin("oct.input_layer", D, D)
        lin("oct.l_embedder.mlp.0", D, 256)
        lin("oct.l_embedder.mlp.2", D, D)
        lin("oct.adaLN_modulation.1", 6 * D, D)
        lin("oct.out_proj", 8, D)
        lin("gs.in_proj", D, 3)
        lin("gs.input_layer", D, D)
        lin("gs.out_proj", 32 * 15, D)
        for i in range(case["blocks"]):
            p = f"oct.blocks.{i}." if octree else f"gs.blocks.{i}."
            if not octree:
                attn(p + "self_attn", False)
                r[p + "norm2.weight"] = 1.0 + 0.1 * _randn(gen, D)
                r[p + "norm2.bias"] = 0.05 * _randn(gen, D)
            attn(p + "cross_attn", True)
            lin(p + "mlp.mlp.0", 4 * D, D)
            lin(p + "mlp.mlp.2", D, 4 * D)
        fd = D // 3 // 2
        freqs = torch.pow(2.0, torch.linspace(0.0, 10.0, fd)).to(DEV)
        r["oct.pos_embedder.freqs"] = r["gs.pos_embedder.freqs"] = freqs
        r["oct.l_embedder.freqs"] = torch.exp(-math.log(1024) * torch.arange(0, 128) / 128.0).to(DEV)
        r["gs.points_offset_perturbation"] = 0.1 * _randn(gen, 96)
        r["gs.base_offset_scale"] = torch.full((1,), 0.5, device=DEV)
        return dict(export=r, x=torch.rand((rows, 3), device=DEV, generator=gen) - 0.5, cond=_randn(gen, case["tokens"], 16))
    D = case["heads"] * HEAD_DIM
    shapes = {"qkv": (3 * D, D), "out": (D, D), "cq": (D, D), "ckv": (2 * D, CTX_DIM), "cout": (D, D),
              "up": (4 * D, D), "down": (D, 4 * D)}
    layers = [{s: (_blocks(gen, "q8_0", n, k, 0.02), _randn(gen, n) * 0.01) for s, (n, k) in shapes.items()}
              for _ in range(case["layers"])]
    B = case["batch"]
    return dict(layers=layers, shift=0.1 * _randn(gen, B, D), scale=0.1 * _randn(gen, B, D),
                x=_randn(gen, B * case["seq"], D).bfloat16(), ctx=_randn(gen, B * case["ctx"], CTX_DIM).bfloat16())


# ------------------------------------------------------------------------------------------------- the entry points
def prepare(case, seed):
    i, op = _inputs(case, seed), case["op"]
    s = dict(case=case, op=op)
    if op == "linear":
        layer = PackedLinear(_Source(i["b"], case["kind"], case["n"], case["k"]), i["bias"]).to(DEV)
        enable_fused_packed(layer)
        s.update(layer=layer, x=i["x"])
    elif op == "mlp":
        m, d, h = case["m"], case["dim"], case["hidden"]
        s.update(up=L.tile_q8_0(i["up"].reshape(-1), h, d), down=L.tile_q8_0(i["down"].reshape(-1), d, h),
                 up_b=i["up_b"], down_b=i["down_b"], x=i["x"], f=i["x"].new_empty(m, h), y=torch.empty_like(i["x"]))
    elif op in ("attention", "attention_f32"):
        s.update(i, out=torch.empty(i["q"].shape, device=DEV, dtype=i["q"].dtype))
    elif op == "norm":
        s.update(x=i.pop("x"), args=i)
        s["out"] = torch.empty_like(s["x"])
    elif op == "packed":
        s.update(w=K.q8_0_linear(i["b"], i["bias"].cpu().numpy(), case["n"], case["k"]), x=i["x"], residual=i["residual"],
                 out=torch.empty((case["m"], case["n"]), device=DEV))
    elif op == "points":
        s.update(i, w=L.point_mlp_pack(*i["w"]))
    elif op == "weights":
        s.update(w=i["w"], layer=PackedLinear(_Source(i["b"], case["kind"], case["n"], case["k"]), None).to(DEV))
    elif op == "decoder":
        octree = case["part"] == "octree"
        cfg = E.DecoderConfig(dim=case["dim"], heads=case["heads"], oct_blocks=case["blocks"] if octree else 0,
                              gs_blocks=0 if octree else case["blocks"], cond=16, per_anchor=32)
        ex = E.Export(decoders=True, decoder_config=cfg)
        for name, v in i["export"].items():
            if not isinstance(v, tuple):
                ex.tensors[name] = E.Tensor([v.numel()], v.cpu().numpy())
                continue
            w, b = v
            if w.dtype == torch.uint8:
                ex.qtensors[name + ".weight"] = E.QTensor(w.shape[0], w.shape[1] * 32, 8, 32, w.reshape(-1), kind="q8_0")
            else:
                ex.tensors[name + ".weight"] = E.Tensor(list(w.shape), w.cpu().numpy().reshape(-1))
            ex.tensors[name + ".bias"] = E.Tensor([b.numel()], b.cpu().numpy())
        s.update(dec=Decoders(ex), x=i["x"], cond=i["cond"])
    else:
        D = case["heads"] * HEAD_DIM
        layers = []
        for given in i["layers"]:
            layer = DenoiserLayer(_gen(seed), DEV, D, 4 * D, CTX_DIM)
            for name, (b, bias) in given.items():
                layer.w[name], layer.b[name] = b.reshape(-1), bias
                layer.wt[name] = L.tile_q8_0(layer.w[name], *layer.shape[name])
            layers.append(layer)
        model = SyntheticDenoiser(layers, case["batch"], case["seq"], case["ctx"], case["heads"], HEAD_DIM, 4 * D)
        model.shift, model.scale = i["shift"], i["scale"]
        model.batch_context_kv()
        s.update(model=model, x0=i["x"], x=torch.empty_like(i["x"]), ctx=i["ctx"])
    return s


def run(s):
    c, op = s["case"], s["op"]
    if op == "linear":
        return s["layer"](s["x"])
    if op == "mlp":
        f = L.gemm(s["x"], s["up"], c["hidden"], bias=s["up_b"], act=L.ACT_GELU_TANH, mode=L.MODE_DEQUANT, out=s["f"],
                   tiled=True, split=True)
        y = L.gemm(f, s["down"], c["dim"], bias=s["down_b"], residual=s["x"], mode=L.MODE_DEQUANT, out=s["y"],
                   tiled=True, split=True)
        return f, y
    if op == "attention":
        D, lq, lk = c["heads"] * HEAD_DIM, c["lq"], c["lk"]
        ldq, ldkv = s["q"].stride(0), s["k"].stride(0)
        return L.attention(s["q"], s["k"], s["v"], c["batch"], lq, lk, c["heads"], HEAD_DIM, ldq, ldkv, lq * ldq,
                           lk * ldkv, s["out"], D, lq * D)
    if op == "attention_f32":
        D = c["heads"] * c["hd"]
        return K.attention(s["q"], c["lq"], D, s["k"], s["v"], c["lk"], 2 * D, c["heads"], c["hd"], s["out"], D)
    if op == "norm":
        return L.layernorm(s["x"], 1e-6, out=s["out"], **s["args"])
    if op == "packed":
        K.set_quant_kernel(1 if c["kernel"] == "int8" else 0)
        return K.gemm_packed(s["x"], c["m"], s["w"], 0, c["n"], s["residual"], c["gelu"], s["out"])
    if op == "points":
        w, b = s["w"], s["b"]
        return L.point_mlp(s["feats"], s["coords"], s["freqs"], w[0], b[0], w[1], b[1], w[2], b[2], s["wh"], s["bh"])
    if op == "weights":
        return L.quantize_q8_0(s["w"]), s["layer"].dequantize(DTYPES[c["dtype"]])
    if op == "decoder":
        K.set_quant_kernel(0)
        if c["part"] == "octree":
            return s["dec"].octree_logits(s["x"], c["rows"], 64.0, s["cond"], c["tokens"])
        return s["dec"].gaussian_features(s["x"], c["rows"], s["cond"], c["tokens"])
    s["x"].copy_(s["x0"])
    return s["model"].step(s["x"], s["ctx"])


# ------------------------------------------------------------------------------------------------- work and bounds
def work(c):
    op = c["op"]
    if op == "linear":
        values, size = BLOCK[c["kind"]]
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=n * k // values * size + 2 * m * (n + k) + (2 * n if c["bias"] else 0), flops=2 * m * n * k)
    if op == "mlp":
        m, d, h = c["m"], c["dim"], c["hidden"]
        return dict(bytes=2 * d * h * 34 // 32 + 2 * m * (d + h + d) + 4 * (d + h), flops=4 * m * d * h)
    if op in ("attention", "attention_f32"):
        B, size = c.get("batch", 1), 4 if op == "attention_f32" else 2
        D = c["heads"] * c.get("hd", HEAD_DIM)
        return dict(bytes=size * B * D * 2 * (c["lq"] + c["lk"]), flops=4 * B * D * c["lq"] * c["lk"])
    if op == "norm":
        size = 4 if c["dtype"] == "fp32" else 2
        params = {"plain": 0, "affine": 2, "ada": 2 * c["batch"]}[c["form"]]
        return dict(bytes=2 * size * c["rows"] * c["dim"] + 4 * params * c["dim"], flops=8 * c["rows"] * c["dim"])
    if op == "packed":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=n * k * 34 // 32 + 4 * (m * k + m * n * (2 if c["residual"] else 1) + n), flops=2 * m * n * k)
    if op == "points":
        m, k1 = c["m"], FEAT + 6 * NFREQ
        weights = k1 * HIDDEN + HIDDEN * HIDDEN + HIDDEN * MID
        return dict(bytes=m * 4 * (FEAT + 3 + OUT) + 2 * weights, flops=2 * m * (weights + MID * OUT))
    if op == "weights":
        values, size = BLOCK[c["kind"]]
        nk = c["n"] * c["k"]
        return dict(bytes=nk * (4 + 34 / 32 + size / values + (4 if c["dtype"] == "fp32" else 2)), flops=3 * nk)
    if op == "decoder":
        D, rows, tok, nb = c["dim"], c["rows"], c["tokens"], c["blocks"]
        octree = c["part"] == "octree"
        outs = 8 if octree else 480
        params = nb * (D * D * (10 if octree else 14) + 2 * D * 16) + D * (D + 3 + outs)
        attn = 4 * D * rows * tok + (0 if octree else 4 * D * rows * rows)
        flops = 2 * rows * D * (D * (10 if octree else 14)) * nb + 2 * tok * 2 * D * 16 * nb + attn * nb
        flops += 2 * rows * D * (D + 3 + outs)
        if octree:
            params += D * (256 + 7 * D)
            flops += 2 * D * (256 + 7 * D)
        return dict(bytes=params * 34 // 32 + 4 * (rows * (3 + outs) + tok * 16), flops=flops)
    B, S, C, D, nl = c["batch"], c["seq"], c["ctx"], c["heads"] * HEAD_DIM, c["layers"]
    gemm = 2 * B * S * D * 14 * D + 2 * B * C * CTX_DIM * 2 * D
    attn = 4 * B * D * S * (S + C)
    return dict(bytes=nl * (14 * D * D + 2 * D * CTX_DIM) * 34 // 32 + 2 * B * (2 * S * D + C * CTX_DIM),
                flops=nl * (gemm + attn))


def tolerance(c):
    """About four times the error against exact() that the sizes here show: the rounding of 16-bit values and results
    (bf16 1.7e-3 a result, fp16 2.1e-4), 32-bit sums elsewhere."""
    op, half = c["op"], c.get("dtype") == "fp16"
    if op == "weights":
        return "exact"  # block bytes, and each expanded value rounded once
    if op == "norm" and c["dtype"] == "fp32":
        return {"rel": 1e-6}
    if op in ("norm", "attention"):
        return {"rel": 1e-3 if half else 7e-3}
    if op in ("linear", "mlp"):
        return {"rel": 1.5e-3 if half else 1.2e-2}
    if op == "attention_f32":
        return {"rel": 4e-6}
    if op == "packed":
        return {"rel": 2e-6 if c["kernel"] == "int8" else 1e-5}  # int8: exact dots; float: 16-bit halves of inputs
    if op == "decoder":
        return {"rel": 2e-5}
    return {"rel": 1.6e-2 if op == "points" else 2e-2}  # bf16 through three layers, through whole blocks


# ------------------------------------------------------------------------------------------------- in 64 bits
def _gelu_erf(v):
    return 0.5 * v * (1.0 + torch.erf(v / math.sqrt(2.0)))


def _gelu_tanh(v):
    return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))


def _norm(x, eps):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + eps)


def _attention(q, k, v, batch, heads):
    """Per head softmax(q k^T / sqrt(d)) v over rows [batch * l, heads * d]."""
    out = torch.empty(q.shape, device=DEV, dtype=torch.float64)
    lq, lk, d = q.shape[0] // batch, k.shape[0] // batch, q.shape[1] // heads
    for b in range(batch):
        for h in range(heads):
            at = slice(h * d, (h + 1) * d)
            qr, kr = slice(b * lq, (b + 1) * lq), slice(b * lk, (b + 1) * lk)
            p = torch.softmax(q[qr, at].double() @ k[kr, at].double().t().contiguous() / math.sqrt(d), dim=-1)
            out[qr, at] = p @ v[kr, at].double()
    return out


def _angles(x, freqs):
    """The embedding's angles (v f) pi as fp32 products, which define them: frequencies reach 2^10."""
    return ((x.unsqueeze(-1) * freqs) * torch.tensor(math.pi, device=DEV)).double()


def _embed(x, freqs):
    a = _angles(x, freqs)
    return torch.cat([torch.sin(a), torch.cos(a)], dim=-1).reshape(x.shape[0], -1)


def _exact_decoder(case, i):
    r, rows, heads = i["export"], case["rows"], case["heads"]
    D, cond = case["dim"], i["cond"].double()
    hd = D // heads

    def lin(name, a):
        w, b = r[name]
        return a @ (_values(w) if w.dtype == torch.uint8 else w.double()).t().contiguous() + b.double()

    def rms(name, a):
        a = a.reshape(-1, heads, hd)
        a = a / a.norm(dim=-1, keepdim=True) * math.sqrt(hd)
        return a.reshape(-1, D) * r[name].double()

    def cross(p, h):
        kv = lin(p + ".to_kv", cond)
        a = _attention(rms(p + ".q_rms_norm.gamma", lin(p + ".to_q", h)), rms(p + ".k_rms_norm.gamma", kv[:, :D]),
                       kv[:, D:], 1, heads)
        return lin(p + ".to_out", a)

    octree = case["part"] == "octree"
    part = "oct" if octree else "gs"
    x = lin(part + ".in_proj", i["x"].double())
    e = _embed(i["x"], r[part + ".pos_embedder.freqs"])
    x[:, :e.shape[1]] += e
    x = lin(part + ".input_layer", x)
    if octree:
        a = (((64.0 * r["oct.l_embedder.freqs"]) * 2.0) * torch.tensor(math.pi, device=DEV)).double()
        silu = torch.nn.functional.silu
        e = silu(lin("oct.l_embedder.mlp.0", torch.cat([torch.cos(a), torch.sin(a)]).reshape(1, -1)))
        mod = lin("oct.adaLN_modulation.1", silu(lin("oct.l_embedder.mlp.2", e))).reshape(6, D)
    for n in range(case["blocks"]):
        p = f"{part}.blocks.{n}."
        if octree:
            x = x + mod[2] * cross(p + "cross_attn", _norm(x, 1e-6) * (1.0 + mod[1]) + mod[0])
            h = _norm(x, 1e-6) * (1.0 + mod[4]) + mod[3]
            x = x + mod[5] * lin(p + "mlp.mlp.2", _gelu_tanh(lin(p + "mlp.mlp.0", h)))
            continue
        qkv = lin(p + "self_attn.to_qkv", _norm(x, 1e-6))
        a = _attention(rms(p + "self_attn.q_rms_norm.gamma", qkv[:, :D]),
                       rms(p + "self_attn.k_rms_norm.gamma", qkv[:, D:2 * D]), qkv[:, 2 * D:], 1, heads)
        x = x + lin(p + "self_attn.to_out", a)
        x = x + cross(p + "cross_attn", _norm(x, 1e-6) * r[p + "norm2.weight"].double() + r[p + "norm2.bias"].double())
        x = x + lin(p + "mlp.mlp.2", _gelu_tanh(lin(p + "mlp.mlp.0", _norm(x, 1e-6))))
    return lin(part + ".out_proj", _norm(x, 1e-5))


def _exact_denoiser(case, i):
    x, ctx, B = i["x"].double(), i["ctx"].double(), case["batch"]
    D = x.shape[1]
    shift, scale = (v.double().repeat_interleave(case["seq"], 0) for v in (i["shift"], i["scale"]))
    for layer in i["layers"]:
        def lin(name, a):
            return a @ _values(layer[name][0]).t().contiguous() + layer[name][1].double()

        qkv = lin("qkv", _norm(x, 1e-6) * (1.0 + scale) + shift)
        x = x + lin("out", _attention(qkv[:, :D], qkv[:, D:2 * D], qkv[:, 2 * D:], B, case["heads"]))
        kv = lin("ckv", ctx)
        x = x + lin("cout", _attention(lin("cq", _norm(x, 1e-6)), kv[:, :D], kv[:, D:], B, case["heads"]))
        x = x + lin("down", _gelu_tanh(lin("up", _norm(x, 1e-6))))
    return x


def exact(case, seed):
    i, op = _inputs(case, seed), case["op"]
    if op == "linear":
        y = i["x"].double() @ _values(i["b"], case["kind"]).t().contiguous()
        return y if i["bias"] is None else y + i["bias"].double()
    if op == "mlp":
        x = i["x"].double()
        f = _gelu_tanh(x @ _values(i["up"]).t().contiguous() + i["up_b"].double())
        return f, f @ _values(i["down"]).t().contiguous() + i["down_b"].double() + x
    if op in ("attention", "attention_f32"):
        return _attention(i["q"], i["k"], i["v"], case.get("batch", 1), case["heads"])
    if op == "norm":
        y = _norm(i["x"].double(), 1e-6)
        if case["form"] == "affine":
            return y * i["gamma"].double() + i["beta"].double()
        if case["form"] == "ada":
            y = y.reshape(case["batch"], -1, case["dim"]) * (1.0 + i["scale"].double().unsqueeze(1)) + i["shift"].double().unsqueeze(1)
        return y.reshape(case["rows"], case["dim"])
    if op == "packed":
        x = i["x"]
        if case["kernel"] == "int8":  # the integer kernel's operands: codes and scale of each 32 values, in fp32
            b = x.reshape(case["m"], -1, 32)
            amax = b.abs().amax(-1, keepdim=True)
            top = torch.full_like(amax, 127.0)  # a tensor, so that both are divisions
            inv = torch.where(amax > 0, top / amax, torch.zeros_like(amax))
            x = (torch.round(b * inv).double() * (amax / top).double()).reshape(case["m"], -1)
        y = x.double() @ _values(i["b"]).t().contiguous() + i["bias"].double()
        y = y if i["residual"] is None else y + i["residual"].double()
        return _gelu_erf(y) if case["gelu"] else y
    if op == "points":
        h = torch.cat([i["feats"].double(), _embed(i["coords"], i["freqs"])], dim=1)
        for w, b in zip(i["w"], i["b"]):
            h = torch.relu(h @ w.double().t().contiguous() + b.double())
        return h @ i["wh"].double().t().contiguous() + i["bh"].double()
    if op == "weights":
        return None, _values(i["b"], case["kind"])
    return _exact_decoder(case, i) if op == "decoder" else _exact_denoiser(case, i)
