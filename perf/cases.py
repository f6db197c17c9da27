"""The timed cases of the quantized-linear, SageAttention and MMDiT block path.

A case is a dict of plain values: `kind` names the entry points it goes
through and the rest are sizes and options. The kinds are the things a
diffusion program does with this library:

    linear   one quantized linear (int8 or e4m3), activation quantization included
    mlp      the two linears of an MLP, GELU between them
    sage     one SageAttention call on fp16 Q, K, V
    bf16     the four linears a quantized checkpoint keeps in bf16
    int4     one INT4 linear with its low-rank branch (W4A16 or W4A4)
    awq      one AWQ INT4 modulation GEMV
    blocks   joint MMDiT blocks, start to end

`exact` restates each of them in float64 with plain torch, quantization steps
included, so that its distance from `run` is what the kernels' arithmetic
adds and not what the formats lose.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "qwen-image.cu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qimg_amd as q  # noqa: E402

DEV = "cuda"
HIDDEN, HEADS, MLP = 3072, 24, 12288

NF4 = (-1.0, -0.6962, -0.5251, -0.3949, -0.2844, -0.1848, -0.0911, 0.0, 0.0796, 0.1609, 0.2461, 0.3379, 0.4407, 0.5626,
       0.7230, 1.0)


def listed():
    return [
        # The modulation linear of a block: one row, the smallest call, bound
        # by latency and by reading the weight.
        {"name": "modulation_int8", "kind": "linear", "M": 1, "N": 18432, "K": 3072, "mode": "int8", "x": "fp32",
         "out": "fp32", "gelu": False},
        # The same layer of an INT4 checkpoint.
        {"name": "modulation_awq", "kind": "awq", "OC": 18432, "IC": 3072},
        # The text stream's MLP: a few hundred rows, an odd number of them.
        {"name": "mlp_text_int8", "kind": "mlp", "M": 269, "mode": "int8", "x": "bf16", "out": "fp32"},
        # A projection over the tokens of a 1024 x 1024 image.
        {"name": "linear_image_int8", "kind": "linear", "M": 4096, "N": 3072, "K": 3072, "mode": "int8", "x": "bf16",
         "out": "fp32", "gelu": False},
        # The MLP over image and text tokens together.
        {"name": "mlp_image_int8", "kind": "mlp", "M": 4352, "mode": "int8", "x": "bf16", "out": "bf16"},
        # The e4m3 MLP over the tokens of a larger image of odd size.
        {"name": "mlp_image_fp8", "kind": "mlp", "M": 6889, "mode": "fp8", "x": "fp32", "out": "fp32"},
        # Joint attention of a 1024 x 1024 image with 256 text tokens.
        {"name": "attention_4352", "kind": "sage", "BH": 24, "S": 4352, "D": 128, "out": "fp32"},
        # Joint attention of a 512 x 512 image with a text of odd length.
        {"name": "attention_1301", "kind": "sage", "BH": 24, "S": 1301, "D": 128, "out": "fp32"},
        # img_in, txt_in, norm_out and proj_out: once per forward.
        {"name": "bf16_layers", "kind": "bf16", "n_img": 4096, "n_txt": 256},
        # One projection of a NF4 + SVD checkpoint.
        {"name": "linear_w4a16", "kind": "int4", "M": 4096, "N": 3072, "K": 3072, "rank": 32, "gs": 64, "form": "nf4",
         "smooth": True, "gelu": False},
        # One projection of a W4A4 + SVD checkpoint over image and text rows.
        {"name": "linear_w4a4", "kind": "int4", "M": 4352, "N": 3072, "K": 3072, "rank": 32, "gs": 64, "form": "w4a4",
         "smooth": True, "gelu": False},
        # Two joint blocks of the denoising loop at 1024 x 1024.
        {"name": "blocks_int8", "kind": "blocks", "n_img": 4096, "n_txt": 256, "batch": 1, "blocks": 2, "mode": "int8"},
    ]


def draw(rng):
    def log(lo, hi):
        return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    kind = rng.choice(["linear", "linear", "mlp", "sage", "sage", "bf16", "int4", "int4", "awq", "blocks"])
    if kind == "linear":
        n, k = rng.choice([(3072, 3072), (12288, 3072), (3072, 12288), (18432, 3072), (9216, 3072), (3072, 1536),
                           (1000, 3072), (2048, 4096)])
        return {"kind": kind, "M": log(1, 4 if n == 18432 else 8192), "N": n, "K": k,
                "mode": rng.choice(["int8", "fp8"]), "x": rng.choice(["fp32", "bf16"]),
                "out": rng.choice(["fp32", "bf16"]), "gelu": n == 12288}
    if kind == "mlp":
        return {"kind": kind, "M": log(16, 6889), "mode": rng.choice(["int8", "fp8"]),
                "x": rng.choice(["fp32", "bf16"]), "out": rng.choice(["fp32", "bf16"])}
    if kind == "sage":
        return {"kind": kind, "BH": rng.choice([12, 24, 24, 48]), "S": log(77, 5120), "D": rng.choice([128, 128, 64]),
                "out": rng.choice(["fp32", "bf16", "fp16"])}
    if kind == "bf16":
        return {"kind": kind, "n_img": log(256, 8192), "n_txt": log(16, 1024)}
    if kind == "int4":
        n, k = rng.choice([(3072, 3072), (3072, 3072), (12288, 3072), (3072, 12288)])
        return {"kind": kind, "M": log(16, 4608), "N": n, "K": k, "rank": rng.choice([16, 32, 32, 64, 128]),
                "gs": rng.choice([64, 64, 128]), "form": rng.choice(["w4a4", "w4a4", "nf4", "nunchaku16"]),
                "smooth": rng.random() < 0.75, "gelu": n == 12288}
    if kind == "awq":
        return {"kind": kind, "OC": 6 * 64 * log(8, 48), "IC": 64 * log(16, 48)}
    return {"kind": kind, "n_img": log(256, 4096), "n_txt": log(16, 512), "batch": rng.choice([1, 1, 2]), "blocks": 1,
            "mode": rng.choice(["int8", "fp8"])}


# ---- inputs -----------------------------------------------------------------
_TD = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
_MODE = {"int8": q.INT8_HADAMARD, "fp8": q.FP8_HADAMARD}


class _Draw:
    """Tensors drawn on the GPU from one seed, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * std

    def codes(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device=DEV, dtype=torch.uint8)

    def acts(self, M, K):
        """Activations: normal, with one channel in a hundred six times as large."""
        gain = 1.0 + 5.0 * (torch.rand(K, generator=self.g, device=DEV) < 0.01).float()
        return self.normal(M, K) * gain

    def qweight(self, N, K, mode):
        """A quantized weight as a checkpoint holds it: rows of N(0, 0.02),
        which the rotation leaves normal, quantized by row."""
        w = self.normal(N, K, std=0.02)
        top = 127.0 if mode == "int8" else 448.0
        amax = w.abs().amax(1)
        w *= (top / amax)[:, None]
        data = w.round_().to(torch.int8) if mode == "int8" else w.to(torch.float8_e4m3fn).view(torch.uint8)
        return q.QuantizedWeight(data, amax / top, K & -K, _MODE[mode])

    def bias(self, N):
        return self.normal(N, std=0.01).bfloat16()


def _pack(codes):
    """Nibble codes [.., K] -> bytes [.., K/2], the even column in the low nibble."""
    return (codes[..., 0::2] | (codes[..., 1::2] << 4)).contiguous()


_BLOCK = [("img_mod", 6 * HIDDEN, HIDDEN), ("txt_mod", 6 * HIDDEN, HIDDEN)] + \
         [(n, HIDDEN, HIDDEN) for n in ("to_q", "to_k", "to_v", "add_q_proj", "add_k_proj", "add_v_proj", "to_out",
                                        "to_add_out")] + \
         [("img_mlp_fc1", MLP, HIDDEN), ("img_mlp_fc2", HIDDEN, MLP), ("txt_mlp_fc1", MLP, HIDDEN),
          ("txt_mlp_fc2", HIDDEN, MLP)]
_NORMS = ("norm_q", "norm_k", "norm_added_q", "norm_added_k")


def _rope(n_txt, n_img):
    """(cos, -sin, sin, cos) rows of a text of n_txt and a grid of n_img
    positions, three axes of 16, 56 and 56 dims."""
    side = max(1, math.isqrt(n_img))
    i = torch.arange(n_img, device=DEV, dtype=torch.float64)
    t = torch.arange(n_txt, device=DEV, dtype=torch.float64) + side
    rows = torch.cat([t, torch.floor(i / side) - side // 2])
    cols = torch.cat([t, i % side - side // 2])
    first = torch.cat([t, torch.zeros_like(i)])
    ang = []
    for pos, dim in ((first, 16), (rows, 56), (cols, 56)):
        omega = 10000.0 ** (-torch.arange(0, dim, 2, device=DEV, dtype=torch.float64) / dim)
        ang.append(pos[:, None] * omega[None])
    a = torch.cat(ang, 1)
    return torch.stack([a.cos(), -a.sin(), a.sin(), a.cos()], -1).float().contiguous()


def _inputs(c, seed):
    d = _Draw(seed)
    s = dict(c)
    kind = c["kind"]
    if kind == "linear":
        s["w"] = d.qweight(c["N"], c["K"], c["mode"])
        s["bias"] = d.bias(c["N"])
        s["in"] = d.acts(c["M"], c["K"]).to(_TD[c["x"]])
    elif kind == "mlp":
        s["w1"], s["w2"] = d.qweight(MLP, HIDDEN, c["mode"]), d.qweight(HIDDEN, MLP, c["mode"])
        s["b1"], s["b2"] = d.bias(MLP), d.bias(HIDDEN)
        s["in"] = d.acts(c["M"], HIDDEN).to(_TD[c["x"]])
    elif kind == "sage":
        # unit-variance Q and K after their RMSNorm, K with a mean of its own
        shape = (c["BH"], c["S"], c["D"])
        s["q"], s["v"] = d.normal(*shape).half(), d.normal(*shape).half()
        s["k"] = (d.normal(*shape) + d.normal(c["BH"], 1, c["D"], std=0.5)).half()
    elif kind == "bf16":
        for name, M, N, K in _bf16_layers(c):
            s[name] = (d.normal(M, K), d.normal(N, K, std=0.02).bfloat16(), d.bias(N))
    elif kind == "int4":
        N, K, r, gs = c["N"], c["K"], c["rank"], c["gs"]
        s["in"] = d.acts(c["M"], K)
        s["bias"] = d.bias(N)
        s["up"] = d.normal(N, r, std=0.1).bfloat16()
        s["down"] = d.normal(K, r, std=0.02).bfloat16()
        s["smooth"] = (d.normal(K, std=0.3)).exp() if c["smooth"] else None
        s["codes"] = d.codes(0, 16, N, K)
        s["packed"] = _pack(s["codes"])
        scale = 0.02 * (d.normal(N, K // gs, std=0.3)).exp()
        # NF4 codes span [-1, 1], two's complement ones [-8, 7]
        s["scales"] = scale * 2.5 if c["form"] == "nf4" else (scale / 4.0).t().contiguous()
    elif kind == "awq":
        OC, IC = c["OC"], c["IC"]
        s["in"] = d.normal(IC)
        s["codes"] = d.codes(0, 16, OC, IC)
        words = torch.zeros(OC, IC // 8, dtype=torch.int64, device=DEV)
        for k in range(8):
            words |= s["codes"][:, k::8].long() << (4 * k)
        words = torch.where(words >= 1 << 31, words - (1 << 32), words)
        s["packed"] = words.to(torch.int32).t().contiguous()
        s["ws"] = (0.005 * d.normal(IC // 64, OC, std=0.3).exp()).bfloat16()
        s["wz"] = (-7.5 * s["ws"].float() + d.normal(IC // 64, OC, std=0.002)).bfloat16()
        s["bias"] = d.bias(OC)
    else:
        s["table"] = [({n: d.qweight(N, K, c["mode"]) for n, N, K in _BLOCK}, {n: d.bias(N) for n, N, _ in _BLOCK},
                       {n: (1.0 + d.normal(128, std=0.1)).bfloat16() for n in _NORMS}) for _ in range(c["blocks"])]
        s["img0"], s["txt0"] = d.normal(c["batch"], c["n_img"], HIDDEN), d.normal(c["batch"], c["n_txt"], HIDDEN)
        s["t_emb"] = d.normal(HIDDEN)
        s["pe"] = _rope(c["n_txt"], c["n_img"])
    return s


def _bf16_layers(c):
    """(name, M, N, K): img_in, txt_in, norm_out on the time embedding, proj_out."""
    return [("img_in", c["n_img"], HIDDEN, 64), ("txt_in", c["n_txt"], HIDDEN, 3584),
            ("norm_out", 1, 2 * HIDDEN, HIDDEN), ("proj_out", c["n_img"], 64, HIDDEN)]


def prepare(case, seed):
    """The inputs, with the output and scratch buffers and handles that a
    program keeps from one step to the next."""
    s = _inputs(case, seed)
    kind = s["kind"]

    def buf(n):
        return torch.empty(max(int(n), 1), dtype=torch.uint8, device=DEV)

    if kind == "linear":
        s["y"] = torch.empty(s["M"], s["N"], dtype=_TD[s["out"]], device=DEV)
        s["scratch"] = buf(q.int8_scratch_bytes(s["M"], s["K"], s["N"]))
    elif kind == "mlp":
        s["h"] = torch.empty(s["M"], MLP, device=DEV)
        s["y"] = torch.empty(s["M"], HIDDEN, dtype=_TD[s["out"]], device=DEV)
        s["scratch"] = buf(q.int8_scratch_bytes(s["M"], MLP, MLP))
    elif kind == "sage":
        s["y"] = torch.empty(s["BH"], s["S"], s["D"], dtype=_TD[s["out"]], device=DEV)
        s["scratch"] = buf(q.sage_scratch_bytes(s["BH"], s["S"], s["D"]))
    elif kind == "bf16":
        s["y"] = {name: torch.empty(M, N, device=DEV) for name, M, N, K in _bf16_layers(case)}
    elif kind == "int4":
        N, K, w4a4 = s["N"], s["K"], s["form"] == "w4a4"
        held = {"w4a4_qweight": s["packed"], "w4a4_wscales": s["scales"]} if w4a4 else \
            {"qweight": s["packed"], "scales4": s["scales"]}
        s["w"] = q.Int4Weight(N, K, s["gs"], svd_up=s["up"], svd_down=s["down"], smooth=s["smooth"],
                              had_block_size=K & -K if s["form"] == "nf4" else 1, nf4_grid=s["form"] == "nf4",
                              w4a16_nunchaku=s["form"] == "nunchaku16", **held)
        s["y"] = torch.empty(s["M"], N, device=DEV)
        s["scratch"] = buf(q.int4_scratch_bytes(s["M"], K, N, s["rank"]))
        del s["codes"]
    elif kind == "awq":
        del s["codes"]
    else:
        s["handle"] = q.BlockTable(s["table"])
        s["img"], s["txt"] = torch.empty_like(s["img0"]), torch.empty_like(s["txt0"])
        s["scratch"] = buf(q.mmdit_block_scratch_bytes(s["n_img"], s["n_txt"], s["batch"]))
    return s


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return q.linear_forward_quantized(s["in"], s["w"], s["bias"], out=s["y"], scratch=s["scratch"],
                                          apply_gelu=s["gelu"])
    if kind == "mlp":
        q.linear_forward_quantized(s["in"], s["w1"], s["b1"], out=s["h"], scratch=s["scratch"], apply_gelu=True)
        return q.linear_forward_quantized(s["h"], s["w2"], s["b2"], out=s["y"], scratch=s["scratch"])
    if kind == "sage":
        return q.attention_forward_sage_fp16io(s["q"], s["k"], s["v"], 1.0 / math.sqrt(s["D"]), out=s["y"],
                                               scratch=s["scratch"])
    if kind == "bf16":
        return {n: q.linear_forward_bf16(*s[n][:2], bias=s[n][2], out=y) for n, y in s["y"].items()}
    if kind == "int4":
        return q.linear_forward_int4(s["in"], s["w"], bias=s["bias"], apply_gelu=s["gelu"], out=s["y"],
                                     scratch=s["scratch"])
    if kind == "awq":
        return q.linear_forward_awq(s["in"], s["packed"], s["ws"], s["wz"], s["OC"], s["IC"], bias=s["bias"])
    # the blocks update the streams in place; a step starts from new ones
    s["img"].copy_(s["img0"])
    s["txt"].copy_(s["txt0"])
    q.mmdit_blocks_forward(s["handle"], s["img"], s["txt"], s["t_emb"], s["pe"], scratch=s["scratch"])
    return s["img"], s["txt"]


def work(c):
    kind = c["kind"]
    size = {"fp32": 4, "bf16": 2, "fp16": 2}

    def lin(M, N, K, x, w, out):
        return M * K * x + N * K * w + M * N * out + N * 6.0, 2.0 * M * N * K

    if kind == "linear":
        b, f = lin(c["M"], c["N"], c["K"], size[c["x"]], 1, size[c["out"]])
    elif kind == "mlp":
        b1, f1 = lin(c["M"], MLP, HIDDEN, size[c["x"]], 1, 0)
        b2, f2 = lin(c["M"], HIDDEN, MLP, 0, 1, size[c["out"]])
        b, f = b1 + b2, f1 + f2
    elif kind == "sage":
        e = c["BH"] * c["S"] * c["D"]
        b, f = e * (6.0 + size[c["out"]]), 4.0 * e * c["S"]
    elif kind == "bf16":
        b = f = 0.0
        for _, M, N, K in _bf16_layers(c):
            b1, f1 = lin(M, N, K, 4, 2, 4)
            b, f = b + b1, f + f1
    elif kind == "int4":
        b, f = lin(c["M"], c["N"], c["K"], 4, 0.5, 4)
        r = c["rank"]
        b += c["N"] * c["K"] // c["gs"] * 4.0 + 2.0 * r * (c["N"] + c["K"])
        f += 2.0 * c["M"] * r * (c["N"] + c["K"])
    elif kind == "awq":
        b, f = c["OC"] * c["IC"] * (0.5 + 4.0 / 64) + 4.0 * c["IC"] + 6.0 * c["OC"], 2.0 * c["OC"] * c["IC"]
    else:
        img, txt, B = c["n_img"], c["n_txt"], c["batch"]
        tok = (img + txt) * B
        f = 2.0 * tok * HIDDEN * (4 * HIDDEN + 2 * MLP) + 4.0 * B * HIDDEN * float(img + txt) ** 2
        f += 2.0 * 2 * 6 * HIDDEN * HIDDEN
        w = sum(N * K + 6.0 * N for _, N, K in _BLOCK)
        b, f = tok * HIDDEN * 8.0 + c["blocks"] * w + (img + txt) * 1024.0, f * c["blocks"]
    return {"bytes": float(b), "flops": float(f)}


def tolerance(c):
    """About four times the distance of these kernels from `exact`, at the
    same sizes."""
    kind = c["kind"]
    if kind == "linear":
        # bf16 outputs: half a step. fp32: a value that another rounding of
        # the scale moves to the next int8 code; in one row of 3072 a single
        # one is 5e-4.
        return {"rel": 7e-3 if c["out"] == "bf16" else 1e-3}
    if kind == "mlp":
        # the same in the quantization of the GELU output, whose steps are coarse
        return {"rel": 8e-3}
    if kind == "sage":
        # P and the output in fp16; bf16 outputs half a step
        return {"rel": 7e-3 if c["out"] == "bf16" else 1.2e-3}
    if kind == "bf16":
        return {"rel": 1e-6}
    if kind == "int4":
        # bf16 roundings of the rotated input; W4A4: INT4 codes on a boundary
        return {"rel": 1e-3 if c["form"] == "w4a4" else 2e-4}
    if kind == "awq":
        return {"rel": 4e-6}
    # A change of rounding in one layer moves int8 codes in all that follow:
    # noise of 1e-7 on the input moves the output of one block by 3e-2.
    return {"rel": 0.12}


# ---- the same in float64 ------------------------------------------------------
def _f64(t):
    return t.double()


def _bf16(t):
    return t.float().bfloat16().double()


def _fwht(x, h):
    """Normalised Walsh-Hadamard transform of the blocks of h columns."""
    M, K = x.shape
    x = x.reshape(M, K // h, h)
    n = 1
    while n < h:
        x = x.reshape(M, -1, h // (2 * n), 2, n)
        a, b = x[..., 0, :], x[..., 1, :]
        x = torch.stack([a + b, a - b], -2)
        n *= 2
    return x.reshape(M, K) / math.sqrt(h)


def _gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))


def _qlinear(x, w, bias, gelu=False):
    """Rotate and quantize the rows of x, multiply by the quantized weight."""
    int8 = w.mode == q.INT8_HADAMARD
    top = 127.0 if int8 else 448.0
    x = _fwht(x, w.had_block_size)
    amax = x.abs().amax(1, keepdim=True)
    v = x * (top / amax.clamp_min(1e-300))
    v = v.round() if int8 else v.float().to(torch.float8_e4m3fn).double()
    wd = w.data.double() if int8 else w.data.view(torch.float8_e4m3fn).double()
    y = (v @ wd.t()) * (amax / top) * w.scales.double()[None] + bias.double()[None]
    return _gelu(y) if gelu else y


def _groups(S, heads, block, pattern):
    """Scale group of each of S tokens: blocks of `block` tokens, `pattern`
    the group of each token in its block."""
    t = torch.arange(S, device=DEV)
    return (t // block) * (int(pattern.max()) + 1) + pattern[t % block]


def _quant_tokens(x, group, n):
    """x [S, D] in int8 with one scale per group of tokens -> (codes, scale [S])."""
    amax = torch.full((n,), 1e-7, dtype=torch.float64, device=DEV)
    amax = amax.scatter_reduce(0, group, x.abs().amax(1), "amax")
    scale = (amax / 127.0 + 1e-7)[group]
    return (x / scale[:, None]).round().clamp(-128, 127), scale


def _sage(qh, kh, vh, scale):
    """SageAttention of [BH, S, D]: K less its mean, Q and K in int8 with a
    scale for each group of tokens, softmax and P.V in float64."""
    BH, S, D = qh.shape
    t = torch.arange(128, device=DEV)
    gq = _groups(S, BH, 128, t // 32 * 8 + t % 8)
    gk = _groups(S, BH, 64, t[:64] % 8 // 2)
    out = torch.empty(BH, S, D, dtype=torch.float64, device=DEV)
    for b in range(BH):
        k = _f64(kh[b])
        qi, qs = _quant_tokens(_f64(qh[b]), gq, int(gq.max()) + 1)
        ki, ks = _quant_tokens(k - k.mean(0, keepdim=True), gk, int(gk.max()) + 1)
        p = (qi * qs[:, None]) @ (ki * ks[:, None]).t()
        out[b] = torch.softmax(p * scale, -1) @ _f64(vh[b])
    return out


def _int4(s):
    K, gs = s["K"], s["gs"]
    v = _f64(s["in"])
    if s["smooth"] is not None:
        v = v / s["smooth"].double()
    xs = _bf16(v)
    low = _bf16(xs @ s["down"].double()) @ s["up"].double().t()
    codes = s["codes"].long()
    if s["form"] == "nf4":
        grid = torch.tensor(NF4, device=DEV).double()
        w = _bf16(grid[codes] * s["scales"].double().repeat_interleave(gs, 1))
        y = _bf16(_fwht(v, K & -K)) @ w.t()
    else:
        n = torch.where(codes >= 8, codes - 16, codes).double()
        ws = s["scales"].double().t().repeat_interleave(gs, 1)
        if s["form"] == "nunchaku16":
            y = xs @ _bf16(n * ws).t()
        else:
            g = v.reshape(-1, K // gs, gs)
            amax = g.abs().amax(-1, keepdim=True)
            r = g * (7.0 / amax.clamp_min(1e-300))
            a = torch.sign(r) * torch.floor(r.abs() + 0.5)
            y = (a.clamp(-7, 7) * (amax / 7.0)).reshape(-1, K) @ (n * ws).t()
    y = y + low + s["bias"].double()
    return _gelu(y) if s["gelu"] else y


def _block(img, txt, t_emb, pe, W, B, norms):
    """One joint block on [n_img, 3072] and [n_txt, 3072]."""
    n_txt = txt.shape[0]

    def lin(x, name, gelu=False):
        return _qlinear(x, W[name], B[name], gelu)

    def ln(x, shift, scale):
        d = x - x.mean(1, keepdim=True)
        return d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-6) * (1.0 + scale) + shift

    def heads(t, i, wt, wi):
        parts = []
        for x, w in ((t, wt), (i, wi)):
            x = x.reshape(-1, HEADS, 128)
            if w is not None:
                x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * norms[w].double()
            parts.append(x)
        x = torch.cat(parts).transpose(0, 1)
        if wt is not None:
            a, b, p = x[..., 0::2], x[..., 1::2], pe.double()[None]
            x = torch.stack([a * p[..., 0] + b * p[..., 1], a * p[..., 2] + b * p[..., 3]], -1).flatten(-2)
        return x.float().half()

    ts = (t_emb.double() / (1.0 + torch.exp(-t_emb.double())))[None]
    im, tm = lin(ts, "img_mod").reshape(6, HIDDEN), lin(ts, "txt_mod").reshape(6, HIDDEN)
    xi, xt = ln(img, im[0], im[1]), ln(txt, tm[0], tm[1])
    qh = heads(lin(xt, "add_q_proj"), lin(xi, "to_q"), "norm_added_q", "norm_q")
    kh = heads(lin(xt, "add_k_proj"), lin(xi, "to_k"), "norm_added_k", "norm_k")
    vh = heads(lin(xt, "add_v_proj"), lin(xi, "to_v"), None, None)
    a = _sage(qh, kh, vh, 1.0 / math.sqrt(128.0)).float().half().double().transpose(0, 1).reshape(-1, HIDDEN)
    img = img + im[2] * lin(a[n_txt:], "to_out")
    txt = txt + tm[2] * lin(a[:n_txt], "to_add_out")
    xi, xt = ln(img, im[3], im[4]), ln(txt, tm[3], tm[4])
    img = img + im[5] * lin(lin(xi, "img_mlp_fc1", True), "img_mlp_fc2")
    txt = txt + tm[5] * lin(lin(xt, "txt_mlp_fc1", True), "txt_mlp_fc2")
    return img, txt


def exact(case, seed):
    s = _inputs(case, seed)
    kind = s["kind"]
    if kind == "linear":
        return _qlinear(_f64(s["in"]), s["w"], s["bias"], s["gelu"])
    if kind == "mlp":
        return _qlinear(_qlinear(_f64(s["in"]), s["w1"], s["b1"], True), s["w2"], s["b2"])
    if kind == "sage":
        return _sage(s["q"], s["k"], s["v"], 1.0 / math.sqrt(s["D"]))
    if kind == "bf16":
        return {n: _bf16(s[n][0]) @ s[n][1].double().t() + s[n][2].double() for n, *_ in _bf16_layers(case)}
    if kind == "int4":
        return _int4(s)
    if kind == "awq":
        n = torch.arange(s["OC"], device=DEV)
        ws, wz = (s[k].double().t().repeat_interleave(64, 1) for k in ("ws", "wz"))
        y = (s["codes"].double() * ws + wz) @ s["in"].double()
        out = torch.empty(1, s["OC"], dtype=torch.float64, device=DEV)
        out[0, n % 6 * (s["OC"] // 6) + n // 6] = y
        return out + s["bias"].double()
    imgs, txts = [], []
    for b in range(s["batch"]):
        img, txt = _f64(s["img0"][b]), _f64(s["txt0"][b])
        for W, B, norms in s["table"]:
            img, txt = _block(img, txt, s["t_emb"], s["pe"], W, B, norms)
        imgs.append(img)
        txts.append(txt)
    return torch.stack(imgs), torch.stack(txts)
