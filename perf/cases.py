"""The work this framework is used for, as cases that a benchmark can prepare, run, time and check.

Each case is one pass through the public entry points of stblarge_amd.ops / stblarge_amd.moe:

  gemv        one quantized projection of 1-4 decode tokens (ops.gemv_fp4 / ops.gemv_fp8)
  gemv_batch  same-shape projections of several experts in one launch (ops.gemv_batch)
  abi_batch   the reference engine's batched GGUF GEMV, fp32 activations (ops.stbl_gemv_mxfp4_batch)
  ffn         one expert's gate/up + SwiGLU + down (ops.expert_ffn)
  moe         a routed layer's expert part over resident slots (ops.moe_experts)
  layer       a routed layer from router logits to output through its expert cache (MoELayer.forward)
  gemm        the multi-token projection of prefill and of batched decode (ops.gemm and its forms)
  act_quant   the activation quantizer that feeds such projections (ops.act_quant)
  load        an expert's fp32 weights quantized into its slot (ops.quant_expert)

Weights are N(0, 0.02) and activations N(0, 1), as the configurations draw them. They are quantized
here in plain torch, so that the inputs of a case do not depend on the library's own quantizers.
"""

import math

import torch

from stblarge_amd import ops
from stblarge_amd.moe import MoELayer

FP4, FP8, FP8_E8M0 = 0, 1, 2
BF16, F32, F64, U8 = torch.bfloat16, torch.float32, torch.float64, torch.uint8


# ---- the cases --------------------------------------------------------------------------------------


def listed():
    return [
        # the configurations' single expert projection of one decode token
        {"name": "gemv_fp4_m1", "kind": "gemv", "fmt": FP4, "rows": 2048, "k": 7168, "m": 1, "f32": False},
        # the down projection of a few tokens (a small batch, or speculative tokens), FP8 weights
        {"name": "gemv_fp8_m3", "kind": "gemv", "fmt": FP8, "rows": 7168, "k": 2048, "m": 3, "f32": False},
        # gate and up of one token's eight routed experts in one launch
        {"name": "gemv_batch16_fp4", "kind": "gemv_batch", "fmt": FP4, "rows": 2048, "k": 7168, "m": 1, "n": 16},
        # the reference engine's own call: gate and up of its six experts, GGUF blocks
        {"name": "abi_batch12", "kind": "abi_batch", "rows": 2304, "k": 5120, "n": 12},
        # the configurations' expert FFN at batch 1, FP8 variant
        {"name": "ffn_fp8", "kind": "ffn", "fmt": FP8, "dim": 7168, "inter": 2048, "m": 1, "official": False},
        # the engine's MoE step of four tokens: six FP4 experts each, an FP8 shared expert, official numerics
        {"name": "moe_v41_t4", "kind": "moe", "dim": 5120, "inter": 2304, "t": 4, "topk": 6, "n": 24,
         "shared_fmt": FP8_E8M0, "official": True, "limit": 10.0},
        # a whole routed layer of one decode token: router, cache lookup, experts, combine, all experts resident
        {"name": "layer_t1", "kind": "layer", "dim": 7168, "inter": 2048, "t": 1, "topk": 8, "n": 32},
        # the configurations' multi-token expert projection: 64 tokens of one expert, FP4 weights
        {"name": "gemm_fp4_m64", "kind": "gemm", "form": "gemm", "fmt": FP4, "m": 64, "n": 2048, "k": 7168,
         "block": 128, "f32": False},
        # prefill with a ragged number of tokens on one expert, FP8 weights
        {"name": "gemm_fp8_m300", "kind": "gemm", "form": "gemm", "fmt": FP8, "m": 300, "n": 2048, "k": 7168,
         "block": 128, "f32": False},
        # the down projection of a long prefill, FP4 weights
        {"name": "gemm_fp4_m1024", "kind": "gemm", "form": "gemm", "fmt": FP4, "m": 1024, "n": 7168, "k": 2048,
         "block": 128, "f32": False},
        # the activations of a prefill quantized once for several projections
        {"name": "act_quant_512", "kind": "act_quant", "rows": 512, "n": 7168, "block": 128, "pow2": True,
         "deq": False},
        # loading an expert: its three fp32 matrices quantized into a cache slot
        {"name": "load_fp8", "kind": "load", "fmt": FP8, "dim": 7168, "inter": 2048},
    ]


def _spread(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // step, max(-(-lo // step), round(v / step))) * step


def draw(rng):
    kind = rng.choice(["gemv", "gemv_batch", "abi_batch", "ffn", "moe", "layer", "gemm", "gemm", "act_quant", "load"])
    fmt = rng.choice([FP4, FP8])
    if kind == "gemv":
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 256, 8192), "k": _spread(rng, 512, 7168, 32),
                "m": rng.randint(1, 4), "f32": rng.random() < 0.25}
    if kind == "gemv_batch":
        n = rng.randint(2, 16)
        return {"kind": kind, "fmt": fmt, "rows": _spread(rng, 256, 7168), "k": _spread(rng, 512, 7168 if n < 9 else 2048, 32),
                "m": rng.randint(1, 4), "n": n}
    if kind == "abi_batch":
        return {"kind": kind, "rows": _spread(rng, 256, 5120), "k": _spread(rng, 512, 5120, 256), "n": rng.randint(1, 12)}
    if kind == "ffn":
        fmt = rng.choice([FP4, FP8, FP8_E8M0])
        step = 128 if fmt == FP8 else 32
        return {"kind": kind, "fmt": fmt, "dim": _spread(rng, 1024, 7168, step), "inter": _spread(rng, 512, 2560, step),
                "m": rng.randint(1, 4), "official": rng.random() < 0.5}
    if kind == "moe":
        t, topk = rng.randint(1, 4), rng.choice([4, 6, 8])
        return {"kind": kind, "dim": _spread(rng, 1024, 5120, 32), "inter": _spread(rng, 512, 1536, 32), "t": t,
                "topk": topk, "n": rng.randint(topk, 24), "shared_fmt": rng.choice([FP4, FP8_E8M0]),
                "official": rng.random() < 0.5, "limit": rng.choice([0.0, 10.0])}
    if kind == "layer":
        return {"kind": kind, "dim": _spread(rng, 1024, 7168, 32), "inter": _spread(rng, 512, 1024, 32),
                "t": rng.randint(1, 4), "topk": rng.choice([4, 6, 8]), "n": rng.choice([16, 24, 32])}
    if kind == "gemm":
        n, k = _spread(rng, 256, 7168, 16), _spread(rng, 512, 7168, 128)
        while n * k > 7168 * 2048:
            n, k = _spread(rng, 256, 7168, 16), _spread(rng, 512, 7168, 128)
        return {"kind": kind, "form": rng.choice(["gemm", "gemm", "q", "packed"]), "fmt": fmt, "m": _spread(rng, 5, 1024),
                "n": n, "k": k, "block": 128 if fmt == FP8 else rng.choice([32, 128]), "f32": rng.random() < 0.25}
    if kind == "act_quant":
        return {"kind": kind, "rows": _spread(rng, 1, 1024), "n": _spread(rng, 512, 7168, 128),
                "block": rng.choice([32, 64, 128]), "pow2": rng.random() < 0.75, "deq": rng.random() < 0.5}
    fmt = rng.choice([FP4, FP8, FP8_E8M0])
    step = 128 if fmt == FP8 else 32
    return {"kind": "load", "fmt": fmt, "dim": _spread(rng, 1024, 7168, step), "inter": _spread(rng, 512, 2048, step)}


# ---- plain torch: formats -----------------------------------------------------------------------------


def _gen(seed, *more):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + sum(v * 7919 ** i for i, v in enumerate(more, 1)))
    return g


def _weight(g, rows, k):
    return torch.randn((rows, k), generator=g, device="cuda") * 0.02


def _act(g, m, k):
    return torch.randn((m, k), generator=g, device="cuda").to(BF16)


def _pow2_ceil(t):
    m, e = torch.frexp(t)
    return torch.ldexp(torch.ones_like(t), torch.where(m == 0.5, e - 1, e))


def _quant_fp4(w):
    """(codes [rows, k/2], E8M0 scales [rows, k/32]): nearest e2m1 value, ties to the even code."""
    rows, k = w.shape
    g = w.view(rows, k // 32, 32)
    s = _pow2_ceil(g.abs().amax(-1).clamp_min(6 * 2.0 ** -126) / 6)
    a = (g / s[..., None]).abs()
    bounds = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device)
    up, down = torch.bucketize(a, bounds, right=True), torch.bucketize(a, bounds)
    code = torch.where(up % 2 == 0, up, down) + 8 * (g < 0)
    code = code.to(U8).view(rows, k // 2, 2)
    return code[..., 0] | (code[..., 1] << 4), (torch.log2(s) + 127).to(U8)


def _e4m3(v):
    return v.clamp(-448, 448).to(torch.float8_e4m3fn)


def _blocks(t, rows, k, b):
    """Per-block values t [ceil(rows/b), ceil(k/b)] spread over [rows, k]."""
    return t.repeat_interleave(b, 0)[:rows].repeat_interleave(b, 1)[:, :k]


def _quant_fp8(w, b, e8m0):
    """(e4m3 codes [rows, k], scales per b x b block: fp32, or E8M0 bytes)."""
    rows, k = w.shape
    a = torch.nn.functional.pad(w.abs(), (0, -k % b, 0, -rows % b))
    s = a.view(a.shape[0] // b, b, a.shape[1] // b, b).amax((1, 3)).clamp_min(1e-4) / 448
    s = _pow2_ceil(s) if e8m0 else s
    codes = _e4m3(w / _blocks(s, rows, k, b)).view(U8)
    return codes, (torch.log2(s) + 127).to(U8) if e8m0 else s


def _quant(w, fmt):
    return _quant_fp4(w) if fmt == FP4 else _quant_fp8(w, 32, True) if fmt == FP8_E8M0 else _quant_fp8(w, 128, False)


def _dequant(codes, scales, fmt):
    """The weights that (codes, scales) stand for, in 64 bits."""
    if fmt == FP4:
        table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=F64, device=codes.device)
        v = table[torch.stack((codes & 15, codes >> 4), -1).long()].view(codes.shape[0], -1)
        return v * torch.exp2(scales.to(F64) - 127).repeat_interleave(32, 1)
    v = codes.view(torch.float8_e4m3fn).to(F64)
    s, b = (torch.exp2(scales.to(F64) - 127), 32) if fmt == FP8_E8M0 else (scales.to(F64), 128)
    return v * _blocks(s, *codes.shape, b)


def _act_scales(x, block, pow2):
    """(x in blocks, its scale per block) of the activation quantizer, fp32."""
    f = x.float().view(*x.shape[:-1], -1, block)
    t = f.abs().amax(-1).clamp_min(1e-4) * torch.tensor(1 / 448, device=x.device)
    return f, _pow2_ceil(t) if pow2 else t


def _act_quant(x, block):
    """(e4m3 codes, E8M0 scale bytes) of bf16 x, power-of-two scales per `block`."""
    f, s = _act_scales(x, block, True)
    return _e4m3(f / s[..., None]).view(U8).view(x.shape), (torch.log2(s) + 127).to(U8)


def _act_values(x, block):
    """What the quantized x stands for, in 64 bits."""
    f, s = _act_scales(x, block, True)
    return (_e4m3(f / s[..., None]).to(F64) * s.to(F64)[..., None]).view(x.shape)


def _expert(g, dim, inter, fmt):
    """[gate codes, gate scales, up codes, up scales, down codes, down scales] of one expert."""
    parts = []
    for rows, k in ((inter, dim), (inter, dim), (dim, inter)):
        parts += list(_quant(_weight(g, rows, k), fmt))
    return parts


def _ffn(parts, x, fmt, weight, limit, official):
    """One expert on x [m, dim] with the roundings that the path states (gate, up and the SwiGLU
    output are bf16; official numerics quantize x and that output), everything else in 64 bits.
    weight: [m, 1]."""
    gate, up, down = (_dequant(parts[i], parts[i + 1], fmt) for i in (0, 2, 4))
    xd = _act_values(x, 32) if official else x.to(F64)
    g, u = ((xd @ w.T).to(BF16).to(F64) for w in (gate, up))
    if limit > 0:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    h = (g / (1 + torch.exp(-g)) * u * weight).to(BF16)
    return (_act_values(h, 32) if official else h.to(F64)) @ down.T


# ---- one case -----------------------------------------------------------------------------------------


def _picks(case, seed):
    """Routed experts and weights of a MoE step: distinct experts per token, popular ones first."""
    g = torch.Generator().manual_seed(seed * 31 + 5)
    p = torch.arange(1, case["n"] + 1, dtype=F64) ** -0.5
    pick = [torch.multinomial(p, case["topk"], generator=g).tolist() for _ in range(case["t"])]
    w = torch.softmax(torch.randn((case["t"], case["topk"]), generator=g), -1).tolist()
    return pick, w


def _gguf(codes, scales):
    """Rows of 17-byte blocks (scale byte; element i in the low nibble of byte 1 + i, 16 + i in the high)."""
    rows = codes.shape[0]
    el = torch.stack((codes & 15, codes >> 4), -1).view(rows, -1, 32)
    return torch.cat((scales[..., None], el[..., :16] | (el[..., 16:] << 4)), -1).view(rows, -1).contiguous()


def _inputs(case, seed):
    """Everything that prepare() and exact() share, from the seed alone."""
    g, kind = _gen(seed, 3), case["kind"]
    if kind == "gemv":
        return (*_quant(_weight(g, case["rows"], case["k"]), case["fmt"]), _act(g, case["m"], case["k"]))
    if kind == "gemv_batch":
        q = [_quant(_weight(g, case["rows"], case["k"]), case["fmt"]) for _ in range(case["n"])]
        return [c for c, _ in q], [s for _, s in q], [_act(g, case["m"], case["k"]) for _ in q]
    if kind == "abi_batch":
        q = [_quant_fp4(_weight(g, case["rows"], case["k"])) for _ in range(case["n"])]
        # the engine quantizes its activations before the call (e4m3 codes times powers of two)
        xs = [_act_values(_act(g, 1, case["k"]), 32).float().view(-1) for _ in q]
        return q, xs
    if kind == "ffn":
        return _expert(g, case["dim"], case["inter"], case["fmt"]), _act(g, case["m"], case["dim"])
    if kind == "moe":
        experts = [_expert(g, case["dim"], case["inter"], FP4) for _ in range(case["n"])]
        shared = _expert(g, case["dim"], case["inter"], case["shared_fmt"])
        return experts, shared, _act(g, case["t"], case["dim"])
    if kind == "layer":
        experts = [_expert(g, case["dim"], case["inter"], FP4) for _ in range(case["n"])]
        shared = _expert(g, case["dim"], case["inter"], FP4)
        logits = torch.randn((case["t"], case["n"]), generator=g, device="cuda") * 2
        return experts, shared, _act(g, case["t"], case["dim"]), logits
    if kind == "gemm":
        return (*_quant(_weight(g, case["n"], case["k"]), case["fmt"]), _act(g, case["m"], case["k"]))
    if kind == "act_quant":
        # rows of different magnitude, as a residual stream has them
        return _act(g, case["rows"], case["n"]) * torch.exp2(torch.randint(-6, 4, (case["rows"], 1), generator=g, device="cuda")).to(BF16)
    return [_weight(g, r, k) for r, k in ((case["inter"], case["dim"]),) * 2 + ((case["dim"], case["inter"]),)]


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    got = _inputs(case, seed)
    if kind == "gemv":
        s["codes"], s["scales"], s["x"] = got
    elif kind == "gemv_batch":
        s["codes"], s["scales"], s["xs"] = got
    elif kind == "abi_batch":
        q, s["xs"] = got
        s["ws"] = [_gguf(c, sc) for c, sc in q]
        s["ys"] = [torch.empty(case["rows"], device="cuda") for _ in q]
    elif kind == "ffn":
        parts, s["x"] = got
        s["slot"] = ops.pack_slot(parts, case["fmt"], case["dim"], case["inter"])
    elif kind == "moe":
        experts, shared, s["x"] = got
        dim, inter = case["dim"], case["inter"]
        s["slots"] = [ops.pack_slot(p, FP4, dim, inter) for p in experts]
        s["slots"].append(ops.pack_slot(shared, case["shared_fmt"], dim, inter))
        s["pick"], s["weights"] = _picks(case, seed)
        s["work"] = torch.empty(ops.moe_work_bytes(case["t"], case["topk"], dim, inter), dtype=U8, device="cuda")
    elif kind == "layer":
        experts, shared, s["x"], s["logits"] = got
        dim, inter, n = case["dim"], case["inter"], case["n"]
        size, _ = ops.expert_layout(FP4, dim, inter)
        pool = torch.empty(n * size, dtype=U8, pin_memory=True)
        for e, p in enumerate(experts):
            pool[e * size:(e + 1) * size].copy_(ops.pack_slot(p, FP4, dim, inter))
        layer = MoELayer(FP4, dim, inter, pool, n, case["topk"], n, shared_slot=ops.pack_slot(shared, FP4, dim, inter),
                         max_tokens=case["t"])
        # a layer that has served for a while: every expert has been routed to and is in its cache
        layer.cache.lookup(list(range(n)))
        s["layer"] = layer
    elif kind == "gemm":
        codes, scales, x = got
        s["codes"], s["scales"] = codes.contiguous(), scales
        if case["form"] == "q":
            s["aq"], s["as"] = _act_quant(x, case["block"])
        else:
            s["x"] = x
        if case["form"] == "packed":
            s["codes"] = ops.gemm_pack(s["codes"], case["fmt"])
    elif kind == "act_quant":
        s["x"] = got
    else:
        s["w"] = got
        s["slot"] = torch.zeros(ops.expert_layout(case["fmt"], case["dim"], case["inter"])[0], dtype=U8, device="cuda")
    torch.cuda.synchronize()
    return s


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "gemv":
        return (ops.gemv_fp4 if c["fmt"] == FP4 else ops.gemv_fp8)(state["codes"], state["scales"], state["x"], out_f32=c["f32"])
    if kind == "gemv_batch":
        return ops.gemv_batch(state["codes"], state["scales"], state["xs"], c["fmt"])
    if kind == "abi_batch":
        return ops.stbl_gemv_mxfp4_batch(state["ys"], state["ws"], state["xs"], c["rows"], c["k"])
    if kind == "ffn":
        return ops.expert_ffn(state["slot"], state["x"], c["fmt"], c["dim"], c["inter"], official=c["official"])
    if kind == "moe":
        return ops.moe_experts(state["x"], state["slots"], state["pick"], state["weights"], FP4, c["dim"], c["inter"],
                               shared=c["n"], limit=c["limit"], official=c["official"], work=state["work"],
                               shared_fmt=c["shared_fmt"])
    if kind == "layer":
        return state["layer"].forward(state["x"], state["logits"])
    if kind == "gemm":
        if c["form"] == "q":
            return ops.gemm_q(state["codes"], state["scales"], state["aq"], state["as"], c["fmt"], c["block"], c["f32"])
        fn = ops.gemm_packed if c["form"] == "packed" else ops.gemm
        return fn(state["codes"], state["scales"], state["x"], c["fmt"], c["block"], c["f32"])
    if kind == "act_quant":
        return ops.act_quant(state["x"], c["block"], c["pow2"], c["deq"])
    return ops.quant_expert(*state["w"], c["fmt"], out=state["slot"])


def _mat(fmt, rows, k):
    """Bytes of one quantized matrix."""
    if fmt == FP4:
        return rows * k // 2 + rows * k // 32
    if fmt == FP8_E8M0:
        return rows * k + -(-rows // 32) * (k // 32)
    return rows * k + 4 * -(-rows // 128) * -(-k // 128)


def _expert_bytes(fmt, dim, inter):
    return 2 * _mat(fmt, inter, dim) + _mat(fmt, dim, inter)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemv", "gemv_batch"):
        n = c.get("n", 1)
        out = 4 if c.get("f32") else 2
        return {"bytes": n * (_mat(c["fmt"], c["rows"], c["k"]) + 2 * c["m"] * c["k"] + out * c["m"] * c["rows"]),
                "flops": 2 * n * c["m"] * c["rows"] * c["k"]}
    if kind == "abi_batch":
        return {"bytes": c["n"] * (c["rows"] * c["k"] // 32 * 17 + 4 * (c["k"] + c["rows"])),
                "flops": 2 * c["n"] * c["rows"] * c["k"]}
    if kind == "ffn":
        return {"bytes": _expert_bytes(c["fmt"], c["dim"], c["inter"]) + 4 * c["m"] * c["dim"],
                "flops": 6 * c["m"] * c["dim"] * c["inter"]}
    if kind in ("moe", "layer"):
        # distinct routed experts of a step: the mean over seeds
        if kind == "moe":
            hit = sum(len({e for row in _picks(c, s)[0] for e in row}) for s in range(8)) / 8
        else:
            hit = c["n"] * (1 - (1 - c["topk"] / c["n"]) ** c["t"])
        return {"bytes": hit * _expert_bytes(FP4, c["dim"], c["inter"]) + 4 * c["t"] * c["dim"]
                + _expert_bytes(c.get("shared_fmt", FP4), c["dim"], c["inter"]),
                "flops": 6 * c["t"] * (c["topk"] + 1) * c["dim"] * c["inter"]}
    if kind == "gemm":
        a = c["m"] * c["k"] + c["m"] * c["k"] // c["block"] if c["form"] == "q" else 2 * c["m"] * c["k"]
        return {"bytes": a + _mat(c["fmt"], c["n"], c["k"]) + (4 if c["f32"] else 2) * c["m"] * c["n"],
                "flops": 2 * c["m"] * c["n"] * c["k"]}
    if kind == "act_quant":
        n = c["rows"] * c["n"]
        return {"bytes": 2 * n + n + 4 * n // c["block"] + (2 * n if c["deq"] else 0), "flops": 0}
    return {"bytes": 12 * c["dim"] * c["inter"] + _expert_bytes(c["fmt"], c["dim"], c["inter"]), "flops": 0}


def tolerance(case):
    """About four times the distance from the 64-bit result that the path shows over the ranges."""
    kind = case["kind"]
    if kind in ("act_quant", "load"):
        return "exact"  # codes and scales are whole numbers, and fp32 values of one rounding each
    if kind == "gemm" and case["f32"]:
        # the scaled MFMA keeps the sum inside a 128-wide step less exactly than fp32: 1.5e-5, 1.1e-4
        return {"rel": 6e-5, "max": 4.5e-4}
    if case.get("f32"):
        return {"rel": 1e-6, "max": 1e-5}  # fp32 sums: 1e-7, 3e-7
    if kind in ("gemv", "gemv_batch", "abi_batch", "gemm"):
        return {"rel": 6.5e-3, "max": 1.6e-2}  # rounded once to bf16: 1.65e-3, 3.9e-3
    return {"rel": 9e-3, "max": 3.5e-2}  # bf16 between an expert's stages and in the sum: 2.25e-3, 8.8e-3


def exact(case, seed):
    c, kind = case, case["kind"]
    got = _inputs(case, seed)
    if kind == "gemv":
        codes, scales, x = got
        return x.to(F64) @ _dequant(codes, scales, c["fmt"]).T
    if kind == "gemv_batch":
        return [x.to(F64) @ _dequant(w, s, c["fmt"]).T for w, s, x in zip(*got)]
    if kind == "abi_batch":
        q, xs = got
        return [_dequant(w, s, FP4) @ x.to(F64) for (w, s), x in zip(q, xs)]
    if kind == "ffn":
        parts, x = got
        return _ffn(parts, x, c["fmt"], torch.ones((c["m"], 1), dtype=F64, device="cuda"), 0.0, c["official"])
    if kind in ("moe", "layer"):
        experts, shared, x = got[:3]
        if kind == "moe":
            pick, w = _picks(c, seed)
        else:
            score = torch.sigmoid(got[3].to(F64))
            top = score.topk(c["topk"], -1)
            pick, w = top.indices.tolist(), (top.values / top.values.sum(-1, keepdim=True)).tolist()
        limit, official, sfmt = c.get("limit", 0.0), c.get("official", False), c.get("shared_fmt", FP4)
        y = _ffn(shared, x, sfmt, torch.ones((c["t"], 1), dtype=F64, device="cuda"), limit, official)
        for e in sorted({e for row in pick for e in row}):
            toks = [i for i, row in enumerate(pick) if e in row]
            wt = torch.tensor([[w[i][pick[i].index(e)]] for i in toks], dtype=F64, device="cuda")
            y[toks] += _ffn(experts[e], x[toks], FP4, wt, limit, official).to(BF16).to(F64)
        return y
    if kind == "gemm":
        codes, scales, x = got
        return _act_values(x, c["block"]) @ _dequant(codes, scales, c["fmt"]).T
    if kind == "act_quant":
        f, s = _act_scales(got, c["block"], c["pow2"])
        out = [None, s.to(F64)]
        return out + [(_e4m3(f / s[..., None]).to(F64) * s.to(F64)[..., None]).view(got.shape)] if c["deq"] else out
    return None
