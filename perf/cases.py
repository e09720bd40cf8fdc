"""The workloads this framework is timed on: its public calls over the sizes that programs use them at.

Shapes come from the DiT configurations (hidden 3072, 24 heads, 4096 image + 256 text tokens; the step drivers' hidden
4096, 32 heads, 4096 target rows over a 4128-row prefix), the text encoder (hidden 4096, 32 / 8 heads, FFN 12288, prompt
rows padded to a multiple of 512) and their neighbours. Weights ~N(0, 0.02), activations ~N(0, 1), everything made on
the GPU from the seed. ``exact`` restates each call in float64 torch: the bfp16 and bf16 roundings that the calls
define (operands, stored intermediates) are applied, sums and functions are float64.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "redline-tiny_amd"))

from rlbfp import forward, host_glue, layouts, ops, run_ln, run_qkv, vlm_run  # noqa: E402

BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
LOG2E = math.log2(math.e)


# ---------------------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------------------

def listed():
    return [
        # the adaLN modulation of one DiT block: one timestep embedding against the shared projection, once per step
        {"name": "modulation", "kind": "gemv", "M": 1, "K": 3072, "N": 18432, "silu": True},
        # encoding a block's activations before its first GEMM (packed bytes and the GEMM's bf16 operand)
        {"name": "act_encode", "kind": "encode", "rows": 4352, "cols": 3072, "order": "rowblock", "dtype": "bf16",
         "deq": True},
        # a short, odd-length prompt through one projection with a bias
        {"name": "text_proj", "kind": "gemm", "M": 77, "K": 4096, "N": 4096, "act": "none", "bias": True, "gate": False,
         "a_fmt": "bf16"},
        # the DiT's joint QKV projection, 1% outlier channels in its input
        {"name": "dit_qkv", "kind": "gemm", "M": 4352, "K": 3072, "N": 9216, "act": "none", "bias": True, "gate": False,
         "a_fmt": "bf16"},
        # the DiT FFN: encode x, up GEMM with SwiGLU and re-quantized H, down GEMM with gate and residual
        {"name": "dit_ffn", "kind": "ffn", "M": 4352, "hid": 3072, "ff": 12288, "gated": True},
        # the text encoder's prefill MLP at 512 prompt rows
        {"name": "te_mlp", "kind": "ffn", "M": 512, "hid": 4096, "ff": 12288, "gated": False},
        # the image and text streams' QKV projections (separate weights) in one grouped call
        {"name": "dit_streams", "kind": "grouped", "Ms": "4096,256", "K": 3072, "N": 9216},
        # joint attention of the DiT from the QKV GEMM's output: per-head norm, RoPE, softmax(QK)V
        {"name": "dit_attention", "kind": "attention", "M": 4352, "heads": 24, "nkv": 4352, "causal": False},
        # residual + LayerNorm + modulate between the DiT's GEMMs
        {"name": "dit_norm", "kind": "norm", "M": 4352, "D": 3072, "norm": "layer", "branch": "bf16", "packed": False,
         "deq": True, "split": 256},
        # the same op as the step drivers issue it, on the packed and C-ordered streams
        {"name": "step_norm", "kind": "stream_norm", "M": 4096, "D": 4096, "split": 0, "branch": "packed"},
        # the attention half of a cached DiT step as forward.py issues it: QKV, QKV post, attention over the target
        # and the cached prefix (last tile padded), out-projection, on packed streams
        {"name": "step_attention", "kind": "stream_attention", "M": 4096, "heads": 32, "prefix": 65, "pad": 32},
        # one text-encoder layer (norms, QKV, causal grouped-query attention, MLP) on a 1070-token prompt
        {"name": "te_layer", "kind": "te_layer", "m": 1536, "hq": 32, "hkv": 8, "ff": 12288, "length": 1070},
    ]


def _spread(rng, lo, hi, step):
    """A multiple of step in lo..hi, spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(max(round(v / step), -(-lo // step)), hi // step)) * step


def draw(rng):
    kind = rng.choice(["gemv", "encode", "decode", "gemm", "gemm", "ffn", "grouped", "attention", "norm",
                       "stream_norm", "stream_attention", "te_layer"])
    if kind == "gemv":
        return {"kind": kind, "M": rng.choice([1, 1, 2, 2, 3, 4, 5, 6, 7, 8]), "K": _spread(rng, 256, 8192, 64),
                "N": _spread(rng, 512, 24576, 128), "silu": rng.random() < 0.7}
    if kind in ("encode", "decode"):
        order = rng.choice(["rowblock", "rowblock", "a_layout", "b_layout", "c_atb"])
        rstep, cstep = {"rowblock": (1, 8), "a_layout": (128, 64), "b_layout": (128, 64), "c_atb": (512, 1024)}[order]
        c = {"kind": kind, "rows": _spread(rng, max(rstep, 16), 8704, rstep),
             "cols": _spread(rng, max(cstep, 64), 12288, cstep), "order": order, "dtype": rng.choice(["bf16", "f32"])}
        if kind == "encode":
            c["deq"] = order == "rowblock" and rng.random() < 0.5
        return c
    if kind == "gemm":
        while True:
            c = {"kind": kind, "M": _spread(rng, 1, 4608, 1), "K": _spread(rng, 256, 12288, 64),
                 "N": _spread(rng, 256, 24576, 128), "act": rng.choice(["none", "none", "gelu_tanh", "swiglu"]),
                 "bias": rng.random() < 0.5, "gate": rng.random() < 0.4,
                 "a_fmt": rng.choice(["bf16", "bf16", "bf16_quantize", "packed_rowblock"])}
            if c["M"] * c["K"] * c["N"] <= 4352 * 3072 * 24576:
                return c
    if kind == "ffn":
        return {"kind": kind, "M": _spread(rng, 32, 4352, 1), "hid": 128 * rng.randint(8, 24),
                "ff": _spread(rng, 2048, 12288, 64), "gated": rng.random() < 0.5}
    if kind == "grouped":
        return {"kind": kind, "Ms": ",".join(str(_spread(rng, 16, 4096 if i == 0 else 1024, 1))
                                             for i in range(rng.randint(2, 4))),
                "K": 64 * rng.randint(16, 48), "N": 128 * rng.randint(16, 72)}
    if kind == "attention":
        M = 128 * rng.randint(1, 34)
        return {"kind": kind, "M": M, "heads": rng.randint(1, 24), "nkv": rng.randint(max(1, M - 200), M),
                "causal": rng.random() < 0.4}
    if kind == "norm":
        return {"kind": kind, "M": _spread(rng, 16, 8704, 1), "D": _spread(rng, 512, 8192, 64),
                "norm": rng.choice(["layer", "rms"]), "branch": rng.choice(["none", "bf16", "bf16", "packed"]),
                "packed": rng.random() < 0.5, "deq": True, "split": rng.choice([0, 0, 100])}
    if kind == "stream_norm":
        return {"kind": kind, "M": 512 * rng.randint(1, 17), "D": 1024 * rng.randint(1, 4),
                "split": 128 * rng.choice([0, 0, 1, 3]), "branch": rng.choice(["packed", "packed", "bf16"])}
    if kind == "stream_attention":
        return {"kind": kind, "M": 512 * rng.randint(1, 8), "heads": 8 * rng.randint(1, 3),
                "prefix": rng.randint(1, 66), "pad": rng.randint(0, 63)}
    m = 512 * rng.randint(1, 3)
    return {"kind": "te_layer", "m": m, "hq": 8 * rng.randint(1, 3), "hkv": rng.choice([4, 8]),
            "ff": 1024 * rng.randint(2, 12), "length": rng.randint(1, m)}


# ---------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=F32) * std

    def angles(self, rows):
        a = (torch.rand((rows, 64), generator=self.g, device="cuda", dtype=F32) * 2 - 1) * math.pi
        return torch.cos(a).to(BF), torch.sin(a).to(BF)


def _ms(case):
    return [int(m) for m in case["Ms"].split(",")]


def _inputs(case, seed):
    """The raw operands of a case, before any packing: shared by prepare and exact."""
    r, k, d = _Rand(seed), case["kind"], {}
    if k == "gemv":
        d["x"] = r.normal(case["M"], case["K"]).to(BF)
        d["W"] = r.normal(case["N"], case["K"], std=0.02)
    elif k in ("encode", "decode"):
        d["x"] = r.normal(case["rows"], case["cols"])
        if case["dtype"] == "bf16":
            d["x"] = d["x"].to(BF)
    elif k == "gemm":
        x = r.normal(case["M"], case["K"])
        x[:, ::100] *= 20.0
        d["x"] = x.to(BF)
        d["W"] = r.normal(case["N"], case["K"], std=0.02)
        nout = case["N"] // 2 if case["act"] == "swiglu" else case["N"]
        d["bias"] = r.normal(case["N"], std=0.1) if case["bias"] else None
        d["gate"] = r.normal(nout) if case["gate"] else None
        d["res"] = r.normal(case["M"], nout).to(BF) if case["gate"] else None
    elif k == "ffn":
        M, hid, ff = case["M"], case["hid"], case["ff"]
        d["x"] = r.normal(M, hid).to(BF)
        d["Wg"], d["Wp"] = r.normal(ff, hid, std=0.02), r.normal(ff, hid, std=0.02)
        d["Wd"] = r.normal(hid, ff, std=0.02)
        if case["gated"]:
            d["gate"], d["res"] = r.normal(2, hid), r.normal(M, hid).to(BF)
    elif k == "grouped":
        d["xs"] = [r.normal(m, case["K"]).to(BF) for m in _ms(case)]
        d["Ws"] = [r.normal(case["N"], case["K"], std=0.02) for _ in _ms(case)]
        d["bs"] = [r.normal(case["N"], std=0.1) for _ in _ms(case)]
    elif k == "attention":
        M, h = case["M"], case["heads"]
        d["C"] = r.normal(M, 3 * h * 128).to(BF)
        d["cos"], d["sin"] = r.angles(M)
        d["wq"] = ((1 + r.normal(128, std=0.1)) * (LOG2E / math.sqrt(128))).to(BF)
        d["wk"] = (1 + r.normal(128, std=0.1)).to(BF)
    elif k in ("norm", "stream_norm"):
        M, D = case["M"], case["D"]
        d["x"] = (2 * r.normal(M, D)).to(BF)
        d["br"] = r.normal(M, D).to(BF) if case["branch"] != "none" else None
        d["g"], d["sc"] = torch.tanh(r.normal(2, D)), 1 + r.normal(2, D, std=0.3)
    elif k == "stream_attention":
        M, h = case["M"], case["heads"]
        hid = h * 128
        d["x"] = r.normal(M, hid).to(BF)
        d["Wqkv"], d["Wo"] = r.normal(3 * hid, hid, std=0.02), r.normal(hid, hid, std=0.02)
        d["cos"], d["sin"] = r.angles(M)
        d["wq"] = ((1 + r.normal(128, std=0.1)) * (LOG2E / math.sqrt(128))).to(BF)
        d["wk"] = (1 + r.normal(128, std=0.1)).to(BF)
        p = case["prefix"] * 64
        d["pC"] = r.normal(p, 3 * hid).to(BF)  # the prefix tokens' QKV rows, which its cache is made from
        d["pcos"], d["psin"] = r.angles(p)
    elif k == "te_layer":
        D, nqkv, ff = case["hq"] * 128, (case["hq"] + 2 * case["hkv"]) * 128, case["ff"]
        d["x"] = 2 * r.normal(case["length"], D)
        d["Wqkv"], d["Wo"] = r.normal(nqkv, D, std=0.02), r.normal(D, D, std=0.02)
        d["Wg"], d["Wp"] = r.normal(ff, D, std=0.02), r.normal(ff, D, std=0.02)
        d["Wd"] = r.normal(D, ff, std=0.02)
        d["wq"], d["wk"] = 1 + r.normal(128, std=0.2), 1 + r.normal(128, std=0.2)
        d["n_in"], d["n_post"] = 1 + r.normal(D, std=0.2), 1 + r.normal(D, std=0.2)
        d["cos"], d["sin"] = r.angles(case["m"])
    return d


class _LayerWeights:
    """One text-encoder layer's packed weights, in the form vlm_run.LM takes them."""

    def __init__(self, d, D):
        self.w = {(0, "qkv"): ops.pack_weight(d["Wqkv"]), (0, "o"): ops.pack_weight(d["Wo"]),
                  (0, "up"): ops.pack_weight(ops.interleave_up(d["Wg"], d["Wp"]).contiguous()),
                  (0, "down"): ops.pack_weight(d["Wd"])}
        self.qk = {0: (d["wq"], d["wk"])}
        self.p_in = {0: vlm_run.rms_params(d["n_in"])}
        self.p_post = {0: vlm_run.rms_params(d["n_post"])}
        self.hp = list(range(D))  # the model's channel order is the packed weights' own


def prepare(case, seed):
    d, k = _inputs(case, seed), case["kind"]
    s = {"case": case}
    if k == "gemv":
        s["w"] = {"modulation.1.weight": host_glue.pack_linear(d["W"]), "modulation.N": case["N"]}
        s["x"], s["b"] = d["x"], s["w"]["modulation.1.weight"]
    elif k == "encode":
        s["x"] = d["x"]
    elif k == "decode":
        s["p"] = ops.quantize(d["x"], order=case["order"])[0]
    elif k == "gemm":
        s["b"] = ops.pack_weight(d["W"])
        if case["a_fmt"] == "bf16":
            s["a"] = ops.quantize(d["x"], packed=False, deq=True)[1]
        elif case["a_fmt"] == "bf16_quantize":
            s["a"] = d["x"]
        else:
            s["a"] = ops.quantize(d["x"])[0]
        s.update(bias=d["bias"], gate=d["gate"], res=d["res"])
    elif k == "ffn":
        s["x"] = d["x"]
        s["up"] = ops.pack_weight(ops.interleave_up(d["Wg"], d["Wp"]).contiguous())
        s["down"] = ops.pack_weight(d["Wd"])
        s["ep"] = {"gate": d["gate"], "gate_split_row": _split(case), "residual": d["res"]} if case["gated"] else {}
    elif k == "grouped":
        s["as"] = [ops.quantize(x, packed=False, deq=True)[1] for x in d["xs"]]
        s["bs"], s["bias"] = [ops.pack_weight(W) for W in d["Ws"]], d["bs"]
    elif k == "attention":
        s.update(d)
        s["lim"] = torch.arange(case["M"], dtype=torch.int32, device="cuda") if case["causal"] else None
    elif k == "norm":
        s["x"], s["params"] = d["x"], run_ln.ln_params(d["g"], d["sc"]).reshape(2, -1)
        s["br"] = ops.quantize(d["br"])[0] if case["branch"] == "packed" else d["br"]
    elif k == "stream_norm":
        n = case["M"] * case["D"]
        s["art"] = "glue-ln-m%d-s%d" % (case["M"], case["split"] // 128)
        s["x"], s["p"] = run_ln.ln_pack_x(d["x"]), run_ln.ln_params(d["g"], d["sc"])
        s["br"] = run_ln.ln_pack_br(d["br"]) if case["branch"] == "packed" else run_ln.ln_pack_x(d["br"])
        s["xo"], s["ao"] = torch.zeros(n, dtype=BF, device="cuda"), forward.v9(n)
    elif k == "stream_attention":
        M, h, pt = case["M"], case["heads"], case["prefix"]
        hid = h * 128
        s["a"] = layouts.to_bfp16_a_layout(d["x"])
        s["wqkv"], s["wo"] = ops.pack_weight(d["Wqkv"]), ops.pack_weight(d["Wo"])
        s["tabs"] = run_qkv.qkv_tables(d["cos"], d["sin"], d["wq"], d["wk"]).reshape(-1)
        s["prefix"] = ops.qkv_post(d["pC"], d["pcos"], d["psin"], d["wq"], d["wk"], h)[1].reshape(-1)
        s["meta"] = {"family": "attn32o", "H": h, "QN": M // 64, "MQ": 64, "NT": 64, "NK": M + 64 * pt,
                     "NKV": M + 64 * pt - case["pad"], "OA": 1, "OHEADS": h, "H0": 0, "KVSPLIT": M // 64, "PT": pt,
                     "P0": 0}
        s["c"], s["q"], s["kv"] = forward.v9(3 * M * hid), forward.v9(M * hid), forward.v9(2 * M * hid)
        s["o"], s["y"] = forward.v9(M * hid), torch.zeros((M, hid), dtype=BF, device="cuda")
    elif k == "te_layer":
        D = case["hq"] * 128
        s["lm"] = vlm_run.LM(_LayerWeights(d, D), d["cos"], d["sin"], m=case["m"], hq=case["hq"], hkv=case["hkv"],
                             length=case["length"])
        s["x"] = d["x"]
    return s


def _split(case):
    return min(256, case["M"] // 2)


# ---------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "gemv":
        if case["silu"]:
            return host_glue.modulation(state["w"], state["x"])
        return ops.gemv(state["x"], state["b"], case["N"], act=None)
    if k == "encode":
        return ops.quantize(state["x"], order=case["order"], packed=True, deq=case["deq"])
    if k == "decode":
        return ops.dequantize(state["p"], case["rows"], case["cols"], order=case["order"],
                              dtype=BF if case["dtype"] == "bf16" else F32)
    if k == "gemm":
        return ops.gemm(state["a"], state["b"], case["N"], case["K"], M=case["M"], a_fmt=case["a_fmt"],
                        act=case["act"], bias=state["bias"], gate=state["gate"], residual=state["res"])
    if k == "ffn":
        hid, ff = case["hid"], case["ff"]
        _, a = ops.quantize(state["x"], packed=False, deq=True)
        h = ops.gemm(a, state["up"], 2 * ff, hid, act="swiglu", quantize_out=True)
        return {"h": h, "y": ops.gemm(h, state["down"], hid, ff, **state["ep"])}
    if k == "grouped":
        return ops.gemm_grouped([ops.GemmSpec(a, b, case["N"], case["K"], bias=v)
                                 for a, b, v in zip(state["as"], state["bs"], state["bias"])])
    if k == "attention":
        _, _, q, kk, vt = ops.qkv_post(state["C"], state["cos"], state["sin"], state["wq"], state["wk"], case["heads"],
                                       tiles=False, native=True)
        return {"k": kk, "vt": vt,
                "o": ops.attention(q, kk, vt, nkv=case["nkv"], lim=state["lim"], quantize_out=True)}
    if k == "norm":
        x, p, a = ops.ln_modulate(state["x"], state["params"], branch=state["br"], split_row=case["split"],
                                  norm=case["norm"], packed=case["packed"], deq=case["deq"])
        return {"x": x, "packed": p, "a": a}
    if k == "stream_norm":
        run_ln.ln_fused(state["art"], state["x"], state["br"], state["p"], state["xo"], state["ao"])
        return {"x": state["xo"], "a": state["ao"]}
    if k == "stream_attention":
        s, M = state, case["M"]
        npu = forward.NPU()
        npu.meta["attn"] = s["meta"]
        npu.run("qkv", "qkv", [s["a"], s["wqkv"], s["c"]])
        npu.run("qkv_post", "glue-qkv32-m%d" % M, [s["c"], s["tabs"], s["q"], s["kv"]])
        npu.run("attn", "attn", [s["q"], s["kv"], s["prefix"], s["o"]])
        npu.run("o", "o", [s["o"], s["wo"], s["y"]])
        return {"kv": s["kv"], "y": s["y"]}
    lm = state["lm"]
    lm.load_x(state["x"])
    lm.layer(0)
    return lm.x_out(0)


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------

def _gemm_work(M, N, K, nout, a=2.0, c=2.0):
    """(bytes, flops) of one GEMM: A, the packed weights, C."""
    return M * K * a + N * K * 9 / 8 + M * nout * c, 2.0 * M * N * K


def _pairs(nq, nkv, causal):
    return sum(min(i + 1, nkv) for i in range(nq)) if causal else nq * nkv


def work(case):
    k = case["kind"]
    if k == "gemv":
        b, f = _gemm_work(case["M"], case["N"], case["K"], case["N"])
    elif k in ("encode", "decode"):
        n, e = case["rows"] * case["cols"], 2 if case["dtype"] == "bf16" else 4
        b, f = n * (e + 9 / 8 + (2 if case.get("deq") else 0)), 0.0
    elif k == "gemm":
        nout = case["N"] // 2 if case["act"] == "swiglu" else case["N"]
        b, f = _gemm_work(case["M"], case["N"], case["K"], nout, a=9 / 8 if "packed" in case["a_fmt"] else 2.0)
        b += case["M"] * nout * 2 if case["gate"] else 0
    elif k == "ffn":
        M, hid, ff = case["M"], case["hid"], case["ff"]
        b = M * hid * 2 + 3 * hid * ff * 9 / 8 + M * ff * 2 + M * hid * (4 if case["gated"] else 2)
        f = 6.0 * M * hid * ff
    elif k == "grouped":
        b = f = 0.0
        for m in _ms(case):
            bb, ff = _gemm_work(m, case["N"], case["K"], case["N"])
            b, f = b + bb, f + ff
    elif k == "attention":
        M, h = case["M"], case["heads"]
        b = M * 3 * h * 128 * 2 + M * 256 + 3 * M * h * 128 * 2
        f = 4.0 * 128 * h * _pairs(M, case["nkv"], case["causal"])
    elif k == "norm":
        br = {"none": 0, "bf16": 2, "packed": 9 / 8}[case["branch"]]
        b, f = case["M"] * case["D"] * (2 + br + 2 + (9 / 8 if case["packed"] else 0) + (2 if case["deq"] else 0)), 0.0
    elif k == "stream_norm":
        b = case["M"] * case["D"] * (2 + (9 / 8 if case["branch"] == "packed" else 2) + 2 + 9 / 8)
        f = 0.0
    elif k == "stream_attention":
        M, hid, p = case["M"], case["heads"] * 128, case["prefix"] * 64
        b = (M * hid + 4 * hid * hid + 2 * p * hid + 2 * M * hid) * 9 / 8 + M * hid * 2
        f = 8.0 * M * hid * hid + 4.0 * 128 * case["heads"] * M * (M + p - case["pad"])
    else:
        m, D, ff = case["m"], case["hq"] * 128, case["ff"]
        nq = -(-case["length"] // 64) * 64
        n = D * (case["hq"] + 2 * case["hkv"]) * 128 + D * D + 3 * D * ff
        b = n * 9 / 8 + case["length"] * D * 4 + m * D * 4
        f = 2.0 * m * n + 4.0 * 128 * case["hq"] * _pairs(nq, nq, True)
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    k = case["kind"]
    if k in ("encode", "decode"):
        return "exact"
    if k in ("norm", "stream_norm"):
        # y is bfp16 (7 bits below the block's maximum): a value at a rounding tie may take either side
        return {"rel": 3e-3, "max": 0.1, "differ": 2e-3}
    if k in ("attention", "stream_attention"):
        # O is bfp16 and 0.5-0.9% off float64 (P is bf16, O's rounding); K and V tiles are bytes
        return {"rel": 2e-2, "max": 0.2, "differ": 2e-3}
    if k == "te_layer":
        return {"rel": 2.5e-2, "max": 0.3}  # attention and four stored intermediates: 0.6-0.9% off float64
    if k == "ffn":
        return {"rel": 1.2e-2, "max": 0.2}  # ties of the re-quantized H, then one bf16 rounding
    return {"rel": 8e-3, "max": 0.1}  # one bf16 rounding: 0.2% off float64


# ---------------------------------------------------------------------------------------------------------------
# float64 restatement
# ---------------------------------------------------------------------------------------------------------------

def _bfp(x):
    """x rounded to bfp16 blocks of 8 consecutive values of the last dim, in float64: the block's exponent is the
    float32 exponent field of its largest magnitude, steps of 2^(E - 133), half to even, clipped to -128 .. 127."""
    b = x.to(F64).reshape(-1, 8)
    m = b.abs().amax(1, keepdim=True).to(F32)
    E = (m.view(torch.int32) >> 23) & 0xFF
    step = ((E.to(torch.int64) + (1023 - 133)) << 52).view(F64)  # 2^(E - 133)
    return (torch.clamp(torch.round(b / step), -128, 127) * step).reshape(x.shape)


def _round(x):
    return x.to(F32).to(BF).to(F64)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _mm(a, W):
    """a (float64, its values as the product takes them) against the Linear weight W, bfp16 along K."""
    return a @ _bfp(W).t()


def _swiglu(a, Wg, Wp):
    return _silu(_mm(a, Wg)) * _mm(a, Wp)


def _head_norm(x, w, cos, sin):
    """Per-head RMSNorm * w and RoPE of x (rows, heads, 128), quantized to bfp16 along the dims."""
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.to(F64)
    a, b = y[..., 0::2], y[..., 1::2]
    c, s = cos.to(F64)[:, None], sin.to(F64)[:, None]
    out = torch.empty_like(y)
    out[..., 0::2], out[..., 1::2] = a * c - b * s, a * s + b * c
    return _bfp(out)


def _qkv(C, hq, hkv, cos, sin, wq, wk):
    """q, k (heads, rows, 128) and vt (heads, 128, rows) of the QKV rows C (float64)."""
    x = C.reshape(C.shape[0], hq + 2 * hkv, 128)
    q = _head_norm(x[:, :hq], wq, cos, sin).transpose(0, 1)
    k = _head_norm(x[:, hq:hq + hkv], wk, cos, sin).transpose(0, 1)
    return q, k, _bfp(x[:, hq + hkv:].permute(1, 2, 0).contiguous())


def _attend(q, k, vt, nkv, causal):
    """softmax2(q k^T) v per query head, (rows, heads * 128); grouped-query when k has fewer heads."""
    h, n = q.shape[:2]
    g, out = h // k.shape[0], []
    for i in range(h):
        s = q[i] @ k[i // g].t()
        s[:, nkv:] = -math.inf
        if causal:
            s += torch.full_like(s, -math.inf).triu(1)
        p = torch.exp2(s - s.amax(1, keepdim=True))
        out.append((p / p.sum(1, keepdim=True)) @ vt[i // g].t())
    return torch.stack(out, 1).reshape(n, h * 128)


def _norm(x, br, g, sc, split, kind):
    """x' = bf16(x + g br) and its norm * sc as bfp16; rows below split take parameter row 1."""
    row = torch.zeros(x.shape[0], dtype=torch.long, device=x.device)
    row[:split] = 1
    g, sc = g.to(BF).to(F64)[row], sc.to(BF).to(F64)[row]
    xp = _round(x.to(F64) + g * br) if br is not None else x.to(F64)
    mean = xp.mean(1, keepdim=True) if kind == "layer" else 0.0
    var = ((xp - mean) ** 2).mean(1, keepdim=True)
    return xp, _bfp((xp - mean) / torch.sqrt(var + 1e-6) * sc)


def exact(case, seed):
    d, k = _inputs(case, seed), case["kind"]
    if k == "gemv":
        x = d["x"].to(F64)
        return _mm(_bfp(_silu(x) if case["silu"] else x), d["W"])
    if k == "encode":
        return [None, _bfp(d["x"]) if case["deq"] else None]
    if k == "decode":
        # blocks run along the columns in every order (b_layout: K, the columns of the Linear weight)
        return _bfp(d["x"])
    if k == "gemm":
        v = _mm(_bfp(d["x"]), d["W"])
        if case["bias"]:
            v += d["bias"].to(F64)
        if case["act"] == "swiglu":
            v = v.reshape(case["M"], -1, 2, 64)
            v = (_silu(v[:, :, 0]) * v[:, :, 1]).reshape(case["M"], -1)
        elif case["act"] == "gelu_tanh":
            v = torch.nn.functional.gelu(v, approximate="tanh")
        return d["res"].to(F64) + d["gate"].to(F64) * v if case["gate"] else v
    if k == "ffn":
        h = _bfp(_round(_swiglu(_bfp(d["x"]), d["Wg"], d["Wp"])))
        y = _mm(h, d["Wd"])
        if case["gated"]:
            row = torch.zeros(case["M"], dtype=torch.long, device="cuda")
            row[:_split(case)] = 1
            y = d["res"].to(F64) + d["gate"].to(F64)[row] * y
        return {"h": h, "y": y}
    if k == "grouped":
        return [_mm(_bfp(x), W) + b.to(F64) for x, W, b in zip(d["xs"], d["Ws"], d["bs"])]
    if k == "attention":
        q, kk, vt = _qkv(d["C"].to(F64), case["heads"], case["heads"], d["cos"], d["sin"], d["wq"], d["wk"])
        return {"k": kk, "vt": vt, "o": _bfp(_attend(q, kk, vt, case["nkv"], case["causal"]))}
    if k == "norm":
        br = None if d["br"] is None else (_bfp(d["br"]) if case["branch"] == "packed" else d["br"].to(F64))
        xp, y = _norm(d["x"], br, d["g"], d["sc"], case["split"], case["norm"])
        return {"x": xp, "packed": None, "a": y if case["deq"] else None}
    if k == "stream_norm":
        br = _bfp(d["br"]) if case["branch"] == "packed" else d["br"].to(F64)
        return {"x": _c_order(_norm(d["x"], br, d["g"], d["sc"], case["split"], "layer")[0]), "a": None}
    if k == "stream_attention":
        h, M = case["heads"], case["M"]
        c = _bfp(_round(_mm(_bfp(d["x"]), d["Wqkv"])))
        q, kt, vt = _qkv(c, h, h, d["cos"], d["sin"], d["wq"], d["wk"])
        _, kp, vp = _qkv(d["pC"].to(F64), h, h, d["pcos"], d["psin"], d["wq"], d["wk"])
        n = M + 64 * case["prefix"] - case["pad"]
        o = _attend(q, torch.cat([kt, kp], 1), torch.cat([vt, vp], 2), n, False)
        return {"kv": None, "y": _mm(_bfp(o), d["Wo"])}
    m, D, n = case["m"], case["hq"] * 128, -(-case["length"] // 64) * 64
    one = torch.ones((2, D), device="cuda")
    x = torch.zeros((m, D), dtype=F64, device="cuda")
    x[:case["length"]] = _round(d["x"].to(F64))
    x1, a = _norm(x, None, one, d["n_in"].expand(2, D), 0, "rms")
    c = _bfp(_round(_mm(a, d["Wqkv"])))
    q, kk, vt = _qkv(c, case["hq"], case["hkv"], d["cos"], d["sin"],
                     (d["wq"].to(F64) * (LOG2E / math.sqrt(128))).to(BF), d["wk"].to(BF))
    o = torch.zeros((m, D), dtype=F64, device="cuda")
    o[:n] = _bfp(_attend(q[:, :n], kk[:, :n], vt[:, :, :n], n, True))
    x2, a = _norm(x1, _bfp(_round(_mm(o, d["Wo"]))), one, d["n_post"].expand(2, D), 0, "rms")
    h = _bfp(_round(_swiglu(a, d["Wg"], d["Wp"])))
    return _round(x2 + _bfp(_round(_mm(h, d["Wd"]))))


def _c_order(x):
    """(M, N) in the C stream's element order: 512 x 1024 groups, 128-column then 128-row tiles, 16 x 16 blocks of
    2 x 2 8 x 8 cells."""
    M, N = x.shape
    t = x.reshape(M // 512, 4, 8, 2, 8, N // 1024, 8, 8, 2, 8)  # rg, row, sbr, br, rib, cg, col, sbc, bc, cib
    return t.permute(0, 5, 6, 1, 2, 7, 3, 8, 4, 9).reshape(-1)
