"""Performance cases of the fused-group entry points: what a program that uses
this framework has it run, from one small matmul to a whole network.

A case is a plain dict.  `prepare` makes its inputs on the GPU from a seed,
`run` is one pass through the public entry points, `exact` the same result in
64-bit arithmetic without this package, `work` the bytes and operations a pass
cannot do without and `tolerance` what another correct implementation at the
same precision may differ by.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "npu-dialect_amd"))

from npu_amd import configs, groups, lower, model_zoo  # noqa: E402

F32, F64, BF16 = torch.float32, torch.float64, torch.bfloat16


def listed():
    return [
        # One fill -> matmul -> bias + ReLU group at the size of the reference's
        # own matmul workload: the smallest call, where the launch counts.
        {"name": "matmul_256x512x256", "kind": "matmul", "M": 256, "K": 512, "N": 256,
         "bias": True, "act": "relu"},
        # The same group as the layer of an MLP over a few thousand rows, the
        # rows and columns no multiple of a tile.
        {"name": "matmul_2000x1024x3000", "kind": "matmul", "M": 2000, "K": 1024, "N": 3000,
         "bias": True, "act": "relu"},
        # 3x3 convolution, NHWC, batch 32, f32: bench.py's headline block.
        {"name": "conv3x3_f32_n32", "kind": "conv_nhwc", "dtype": "f32", "B": 32, "H": 56, "W": 56,
         "C": 64, "F": 64, "k": 3, "bias": True, "res": False, "act": "relu"},
        # The second 3x3 convolution of a ResNet basic block in bf16, with the
        # block's input added: a channel count and option besides the headline's.
        {"name": "conv3x3_bf16_res_n32", "kind": "conv_nhwc", "dtype": "bf16", "B": 32, "H": 28,
         "W": 28, "C": 128, "F": 128, "k": 3, "bias": True, "res": True, "act": "relu"},
        # The reference's own layout, NCHW: a ResNet block's second convolution
        # with its add and ReLU, a batch of eight.
        {"name": "conv_nchw_res_n8", "kind": "conv_nchw", "B": 8, "H": 56, "W": 56, "C": 64, "F": 64,
         "k": 3, "stride": 1, "bias": True, "res": True, "act": "relu"},
        # A whole network as the reference's model zoo writes it, lowered from its
        # linalg text: one image, 22 groups, the logits.
        {"name": "resnet18", "kind": "model", "model": "resnet18"},
        # MobileNetV2's inverted residual block at its second stage, batch 32 ...
        {"name": "irb_24x144_n32", "kind": "irb", "B": 32, "H": 56, "W": 56, "C": 24, "E": 144},
        # ... and at the 14x14 stage, where most of the network's blocks are.
        {"name": "irb_64x384_n32", "kind": "irb", "B": 32, "H": 14, "W": 14, "C": 64, "E": 384},
        # The int8 ResNet-50 bottleneck of the first stage, batch 32 ...
        {"name": "qbottleneck_256x64_n32", "kind": "qbottleneck", "B": 32, "H": 56, "W": 56,
         "C": 256, "M1": 64},
        # ... and of the 14x14 stage, which holds most of the network's blocks.
        {"name": "qbottleneck_1024x256_n32", "kind": "qbottleneck", "B": 32, "H": 14, "W": 14,
         "C": 1024, "M1": 256},
        # One decoder layer over a prompt of 512 tokens, the size of the tests and
        # the benchmark: five short launches.
        {"name": "llama_layer_s512", "kind": "llama", "S": 512, "D": 512, "heads": 8, "ffn": 1408},
        # The same over a long prompt with a wider model.
        {"name": "llama_layer_s2048", "kind": "llama", "S": 2048, "D": 768, "heads": 12, "ffn": 2048},
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))
    return max(lo, min(hi, int(v) // step * step))


def _fits(case, like):
    """Whether a drawn case costs no more than the listed one named `like`."""
    ref = next(c for c in listed() if c["name"] == like)
    w, r = work(case), work(ref)
    return w["bytes"] <= r["bytes"] and w["flops"] <= r["flops"]


def _draw_matmul(rng):
    return {"kind": "matmul", "M": _log_int(rng, 1, 2000), "K": _log_int(rng, 16, 2048, 4),
            "N": _log_int(rng, 4, 4096), "bias": rng.random() < 0.7,
            "act": rng.choice(["none", "relu", "relu6"])}


def _draw_conv_nhwc(rng):
    h = _log_int(rng, 7, 112)
    return {"kind": "conv_nhwc", "dtype": rng.choice(["f32", "bf16"]), "B": _log_int(rng, 1, 32),
            "H": h, "W": max(5, h + rng.randint(-2, 2)), "C": 8 * _log_int(rng, 2, 64),
            "F": _log_int(rng, 8, 512), "k": rng.choice([1, 3, 3, 5]), "bias": rng.random() < 0.7,
            "res": rng.random() < 0.4, "act": rng.choice(["none", "relu", "relu6"])}


def _draw_conv_nchw(rng):
    h = _log_int(rng, 7, 112)
    return {"kind": "conv_nchw", "B": _log_int(rng, 1, 16), "H": h, "W": max(7, h + rng.randint(-2, 2)),
            "C": _log_int(rng, 3, 512), "F": _log_int(rng, 8, 512), "k": rng.choice([1, 3, 3, 5, 7]),
            "stride": rng.choice([1, 1, 2]), "bias": rng.random() < 0.5, "res": rng.random() < 0.4,
            "act": rng.choice(["none", "relu"])}


def _draw_irb(rng):
    c, e = rng.choice([(16, 96), (24, 144), (32, 192), (64, 384), (96, 576), (160, 960)])
    h = _log_int(rng, 7, 56)
    return {"kind": "irb", "B": _log_int(rng, 1, 32), "H": h, "W": h + rng.randint(0, 3), "C": c, "E": e}


def _draw_qbottleneck(rng):
    c, m = rng.choice([(64, 64), (256, 64), (512, 128), (1024, 256), (2048, 512)])
    h = _log_int(rng, 7, 56)
    return {"kind": "qbottleneck", "B": _log_int(rng, 1, 32), "H": h, "W": h + rng.randint(0, 3),
            "C": c, "M1": m}


def _draw_llama(rng):
    dh = rng.choice([64, 64, 128])
    heads = rng.randint(1, 768 // dh)
    return {"kind": "llama", "S": _log_int(rng, 1, 2048), "D": dh * heads, "heads": heads,
            "ffn": 64 * _log_int(rng, 2, 32)}


def _draw_model(rng):
    return {"kind": "model", "model": rng.choice(["resnet18", "autoencoder", "autoencoder_deep",
                                                  "dcgan_generator"])}


_DRAWS = [(_draw_matmul, "matmul_2000x1024x3000"), (_draw_conv_nhwc, "conv3x3_f32_n32"),
          (_draw_conv_nchw, "resnet18"), (_draw_irb, "irb_24x144_n32"),
          (_draw_qbottleneck, "qbottleneck_256x64_n32"), (_draw_llama, "llama_layer_s2048"),
          (_draw_model, "resnet18")]


def draw(rng):
    make, like = _DRAWS[rng.choices(range(len(_DRAWS)), weights=[3, 3, 3, 2, 2, 3, 1])[0]]
    while True:
        case = make(rng)
        if _fits(case, like):
            return case


# ---- the networks, as the 64-bit result computes them ------------------------
def _resnet18_layers():
    """(filter name, F, C, k, stride, pad) in the order of the network's
    parameters, the shortcut convolutions included."""
    ls = [("w_conv1", 64, 3, 7, 2, 3), ("w_pool", 64, 64, 3, 2, 1)]
    ic = 64
    for s, oc in enumerate([64, 128, 256, 512]):
        for b in range(2):
            st = 2 if s and b == 0 else 1
            ls += [(f"w_s{s}_b{b}_c1", oc, ic, 3, st, 1), (f"w_s{s}_b{b}_c2", oc, oc, 3, 1, 1)]
            if ic != oc:
                ls.append((f"w_s{s}_b{b}_sc", oc, ic, 1, st, 0))
            ic = oc
    return ls + [("w_fc", 1000, 512, 7, 1, 0)]


_DCGAN = [(512, True), (256, True), (128, True), (64, True), (3, False)]  # 3x3, pad 1, [ReLU]
_AUTOENCODER = {"autoencoder": (784, [512, 256, 128, 64]),
                "autoencoder_deep": (1024, [1024, 512, 256, 128, 64, 32])}


def _model_params(name):
    """Parameter name -> (shape, fan-in); the first is the input."""
    if name == "resnet18":
        p = {"input": ([1, 3, 224, 224], 0)}
        for n, f, c, k, _, _ in _resnet18_layers():
            p[n] = ([f, c, k, k], c * k * k)
        return p
    if name == "dcgan_generator":
        p, c = {"input": ([1, 100, 4, 4], 0)}, 100
        for i, (oc, _) in enumerate(_DCGAN):
            p[f"w{i}"] = ([oc, c, 3, 3], 9 * c)
            c = oc
        return p
    din, sizes = _AUTOENCODER[name]
    p, prev = {"input": ([1, din], 0)}, din
    for i, s in enumerate(sizes):
        p[f"w_enc{i}"] = ([prev, s], prev)
        prev = s
    for i, s in enumerate(list(reversed(sizes[:-1])) + [din]):
        p[f"w_dec{i}"] = ([prev, s], prev)
        prev = s
    return p


def _model_flops(name):
    if name == "resnet18":
        total, h = 0, {}
        side = 224
        for n, f, c, k, st, pad in _resnet18_layers():
            src = h.get("block", side) if n.endswith("_sc") else side
            ho = (src + 2 * pad - k) // st + 1
            total += 2 * f * c * k * k * ho * ho
            if n.endswith("_c1"):
                h["block"] = side
            if not n.endswith("_sc"):
                side = ho
        return total
    ps = _model_params(name)
    out = 16 if name == "dcgan_generator" else 1
    return sum(2 * math.prod(s) * out for n, (s, _) in ps.items() if n != "input")


# ---- inputs -------------------------------------------------------------------
def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))

    def uni(shape, lo, hi):
        return torch.rand(shape, generator=g, device="cuda", dtype=F32) * (hi - lo) + lo

    def nrm(shape, sd):
        return torch.randn(shape, generator=g, device="cuda", dtype=F32) * sd

    k = case["kind"]
    if k == "matmul":
        return {"A": uni((case["M"], case["K"]), -1, 1), "B": uni((case["K"], case["N"]), -1, 1),
                "bias": uni((case["N"],), -1, 1) if case["bias"] else None}
    if k in ("conv_nhwc", "conv_nchw"):
        b, h, w, c, f, kk = (case[n] for n in ("B", "H", "W", "C", "F", "k"))
        ho, wo = _conv_out(case)
        nhwc = k == "conv_nhwc"
        d = {"x": uni((b, h, w, c) if nhwc else (b, c, h, w), 0, 1),
             "w": nrm((f, kk, kk, c) if nhwc else (f, c, kk, kk), math.sqrt(2 / (c * kk * kk))),
             "res": uni((b, ho, wo, f) if nhwc else (b, f, ho, wo), 0, 1) if case["res"] else None}
        if nhwc and case["dtype"] == "bf16":
            d = {n: None if t is None else t.to(BF16) for n, t in d.items()}
        d["bias"] = uni((f,), -0.1, 0.1) if case["bias"] else None
        return d
    if k == "model":
        return {n: uni(s, 0, 1) if not fan else nrm(s, math.sqrt(2 / fan))
                for n, (s, fan) in _model_params(case["model"]).items()}
    if k == "irb":
        c, e = case["C"], case["E"]
        return {"x": uni((case["B"], case["H"], case["W"], c), 0, 1), "we": nrm((e, c), math.sqrt(2 / c)),
                "wdw": nrm((3, 3, e), math.sqrt(2 / 9)), "wp": nrm((c, e), math.sqrt(2 / e))}
    if k == "qbottleneck":
        return _quantized(case, g, nrm)
    s, d, f = case["S"], case["D"], case["ffn"]
    bf = lambda shape, sd: nrm(shape, sd).to(BF16)
    dh = d // case["heads"]
    cos, sin = (torch.from_numpy(t).cuda() for t in configs.rope_tables(s, dh))
    return {"x": bf((s, d), 1.0), "wq": bf((d, d), 0.02), "wk": bf((d, d), 0.02),
            "wv": bf((d, d), 0.02), "wo": bf((d, d), 0.02), "wg": bf((d, f), 0.02),
            "wu": bf((d, f), 0.02), "wd": bf((f, d), 0.02), "g1": uni((d,), 0.5, 1.5),
            "g2": uni((d,), 0.5, 1.5), "cos_t": cos, "sin_t": sin}


def _quantized(case, g, nrm):
    """An int8 bottleneck as post-training quantization leaves it: filters
    per channel and symmetric, activation scales from the 99.9th percentile
    of the first image."""
    b, h, w, c, m = (case[n] for n in ("B", "H", "W", "C", "M1"))
    x = torch.randint(0, 128, (b, h, w, c), generator=g, device="cuda", dtype=torch.int8)

    def quant(wf):
        flat = wf.reshape(wf.shape[0], -1).to(F64)
        sc = flat.abs().amax(1) / 127
        return (flat / sc[:, None]).round().clamp(-127, 127).to(torch.int8).reshape(wf.shape), sc

    def multiplier(real):
        mm, ss = configs.quant_multiplier(real.cpu().numpy())
        return torch.from_numpy(mm).cuda(), torch.from_numpy(ss).cuda()

    w1, sw1 = quant(nrm((m, c), math.sqrt(2 / c)))
    w2, sw2 = quant(nrm((m, 3, 3, m), math.sqrt(2 / (9 * m))))
    w3, sw3 = quant(nrm((c, m), math.sqrt(2 / m)))
    sx = 1 / 127
    act_scale = lambda a: max(float(np.percentile(a.clamp(min=0).cpu().numpy(), 99.9)), 1e-6) / 127
    acc1 = _conv64(x[:1], w1.reshape(m, 1, 1, c), 0, 1)
    sy1 = act_scale(acc1 * (sx * sw1))
    m1, s1 = multiplier(sx * sw1 / sy1)
    acc2 = _conv64(_requant64(acc1, m1, s1).clamp(0, 127), w2, 1, 1)
    sy2 = act_scale(acc2 * (sy1 * sw2))
    m2, s2 = multiplier(sy1 * sw2 / sy2)
    m3, s3 = multiplier(sy2 * sw3 / sx)
    return {"x": x, "w1": w1, "w2": w2, "w3": w3, "m1": m1, "s1": s1, "m2": m2, "s2": s2,
            "m3": m3, "s3": s3}


def _conv_out(case):
    p = 2 * (case["k"] // 2) - case["k"]
    st = case.get("stride", 1)
    return (case["H"] + p) // st + 1, (case["W"] + p) // st + 1


def prepare(case, seed):
    d = _inputs(case, seed)
    k = case["kind"]
    st = {"case": case, "in": d}
    if k == "matmul":
        st["out"] = torch.empty((case["M"], case["N"]), dtype=F32, device="cuda")
    elif k in ("conv_nhwc", "conv_nchw"):
        ho, wo = _conv_out(case)
        b, f = case["B"], case["F"]
        st["out"] = torch.empty((b, ho, wo, f) if k == "conv_nhwc" else (b, f, ho, wo),
                                dtype=d["x"].dtype, device="cuda")
    elif k == "model":
        st["program"] = lower.lower_text(model_zoo.model(case["model"]))
    elif k in ("irb", "qbottleneck"):
        st["out"] = torch.empty_like(d["x"])
    else:
        e = lambda n: torch.empty((case["S"], n), dtype=BF16, device="cuda")
        st["bufs"] = {n: e(case["ffn"] if n == "act" else case["D"])
                      for n in ("Q", "K", "V", "A", "h", "act", "out")}
    return st


def run(state):
    case, d = state["case"], state["in"]
    k = case["kind"]
    if k == "matmul":
        return groups.fused_matmul_bias_act(d["A"], d["B"], d["bias"], state["out"], case["act"])
    if k == "conv_nhwc":
        if d["res"] is None:
            return groups.fused_conv2d_nhwc_bias_act(d["x"], d["w"], d["bias"], state["out"],
                                                     case["k"] // 2, case["act"])
        return groups.fused_conv2d_nhwc_bias_res_act(d["x"], d["w"], d["bias"], d["res"],
                                                     state["out"], case["k"] // 2, case["act"])
    if k == "conv_nchw":
        if d["res"] is None:
            return groups.fused_conv2d_nchw_bias_act(d["x"], d["w"], d["bias"], state["out"],
                                                     case["k"] // 2, case["act"],
                                                     stride=case["stride"])
        return groups.fused_conv2d_nchw_bias_res_act(d["x"], d["w"], d["bias"], d["res"],
                                                     state["out"], case["k"] // 2, case["act"],
                                                     stride=case["stride"])
    if k == "model":
        return list(state["program"].run(d).values())
    if k == "irb":
        return groups.fused_irb_f32(d["x"], d["we"], d["wdw"], d["wp"], state["out"])
    if k == "qbottleneck":
        return groups.fused_qbottleneck_i8(d["x"], d["w1"], d["w2"], d["w3"], d["m1"], d["s1"],
                                           d["m2"], d["s2"], d["m3"], d["s3"], state["out"])
    groups.llama_layer(d, state["bufs"], case["heads"])
    return state["bufs"]


# ---- bytes and operations -------------------------------------------------------
def work(case):
    k = case["kind"]
    if k == "matmul":
        m, kk, n = case["M"], case["K"], case["N"]
        return {"bytes": 4 * (m * kk + kk * n + m * n + (n if case["bias"] else 0)),
                "flops": 2 * m * n * kk}
    if k in ("conv_nhwc", "conv_nchw"):
        es = 2 if case.get("dtype") == "bf16" else 4
        b, h, w, c, f, kk = (case[n] for n in ("B", "H", "W", "C", "F", "k"))
        ho, wo = _conv_out(case)
        out = b * ho * wo * f
        return {"bytes": es * (b * h * w * c + f * c * kk * kk + out * (2 if case["res"] else 1)) +
                (4 * f if case["bias"] else 0), "flops": 2 * out * c * kk * kk}
    if k == "model":
        outs = {"resnet18": 1000, "dcgan_generator": 48, "autoencoder": 784, "autoencoder_deep": 1024}
        params = sum(math.prod(s) for s, _ in _model_params(case["model"]).values())
        return {"bytes": 4 * (params + outs[case["model"]]), "flops": _model_flops(case["model"])}
    p = case["B"] * case["H"] * case["W"] if "B" in case else 0
    if k == "irb":
        c, e = case["C"], case["E"]
        return {"bytes": 4 * (2 * p * c + 2 * c * e + 9 * e), "flops": 2 * p * (2 * c * e + 9 * e)}
    if k == "qbottleneck":
        c, m = case["C"], case["M1"]
        return {"bytes": 2 * p * c + 2 * c * m + 9 * m * m + 4 * (4 * m + 2 * c),
                "flops": 2 * p * (2 * c * m + 9 * m * m)}
    s, d, f, dh = case["S"], case["D"], case["ffn"], case["D"] // case["heads"]
    weights = 2 * (4 * d * d + 3 * d * f)
    # returned: Q, K, V, the attention's output, h, out [S, D] and act [S, ffn]
    return {"bytes": weights + 8 * d + 8 * s * (dh // 2) + 2 * s * (7 * d + f),
            "flops": 2 * s * (4 * d * d + 3 * d * f) + 4 * d * (s * (s + 1) // 2)}


def tolerance(case):
    k = case["kind"]
    if k == "qbottleneck":
        return "exact"
    # about four times the error against 64 bits that the groups show: bf16
    # 0.0016 (one rounding) to 0.0039 (a layer's five groups), f32 1e-7 to 4e-7
    # and more for the longest sums, a network's 21 layers 2.8e-6
    if k == "llama":
        return {"rel": 1e-2}
    if case.get("dtype") == "bf16":
        return {"rel": 7e-3}
    return {"rel": 1.2e-5 if k == "model" else 4e-6}


# ---- the same in 64 bits ----------------------------------------------------------
def _conv64(x, w, pad, st):
    """x [B,H,W,C], w [F,KH,KW,C] -> [B,Ho,Wo,F], f64, one tap at a time."""
    x, w = x.to(F64), w.to(F64)
    f, kh, kw, c = w.shape
    x = torch.nn.functional.pad(x, (0, 0, pad, pad, pad, pad))
    b, h, wd, _ = x.shape
    ho, wo = (h - kh) // st + 1, (wd - kw) // st + 1
    acc = torch.zeros((b * ho * wo, f), dtype=F64, device=x.device)
    for i in range(kh):
        for j in range(kw):
            tap = x[:, i:i + (ho - 1) * st + 1:st, j:j + (wo - 1) * st + 1:st, :]
            acc += tap.reshape(-1, c) @ w[:, i, j, :].t().contiguous()
    return acc.reshape(b, ho, wo, f)


def _conv64_nchw(x, w, pad, st):
    return _conv64(x.permute(0, 2, 3, 1), w.permute(0, 2, 3, 1), pad, st).permute(0, 3, 1, 2)


def _requant64(acc, m, s):
    m, s = m.to(torch.int64), s.to(torch.int64)
    return (acc.to(torch.int64) * m + (torch.ones_like(s) << (s - 1))) >> s


def _act64(v, act):
    if act == "none":
        return v
    return v.clamp(min=0) if act == "relu" else v.clamp(0, 6)


def _model64(name, d):
    d = {n: t.to(F64) for n, t in d.items()}
    x = d["input"]
    if name == "resnet18":
        inp = x
        for n, _, _, _, st, pad in _resnet18_layers():
            if n.endswith("_c1"):
                inp = x
                x = _conv64_nchw(x, d[n], pad, st).clamp(min=0)
            elif n.endswith("_c2"):
                sc = n[:-2] + "sc"
                r = _conv64_nchw(inp, d[sc], 0, 2) if sc in d else inp
                x = (_conv64_nchw(x, d[n], pad, st) + r).clamp(min=0)
            elif not n.endswith("_sc"):
                x = _conv64_nchw(x, d[n], pad, st)
                x = x if n == "w_fc" else x.clamp(min=0)
        return x.contiguous()
    if name == "dcgan_generator":
        for i, (_, relu) in enumerate(_DCGAN):
            x = _conv64_nchw(x, d[f"w{i}"], 1, 1)
            x = x.clamp(min=0) if relu else x
        return x.contiguous()
    ws = [n for n in d if n != "input"]
    for n in ws:
        x = x @ d[n]
        x = x if n == ws[-1] else x.clamp(min=0)
    return x


def _rope64(v, cos, sin, heads):
    s, d = v.shape
    p = v.reshape(s, heads, d // heads // 2, 2)
    c, sn = cos[:, None, :], sin[:, None, :]
    return torch.stack([p[..., 0] * c - p[..., 1] * sn, p[..., 0] * sn + p[..., 1] * c], -1).reshape(s, d)


def _llama64(case, d):
    d = {n: t.to(F64) for n, t in d.items()}
    s, heads = case["S"], case["heads"]
    dh = case["D"] // heads
    norm = lambda v, gain: v * torch.rsqrt((v * v).mean(1, keepdim=True) + 1e-5) * gain
    xn = norm(d["x"], d["g1"])
    q = _rope64(xn @ d["wq"], d["cos_t"], d["sin_t"], heads)
    k = _rope64(xn @ d["wk"], d["cos_t"], d["sin_t"], heads)
    v = xn @ d["wv"]
    mask = torch.ones((s, s), dtype=torch.bool, device=q.device).triu(1)
    a = torch.empty_like(q)
    for h in range(heads):
        c = slice(h * dh, (h + 1) * dh)
        sc = (q[:, c] @ k[:, c].t().contiguous()) * dh ** -0.5
        a[:, c] = torch.softmax(sc.masked_fill(mask, float("-inf")), 1) @ v[:, c].contiguous()
    hid = d["x"] + a @ d["wo"]
    hn = norm(hid, d["g2"])
    act = torch.nn.functional.silu(hn @ d["wg"]) * (hn @ d["wu"])
    return {"Q": q, "K": k, "V": v, "A": a, "h": hid, "act": act, "out": hid + act @ d["wd"]}


def exact(case, seed):
    d = _inputs(case, seed)
    k = case["kind"]
    if k == "matmul":
        v = d["A"].to(F64) @ d["B"].to(F64)
        return _act64(v if d["bias"] is None else v + d["bias"].to(F64), case["act"])
    if k in ("conv_nhwc", "conv_nchw"):
        if k == "conv_nhwc":
            v = _conv64(d["x"], d["w"], case["k"] // 2, 1)
        else:
            v = _conv64_nchw(d["x"], d["w"], case["k"] // 2, case["stride"])
        if d["bias"] is not None:
            b = d["bias"].to(F64)
            v = v + (b if k == "conv_nhwc" else b[:, None, None])
        if d["res"] is not None:
            v = v + d["res"].to(F64)
        return _act64(v, case["act"]).contiguous()
    if k == "model":
        return [_model64(case["model"], d)]
    if k == "irb":
        e, c = d["we"].shape
        ex = _conv64(d["x"], d["we"].reshape(e, 1, 1, c), 0, 1).clamp(0, 6)
        exp = torch.nn.functional.pad(ex, (0, 0, 1, 1, 1, 1))
        h, w, wdw = case["H"], case["W"], d["wdw"].to(F64)
        dw = sum(exp[:, i:i + h, j:j + w, :] * wdw[i, j] for i in range(3) for j in range(3)).clamp(0, 6)
        return _conv64(dw, d["wp"].reshape(c, 1, 1, e), 0, 1) + d["x"].to(F64)
    if k == "qbottleneck":
        m, c = d["w1"].shape
        y = _requant64(_conv64(d["x"], d["w1"].reshape(m, 1, 1, c), 0, 1), d["m1"], d["s1"]).clamp(0, 127)
        y = _requant64(_conv64(y, d["w2"], 1, 1), d["m2"], d["s2"]).clamp(0, 127)
        y = _requant64(_conv64(y, d["w3"].reshape(c, 1, 1, m), 0, 1), d["m3"], d["s3"]) + d["x"].to(torch.int64)
        return y.clamp(0, 127).to(torch.int8)
    return _llama64(case, d)
