"""Performance cases of the per-layer quantization path.

Each case is one thing a quantization run has the framework do, through the
entry points a driver calls: calibration hooks (``add_batch``, the saliency and
gradient caches), per-layer quantization (``fasterquant`` of GPTQ, GPTAQ and
G2PTQ), round-to-nearest with export, and the single-block operator.

``op`` of a case:

- ``block``     ``run_eager``: one prepared block of columns on the transposed layout
- ``calibrate`` one linear's output gradients to saliencies and weight gradients to
                their running mean (two batches)
- ``rtn``       round-to-nearest: ``find_params`` (min/max or clip search),
                ``fake_quantize``, compressed-tensors packing
- ``hessian``   a linear's calibration batches through ``add_batch``, then its Hessian read
- ``quantize``  GPTQ ``fasterquant`` from a finished Hessian
- ``layer``     GPTAQ or G2PTQ: calibration batches and ``fasterquant``
- ``experts``   a mixture-of-experts layer: routed calibration tokens of every expert,
                gate and up sharing a Hessian, and ``fasterquant`` of each shape's launch
"""
import math

import torch

from g2ptq_amd import (G2PTQ, GPTAQ, GPTQ, SharedInputHessian, WeightQuantizer,
                       make_group_quantizers, merge_group_quantizers)
from g2ptq_amd import g2ptq_utils, gptaq_utils, gptq_utils
from g2ptq_amd.calib_utils import GradientCache, SaliencyCache
from g2ptq_amd.compressed_tensors_utils import compress

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DAMP = 0.01
GPTAQ_ALPHA = 0.25
G2PTQ_ALPHA = 0.1


def listed():
    return [
        # the reference's block operator on a k/v projection's first block: latency
        {"name": "block_gptq", "op": "block", "method": "gptq", "layers": 1, "rows": 1024,
         "width": 128},
        # one linear's backward hooks over two calibration batches (G2PTQ's statistics)
        {"name": "calibrate", "op": "calibrate", "tokens": 8192, "rows": 4096, "cols": 4096,
         "groups": 4, "dtype": "bf16"},
        # round-to-nearest of an attention projection with the clip search, asymmetric
        {"name": "rtn_clip_asym", "op": "rtn", "rows": 4096, "cols": 4096, "group": 128,
         "bits": 4, "sym": False, "clip": True},
        # the Hessian of a hidden-size input, bf16 model
        {"name": "hessian_bf16", "op": "hessian", "method": "gptq", "cols": 4096, "tokens": 65536,
         "batch": 8192, "dtype": "bf16", "groups": 1},
        # the same input of an fp16 model
        {"name": "hessian_fp16", "op": "hessian", "method": "gptq", "cols": 4096, "tokens": 32768,
         "batch": 8192, "dtype": "fp16", "groups": 1},
        # an fp32 model with a ragged hidden size and a ragged last batch
        {"name": "hessian_fp32", "op": "hessian", "method": "gptq", "cols": 2752, "tokens": 14000,
         "batch": 4096, "dtype": "fp32", "groups": 1},
        # one attention projection, W4 groups of 128
        {"name": "gptq_proj", "op": "quantize", "layers": 1, "rows": 4096, "cols": 4096,
         "group": 128, "bits": 4, "sym": True, "clip": False, "order": "none"},
        # the block's widest input: down_proj
        {"name": "gptq_down", "op": "quantize", "layers": 1, "rows": 4096, "cols": 14336,
         "group": 128, "bits": 4, "sym": True, "clip": False, "order": "none"},
        # the clip search on every group as the scripts run it, k and v in one launch
        {"name": "gptq_clip", "op": "quantize", "layers": 2, "rows": 1024, "cols": 4096,
         "group": 128, "bits": 4, "sym": True, "clip": True, "order": "none"},
        # asymmetric calibration, two bits in groups of 64
        {"name": "gptaq_layer", "op": "layer", "method": "gptaq", "rows": 4096, "cols": 4096,
         "tokens": 16384, "batch": 4096, "group": 64, "bits": 2, "groups": 1},
        # saliency-weighted Hessians of four row groups and the trust region, three bits
        {"name": "g2ptq_layer", "op": "layer", "method": "g2ptq", "rows": 4096, "cols": 4096,
         "tokens": 16384, "batch": 4096, "group": 128, "bits": 3, "groups": 4},
        # a mixture-of-experts layer, top-8 routing with uneven expert popularity
        {"name": "experts", "op": "experts", "experts": 16, "hidden": 2048, "inter": 768,
         "tokens": 8192, "batch": 2048, "group": 128, "bits": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, m):
    """A multiple of m between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, _log(rng, lo, hi) // m * m))


def draw(rng):
    op = rng.choice(["block", "calibrate", "rtn", "hessian", "hessian", "quantize", "quantize",
                     "layer", "experts"])
    if op == "block":
        return {"op": op, "method": rng.choice(["gptq", "gptaq", "g2ptq"]),
                "layers": rng.choice([1, 1, 2, 4]), "rows": _log(rng, 256, 8192),
                "width": rng.choice([128, 128, 96, 100])}
    if op == "calibrate":
        groups = rng.choice([1, 2, 4])
        return {"op": op, "tokens": _log(rng, 1000, 16384), "rows": _mult(rng, 1024, 8192, 4),
                "cols": _log(rng, 1024, 8192), "groups": groups,
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if op == "rtn":
        clip = rng.random() < 0.6
        group = rng.choice([32, 64, 128])
        return {"op": op, "rows": _log(rng, 512, 6000), "cols": _mult(rng, 1024, 4096, 128),
                "group": group, "bits": rng.choice([2, 3, 4, 8]), "sym": rng.random() < 0.5,
                "clip": clip}
    if op == "hessian":
        method = rng.choice(["gptq", "gptq", "gptaq", "g2ptq"])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        return {"op": op, "method": method, "cols": _log(rng, 700, 5120),
                "tokens": _log(rng, 2000, 16384 if method == "g2ptq" or dtype != "bf16" else 40000),
                "batch": rng.choice([2048, 4096, 8192]), "dtype": dtype,
                "groups": rng.choice([2, 4]) if method == "g2ptq" else 1}
    if op == "quantize":
        group = rng.choice([64, 128, 128, 128, -1])
        cols = _log(rng, 700, 6000) if group == -1 else _mult(rng, 768, 8192, 128)
        return {"op": op, "layers": rng.choice([1, 1, 2, 3]), "rows": _log(rng, 512, 5000),
                "cols": cols, "group": group, "bits": rng.choice([3, 4, 4, 8]),
                "sym": rng.random() < 0.6, "clip": rng.random() < 0.5,
                "order": rng.choice(["none", "none", "act", "static_act"])}
    if op == "layer":
        method = rng.choice(["gptaq", "g2ptq"])
        groups = rng.choice([2, 4]) if method == "g2ptq" else 1
        return {"op": op, "method": method, "rows": _mult(rng, 512, 4096, 4),
                "cols": _mult(rng, 768, 4096, 128), "tokens": _log(rng, 3000, 16384),
                "batch": rng.choice([2048, 4096]), "group": rng.choice([64, 128]),
                "bits": rng.choice([2, 3, 4]), "groups": groups}
    return {"op": op, "experts": rng.choice([4, 6, 8, 12, 16]),
            "hidden": _mult(rng, 1024, 2048, 128), "inter": _mult(rng, 512, 1024, 128),
            "tokens": _log(rng, 2000, 8192), "batch": 2048, "group": rng.choice([64, 128]),
            "bits": rng.choice([3, 4])}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _channels(g, C):
    """LogNormal channel scales: activations have a few much larger channels."""
    return torch.exp(_randn(g, C))


def _tokens(g, n, C, sig, dtype):
    return (_randn(g, n, C) * sig).to(dtype)


def _weight(g, R, C):
    return (_randn(g, R, C) * 0.02).bfloat16()


def _linear(w):
    lin = torch.nn.Linear(1, 1, bias=False, device=DEV)
    lin.weight = torch.nn.Parameter(w.clone(), requires_grad=False)
    return lin


def _batches(n, batch):
    return [(t, min(n, t + batch)) for t in range(0, n, batch)]


def _saliency(g, n, G, rows):
    """σ_t²·χ²_{R/G}/(R/G), σ_t LogNormal(0, 0.5): the χ² mean as 1 + √(2/k)·N(0, 1)."""
    k = max(1, rows // G)
    sig = torch.exp(0.5 * _randn(g, n, 1))
    return sig ** 2 * (1 + math.sqrt(2 / k) * _randn(g, n, G)).clamp_min(0.05)


def _routing(g, case):
    """Per batch and expert: the positions of its routed tokens (top-8, Zipf popularity)."""
    E = case["experts"]
    logp = -1.1 * torch.log(torch.arange(1, E + 1, device=DEV, dtype=torch.float32))
    top_k = max(1, min(8, E // 2))
    out = []
    for t0, t1 in _batches(case["tokens"], case["batch"]):
        u = torch.rand(t1 - t0, E, device=DEV, generator=g).clamp_(1e-20, 1.0)
        top = torch.topk(logp - torch.log(-torch.log(u)), top_k, dim=1).indices
        order = torch.argsort(top.reshape(-1), stable=True)
        tok = torch.div(order, top_k, rounding_mode="floor") + t0
        out.append(tok.split(torch.bincount(top.reshape(-1), minlength=E).tolist()))
    return out


def _dense_hessian(g, C):
    """A finished GPTQ Hessian of 1.25·C LogNormal tokens (fp32)."""
    n = (5 * C // 4 + 63) // 64 * 64
    sig = _channels(g, C)
    H = torch.zeros(C, C, device=DEV)
    for t0, t1 in _batches(n, 8192):
        x = _tokens(g, t1 - t0, C, sig, torch.bfloat16).float()
        H += x.t().mm(x)
    H = (H + H.t()) * (1.0 / n)
    return H.contiguous()


def _quantizers(case, columns):
    q = WeightQuantizer()
    q.configure(case["bits"], perchannel=True, sym=case.get("sym", True),
                mse=case.get("clip", False))
    return make_group_quantizers(q, columns, case["group"])


def prepare(case, seed):
    g = _generator(seed)
    op = case["op"]
    if op == "block":
        B, R, n = case["layers"], case["rows"], case["width"]
        # a factor's diagonal block: positive diagonal, smaller entries to its right
        U = torch.triu(_randn(g, B, n, n) * 0.1, 1)
        U += torch.diag_embed(torch.exp(0.3 * _randn(g, B, n)))
        w = _randn(g, B, n, R) * 0.02
        scale = (w.abs().amax(1, keepdim=True) / 7.5).expand(B, n, R).contiguous()
        st = {"weight": w, "hinv": U, "scale": scale, "zero": torch.zeros_like(scale),
              "int_weight": torch.empty_like(w), "error": torch.empty_like(w)}
        if case["method"] == "gptaq":
            st["p"] = torch.triu(_randn(g, B, n, n) * 0.01, 1)
            st["column_weight"] = torch.empty(B, R, device=DEV)
        elif case["method"] == "g2ptq":
            st["z"] = _randn(g, B, n, R) * 1e-5
            st["ghinv"] = _randn(g, B, n, R) * 1e-4
        return {"case": case, "t": st}
    if op == "calibrate":
        dt = DTYPES[case["dtype"]]
        R, C, n = case["rows"], case["cols"], case["tokens"]
        scale = torch.exp(_randn(g, R))
        return {"case": case, "out": [(_randn(g, n, R) * scale).to(dt) for _ in range(2)],
                "wgrad": [(_randn(g, R, C) * 1e-2).to(dt) for _ in range(2)],
                "inp": torch.empty(n, C, device=DEV, dtype=dt)}
    if op == "rtn":
        q = WeightQuantizer()
        q.configure(case["bits"], perchannel=True, sym=case["sym"], mse=case["clip"],
                    weight_groupsize=case["group"])
        w = _weight(g, case["rows"], case["cols"])
        return {"case": case, "q": q, "w": w, "lin": _linear(w)}
    if op == "hessian" or op == "layer":
        C, n = case["cols"], case["tokens"]
        dt = DTYPES[case.get("dtype", "bf16")]
        sig = _channels(g, C)
        cuts = _batches(n, case["batch"])
        rows = case.get("rows", 8 * case["groups"])
        st = {"case": case, "x": [_tokens(g, b - a, C, sig, dt) for a, b in cuts],
              "w": _weight(g, rows, C)}
        st["lin"] = _linear(st["w"])
        if case["method"] == "gptaq":
            st["fp"] = [(x.float() + 0.05 * sig * _randn(g, *x.shape)).to(dt) for x in st["x"]]
        elif case["method"] == "g2ptq":
            st["sal"] = [_saliency(g, b - a, case["groups"], case.get("rows", C))
                         for a, b in cuts]
            # rows with heavy-tailed magnitudes
            tau = (_randn(g, rows).abs() / _randn(g, rows).abs().clamp_min(0.2)).unsqueeze(1)
            st["grad"] = _randn(g, rows, C) * 1e-3 * tau
        return st
    if op == "quantize":
        B = case["layers"]
        w = [_weight(g, case["rows"], case["cols"]) for _ in range(B)]
        H = _dense_hessian(g, case["cols"])
        # the layers of one launch have their own inputs: scaled channels of one Hessian
        s = [torch.exp(0.1 * b * _randn(g, case["cols"])) for b in range(B)]
        H = torch.stack([H * s[b].unsqueeze(0) * s[b].unsqueeze(1) for b in range(B)])
        return {"case": case, "w": w, "lin": [_linear(x) for x in w], "H": H}
    if op == "experts":
        E, h, i, n = case["experts"], case["hidden"], case["inter"], case["tokens"]
        X = _tokens(g, n, h, _channels(g, h), torch.bfloat16)
        sig = _channels(g, i)
        routed = []
        for batch in _routing(g, case):
            routed.append([(X[t], _tokens(g, t.shape[0], i, sig, torch.bfloat16)) for t in batch])
        w = {"gu": [_weight(g, i, h) for _ in range(2 * E)],
             "down": [_weight(g, h, i) for _ in range(E)]}
        return {"case": case, "routed": routed, "w": w,
                "lin": {k: [_linear(x) for x in v] for k, v in w.items()}}
    raise ValueError(op)


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _restore(lins, weights):
    """The weights as they were before an earlier pass quantized them."""
    for lin, w in zip(lins, weights):
        lin.weight.data.copy_(w)


def _params(quantizers, rows, group):
    m = merge_group_quantizers(quantizers, 0, rows, group)
    return [m.scale, m.zero]


def _order(case):
    order = case.get("order", "none")
    return {"actorder": order != "none", "static_groups": order == "static_act"}


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "block":
        t = dict(state["t"])
        t["weight"] = t["weight"].clone()  # the operator writes its results over its inputs
        if "ghinv" in t:
            t["ghinv"] = t["ghinv"].clone()
        mod = {"gptq": gptq_utils, "gptaq": gptaq_utils, "g2ptq": g2ptq_utils}[case["method"]]
        return list(mod.run_eager(maxq=7, backend="hip", **t))
    if op == "calibrate":
        sal = SaliencyCache(["linear"], case["groups"])
        grad = GradientCache(["linear"], case["groups"])
        sal.hooks_enabled = grad.hooks_enabled = True
        for go, gw in zip(state["out"], state["wgrad"]):
            grad.forward_hook(None, (state["inp"],), None, "linear")
            sal.grad_hook(go, "linear", "block")
            grad.cache_gradient(gw, "linear", "block")
        return [sal.saliency_cache["linear"]["block"], grad.gradients_cache["linear"]["block"]]
    if op == "rtn":
        q, w = state["q"], state["w"]
        q.find_params(w)
        fq, codes, scale = q.fake_quantize(w)
        g = case["group"]
        full = scale.repeat_interleave(g, dim=1)
        compress(state["lin"], full, codes, case["bits"], g)
        packed = state["lin"]._export_qparams["weight_packed"]
        return [q.scale, q.zero, fq, packed]
    if op == "hessian":
        lin, method = state["lin"], case["method"]
        if method == "gptq":
            m = GPTQ([lin])
        elif method == "gptaq":
            m = GPTAQ([lin])
            m.fp_inp[0] = list(state["fp"])
        else:
            m = G2PTQ([lin], [state["sal"]], [state["grad"]], case["groups"])
        for x in state["x"]:
            m.add_batch(0, x.unsqueeze(0), None)
        return [m.H, m.dXXT] if method == "gptaq" else [m.H]
    if op == "quantize":
        _restore(state["lin"], state["w"])
        m = GPTQ(state["lin"])
        m.H = state["H"]
        m.quantizer = _quantizers(case, case["cols"])
        m.fasterquant(blocksize=128, percdamp=DAMP, groupsize=case["group"], backend="hip",
                      **_order(case))
        return ([lin.weight.data for lin in state["lin"]]
                + _params(m.quantizer, case["layers"] * case["rows"], case["group"]))
    if op == "layer":
        lin = state["lin"]
        _restore([lin], [state["w"]])
        kw = {"blocksize": 128, "percdamp": DAMP, "groupsize": case["group"], "backend": "hip"}
        if case["method"] == "gptaq":
            m = GPTAQ([lin])
            m.fp_inp[0] = list(state["fp"])
            kw["alpha"] = GPTAQ_ALPHA
        else:
            m = G2PTQ([lin], [state["sal"]], [state["grad"]], case["groups"])
            kw["alpha"] = G2PTQ_ALPHA
        m.quantizer = _quantizers(case, case["cols"])
        for x in state["x"]:
            m.add_batch(0, x.unsqueeze(0), None)
        m.fasterquant(**kw)
        return [lin.weight.data] + _params(m.quantizer, case["rows"], case["group"])
    if op == "experts":
        E, lins = case["experts"], state["lin"]
        for k in ("gu", "down"):
            _restore(lins[k], state["w"][k])
        gu, down = GPTQ(lins["gu"]), GPTQ(lins["down"])
        gu.quantizer = _quantizers(case, case["hidden"])
        down.quantizer = _quantizers(case, case["inter"])
        shares = [SharedInputHessian([(gu, 2 * e), (gu, 2 * e + 1)]) for e in range(E)]
        for batch in state["routed"]:
            for e, (xg, xd) in enumerate(batch):
                if xg.shape[0]:
                    shares[e].add_batch(xg)
                    down.add_batch(e, xd, None)
        for s in shares:
            s.finalize()
        kw = {"blocksize": 128, "percdamp": DAMP, "groupsize": case["group"], "backend": "hip"}
        gu.fasterquant(**kw)
        down.fasterquant(**kw)
        return ([lin.weight.data for k in ("gu", "down") for lin in lins[k]]
                + _params(gu.quantizer, 2 * E * case["inter"], case["group"])[:1]
                + _params(down.quantizer, E * case["hidden"], case["group"])[:1])
    raise ValueError(op)


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------

def _quantize_work(layers, rows, cols, factors, extra=1):
    """Factor (2C³/3 each) and compensation (R·C² per product) of one launch."""
    flops = factors * 2 * cols ** 3 / 3 + extra * layers * rows * cols ** 2
    return flops, layers * rows * cols * 4 + factors * cols * cols * 4


def work(case):
    op = case["op"]
    if op == "block":
        B, R, n = case["layers"], case["rows"], case["width"]
        return {"bytes": 4 * B * (R * n * 6 + n * n), "flops": B * R * n * n}
    if op == "calibrate":
        b = {"bf16": 2, "fp16": 2, "fp32": 4}[case["dtype"]]
        n = 2 * case["tokens"] * case["rows"] * b + 2 * case["rows"] * case["cols"] * b
        return {"bytes": n + 2 * case["tokens"] * case["groups"] * 4
                + case["rows"] * case["cols"] * 4,
                "flops": 2 * 2 * case["tokens"] * case["rows"]}
    if op == "rtn":
        n = case["rows"] * case["cols"]
        # the symmetric search has at most 2·25 distinct scales, the other 625 ranges
        tries = (50 if case["sym"] else 625) if case["clip"] else 1
        return {"bytes": n * 4 + n * case["bits"] / 8 + n / case["group"] * 8,
                "flops": n * tries * 10}
    if op == "hessian" or op == "layer":
        C, n = case["cols"], case["tokens"]
        b = {"bf16": 2, "fp16": 2, "fp32": 4}[case.get("dtype", "bf16")]
        streams = 2 if case["method"] == "gptaq" else 1
        mats = 2 if case["method"] == "gptaq" else case["groups"]
        # symmetric products are half a product; the cross term is a whole one
        flops = n * C * C * (3 if case["method"] == "gptaq" else case["groups"])
        out = {"bytes": n * C * b * streams + mats * C * C * 4, "flops": flops}
        if op == "layer":
            G, R = case["groups"], case["rows"]
            extra = 2 if case["method"] == "gptaq" else 4
            f, by = _quantize_work(1, R, C, G, extra)
            if case["method"] == "gptaq":
                f += 2 * C ** 3 / 3 + C ** 3  # P
            out["flops"] += f
            out["bytes"] += by
        return out
    if op == "quantize":
        f, b = _quantize_work(case["layers"], case["rows"], case["cols"], case["layers"])
        return {"bytes": b, "flops": f}
    E, h, i = case["experts"], case["hidden"], case["inter"]
    k = max(1, min(8, E // 2))
    f1, b1 = _quantize_work(2 * E, i, h, E)
    f2, b2 = _quantize_work(E, h, i, E)
    n = case["tokens"] * k
    return {"bytes": b1 + b2 + n * (h + i) * 2, "flops": f1 + f2 + n * (h * h + i * i)}


def tolerance(case):
    op = case["op"]
    if op == "block":
        # every element receives the reference's rounded operations in its order
        return "exact"
    if op == "calibrate":
        return {"rel": 1e-6, "max": 1e-5}
    if op == "rtn":
        # a near-tie between two clip candidates may go either way, and changes a group
        return {"rel": 0.01, "max": 0.6, "differ": 0.005}
    if op == "hessian":
        # fp32 sums; the weighted and cross terms carry 16 significant bits of one operand
        return {"rel": 3e-6, "max": 1e-4} if case["method"] == "gptq" else \
            {"rel": 2e-5, "max": 5e-4}
    # a code at a rounding tie goes either way with the order of the fp32 sums, and the rest
    # of its row with it
    return {"rel": 0.03, "max": 0.99}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
# The quantization grid is defined in fp32 (a symmetric group's largest value sits on a tie
# of its grid), so scales and codes are formed in fp32 from values rounded to fp32; products,
# factors, errors and sums are 64-bit.

def _grid(xmin, xmax, bits, sym):
    half = 2 ** (bits - 1)
    # divisors as tensors: torch multiplies by the reciprocal of a number
    if sym:
        s = torch.maximum(xmin.abs(), xmax) / torch.full_like(xmin, (2 * half - 1) / 2)
        return s, torch.zeros_like(s)
    s = (xmax - xmin) / torch.full_like(xmin, 2 * half - 1)
    return s, torch.clamp(torch.round(-half - xmin / s), -half, half - 1)


def _codes(x, s, z, bits):
    half = 2 ** (bits - 1)
    return torch.clamp(torch.round(x / s) + z, -half, half - 1)


def _fit(x, bits, sym, clip):
    """Scale and zero (rows, 1) of fp32 groups (rows, width)."""
    xmin = x.amin(1, keepdim=True).clamp_max(0)
    xmax = x.amax(1, keepdim=True).clamp_min(0)
    s, z = _grid(xmin, xmax, bits, sym)
    if not clip:
        return s, torch.round(z)
    best = torch.full_like(s, math.inf, dtype=torch.float64)
    for i in range(25):
        for j in range(25):
            s1, z1 = _grid((1 - i / 50) * xmin, (1 - j / 50) * xmax, bits, sym)
            d = s1 * (_codes(x, s1, z1, bits) - z1) - x
            err = d.double().abs_().pow_(2.4).sum(1, keepdim=True)
            better = err < best
            s, z = torch.where(better, s1, s), torch.where(better, z1, z)
            best = torch.where(better, err, best)
    return s, torch.round(z)


def _factor64(H):
    C = H.shape[-1]
    A = H.double()
    A = A + torch.eye(C, device=DEV, dtype=torch.float64) * (DAMP * A.diagonal().mean())
    Ai = torch.cholesky_inverse(torch.linalg.cholesky(A))
    return torch.linalg.cholesky((Ai + Ai.t()) / 2).t().contiguous()


def _sweep64(W, U, case, P=None, Z=None, GH=None, static=None, perm=None):
    """The lazy-batch loop on W (rows, C): the dequantized weights and the parameters."""
    R, C = W.shape
    bits, sym, clip = case["bits"], case.get("sym", True), case.get("clip", False)
    gs = C if case["group"] == -1 else case["group"]
    W = W.double().clone()
    Q = torch.empty_like(W)
    S = torch.empty(R, -(-C // gs), device=DEV)
    Zr = torch.empty_like(S)
    if static is not None:
        S, Zr = static
    for i1 in range(0, C, 128):
        i2 = min(i1 + 128, C)
        E = torch.empty(R, i2 - i1, device=DEV, dtype=torch.float64)
        w = W[:, i1:i2].clone()
        gh = GH[:, i1:i2].clone() if GH is not None else None
        for c in range(i1, i2):
            k = c - i1
            gi = (perm[c] if perm is not None else c) // gs
            if static is None and c % gs == 0:
                S[:, gi:gi + 1], Zr[:, gi:gi + 1] = _fit(W[:, c:c + gs].float(), bits, sym, clip)
            x = w[:, k].clone()
            s, z = S[:, gi], Zr[:, gi]
            q = (s * (_codes(x.float(), s, z, bits) - z)).double()
            e = x - q
            if gh is not None:
                e = e - gh[:, k]
            e = e / U[c, c]
            Q[:, c], E[:, k] = q, e
            if k + 1 < i2 - i1:
                u = U[c, c + 1:i2]
                if gh is not None:
                    w[:, k + 1:] -= gh[:, k + 1:]
                    gh[:, k + 1:] -= torch.outer(Z[:, c], u)
                w[:, k + 1:] -= torch.outer(e, u)
                if P is not None:
                    w[:, k + 1:] += torch.outer(x, P[c, c + 1:i2])
        if i2 == C:
            break
        if GH is not None:
            d = torch.arange(127, 127 - (i2 - i1), -1, device=DEV, dtype=torch.float64)
            W[:, i2:] -= 128 * GH[:, i2:] - (Z[:, i1:i2] * d).mm(U[i1:i2, i2:])
            GH[:, i2:] -= Z[:, i1:i2].mm(U[i1:i2, i2:])
        W[:, i2:] -= E.mm(U[i1:i2, i2:])
        if P is not None:
            W[:, i2:] += Q[:, i1:i2].mm(P[i1:i2, i2:])
    return Q, S, Zr


def _hessians64(st):
    """The Hessians (and cross term) of a hessian or layer state."""
    case = st["case"]
    C = case["cols"]
    H = torch.zeros(case["groups"], C, C, device=DEV, dtype=torch.float64)
    D = torch.zeros(C, C, device=DEV, dtype=torch.float64)
    k = len(st["x"])
    for b, x in enumerate(st["x"]):
        x64 = x.double()
        if case["method"] == "g2ptq":
            for g in range(case["groups"]):
                s = st["sal"][b][:, g:g + 1].double()
                H[g] += (x64 * s).t().mm(x64) / (x.shape[0] * k)
        else:
            H[0] += x64.t().mm(x64) * (2 / k)
        if case["method"] == "gptaq":
            D += (st["fp"][b].double() - x64).t().mm(x64) * (2 / k)
    return H, D


def _trust64(W, Q0, G, U):
    Ai = U.t().mm(U)
    GA = G.mm(Ai)
    d = Ai.diagonal()
    e = Q0 - W
    loss = ((e * GA + e * e / 2) / d).abs()
    room = (G * GA).sum(1, keepdim=True) - GA * GA / d
    tl = 2 * G2PTQ_ALPHA * loss
    room = torch.maximum(room, tl).clamp_min(torch.finfo(torch.float32).tiny)
    beta = (1 - torch.sqrt((1 - tl / room).clamp_min(0))).mean(1, keepdim=True)
    return beta * G.mm(U.t()), beta * GA


def exact(case, seed):
    op = case["op"]
    if op == "quantize" and case["cols"] > 8192:
        return None
    st = prepare(case, seed)
    if op == "block":
        t = st["t"]
        w, U = t["weight"].double(), t["hinv"].double()
        q, codes, err = torch.empty_like(w), torch.empty_like(w), torch.empty_like(w)
        gh = t["ghinv"].double() if "ghinv" in t else None
        for k in range(case["width"]):
            x = w[:, k].clone()
            s, z = t["scale"][:, k], t["zero"][:, k]
            c = _codes(x.float(), s, z, 4)
            q[:, k], codes[:, k] = (s * (c - z)).double(), c.double()
            e = x - q[:, k] - (gh[:, k] if gh is not None else 0)
            err[:, k] = e / U[:, k, k].unsqueeze(1)
            u = U[:, k, k + 1:].unsqueeze(2)
            if gh is not None:
                w[:, k + 1:] -= gh[:, k + 1:]
                gh[:, k + 1:] -= u * t["z"][:, k].double().unsqueeze(1)
            w[:, k + 1:] -= u * err[:, k].unsqueeze(1)
            if "p" in t:
                w[:, k + 1:] += t["p"][:, k, k + 1:].double().unsqueeze(2) * x.unsqueeze(1)
        return [q, codes, err]
    if op == "calibrate":
        G = case["groups"]
        sal = [x.double().pow(2).view(x.shape[0], G, -1).mean(-1) for x in st["out"]]
        g = (st["wgrad"][0].double() + st["wgrad"][1].double()) / (2 * case["tokens"])
        return [sal, g]
    if op == "rtn":
        R, C, gs = case["rows"], case["cols"], case["group"]
        x = st["w"].float().view(-1, gs)
        s, z = _fit(x, case["bits"], case["sym"], case["clip"])
        fq = s.double() * (_codes(x, s, z, case["bits"]) - z)
        return [s.view(R, -1), z.view(R, -1), fq.view(R, C), None]
    if op == "hessian":
        H, D = _hessians64(st)
        return [H, D.unsqueeze(0)] if case["method"] == "gptaq" else \
            [H.unsqueeze(0) if case["method"] == "g2ptq" else H]
    if op == "quantize":
        B, R, C = case["layers"], case["rows"], case["cols"]
        W = torch.stack(st["w"]).float()
        gs = C if case["group"] == -1 else case["group"]
        actorder, static_groups = _order(case)["actorder"], _order(case)["static_groups"]
        static = perm = None
        if static_groups or case["group"] == -1:
            s, z = _fit(W.reshape(-1, gs), case["bits"], case["sym"], case["clip"])
            static = (s.view(B * R, -1), z.view(B * R, -1))
        H = st["H"]
        if actorder:
            key = H.diagonal(dim1=1, dim2=2).sum(0) / B
            p = torch.argsort(key, descending=True, stable=True)
            W, H = W[:, :, p], H[:, p][:, :, p]
            if static_groups:
                perm = p.tolist()
        outs, S, Z = [], [], []
        for b in range(B):
            rows = slice(b * R, (b + 1) * R)
            part = None if static is None else (static[0][rows], static[1][rows])
            Q, s, z = _sweep64(W[b], _factor64(H[b]), case, static=part, perm=perm)
            if actorder:
                Q = Q[:, torch.argsort(p)]
            outs.append(Q)
            S.append(s)
            Z.append(z)
        return outs + [torch.cat(S), torch.cat(Z)]
    if op == "layer":
        H, D = _hessians64(st)
        W = st["w"].float()
        if case["method"] == "gptaq":
            U = _factor64(H[0])
            P = GPTAQ_ALPHA * torch.triu(D.mm(U.t()), 1).mm(U)
            Q, s, z = _sweep64(W, U, case, P=P)
            return [Q, s, z]
        G, R, gs = case["groups"], case["rows"], case["group"]
        s0, z0 = _fit(W.view(-1, gs), case["bits"], True, False)
        Q0 = (s0 * (_codes(W.view(-1, gs), s0, z0, case["bits"]) - z0)).view(W.shape).double()
        parts = []
        for b in range(G):
            rows = slice(b * R // G, (b + 1) * R // G)
            U = _factor64(H[b])
            Z, GH = _trust64(W[rows].double(), Q0[rows], st["grad"][rows].double(), U)
            parts.append(_sweep64(W[rows], U, case, Z=Z, GH=GH))
        return [torch.cat([p[i] for p in parts]) for i in range(3)]
    if op == "experts":
        E = case["experts"]
        outs, scales = {"gu": [], "down": []}, {"gu": [], "down": []}
        for e in range(E):
            for key, which, members in (("gu", 0, (2 * e, 2 * e + 1)), ("down", 1, (e,))):
                xs = [b[e][which].double() for b in st["routed"] if b[e][which].shape[0]]
                H = sum(x.t().mm(x) for x in xs) * (2 / len(xs))
                U = _factor64(H)
                for m in members:
                    Q, s, _ = _sweep64(st["w"][key][m].float(), U, case)
                    outs[key].append(Q)
                    scales[key].append(s)
        return outs["gu"] + outs["down"] + [torch.cat(scales["gu"]), torch.cat(scales["down"])]
    raise ValueError(op)
