"""The measured work of this framework: FP4 / INT4 quantized linear layers of a
dense transformer, the routed-expert MLP, and the weight (de)quantizers, each
through the public entry points of `mmfp4` and over the range of sizes that
serving and model conversion have.

A case is a dict of plain values; its "path" says what runs:

  gemm      one quantized linear layer, `marlin_gemm_fp4` / `marlin_gemm_int4`
  layer     the projections of one decoder layer: fp4 takes the fused entry
            points (q/k/v in one call, gate and up in one call with SiLU), int4
            the plain GEMM four times over the concatenated matrices
  mlp       gate_up + SiLU and the down projection on row-packed MMFP4 weights
            (`mmfp4_fused_gate_up`, `MMFP4Linear`)
  moe       softmax + top-k of the gate's logits, then the routed-expert SwiGLU
            MLP, with a shared expert when `shared`
  dequant   bulk dequantization of one matrix to fp16
  quantize  quantization of one fp16 matrix

Weights are N(0, 0.02) quantized in groups along K, activations N(0, 1) in
fp16, router logits N(0, 1) with a per-expert bias (uneven expert loads).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parent.parent / "metal-marlin_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mmfp4  # noqa: E402

E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0,
        -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def listed():
    # One decoder layer of the benchmark's dense model (hidden 4096, 1024 k/v
    # columns, intermediate 14336) and its expert model (hidden 2048,
    # intermediate 768, 128 experts, top-8).
    dense = {"hidden": 4096, "kv": 1024, "inter": 14336, "group": 128}
    moe = {"path": "moe", "experts": 128, "topk": 8, "hidden": 2048, "inter": 768, "group": 128,
           "shared": 0}
    return [
        # the smallest call: one projection for one token, where launch latency counts
        {"name": "gemm_m1", "path": "gemm", "fmt": "fp4", "m": 1, "n": 4096, "k": 4096,
         "group": 128},
        # single-stream decode: one token through a layer
        {"name": "layer_fp4_m1", "path": "layer", "fmt": "fp4", "m": 1, **dense},
        # batched decode, 32 sequences
        {"name": "layer_fp4_m32", "path": "layer", "fmt": "fp4", "m": 32, **dense},
        # a short or mixed batch: an odd number of rows between decode and prefill
        {"name": "layer_fp4_m100", "path": "layer", "fmt": "fp4", "m": 100, **dense},
        # prefill of a prompt
        {"name": "layer_fp4_m2048", "path": "layer", "fmt": "fp4", "m": 2048, **dense},
        # batched decode on asymmetric INT4 weights
        {"name": "layer_int4_m16", "path": "layer", "fmt": "int4", "m": 16, **dense},
        # decode through an MLP held in the row-packed (MMFP4) checkpoint layout
        {"name": "mlp_m1", "path": "mlp", "m": 1, "hidden": 4096, "inter": 14336, "group": 128},
        # the largest: long-prompt prefill on the same layout
        {"name": "mlp_m8192", "path": "mlp", "m": 8192, "hidden": 4096, "inter": 14336,
         "group": 128},
        # expert model, batched decode and prefill
        {"name": "moe_t32", "tokens": 32, **moe},
        {"name": "moe_t1024", "tokens": 1024, **moe},
        # a checkpoint matrix expanded to fp16
        {"name": "dequant_fp4", "path": "dequant", "fmt": "fp4", "n": 14336, "k": 4096,
         "group": 128},
        # a matrix quantized when a model is converted
        {"name": "quantize_fp4", "path": "quantize", "fmt": "fp4", "n": 14336, "k": 4096,
         "group": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("gemm", "gemm", "layer", "layer", "mlp", "moe", "moe", "dequant",
                       "quantize"))
    group = rng.choice((32, 64, 128, 128, 128))
    fmt = rng.choice(("fp4", "fp4", "int4"))
    if path == "gemm":
        k = 128 * _log(rng, 4, 112)
        # widths: multiples of 8, or (a vocabulary, say) any number at all
        n = 8 * _log(rng, 64, 3584) + rng.choice((0, 0, 0, 4, 1))
        m = min(_log(rng, 1, 8192), 1_400_000_000_000 // (n * k))   # at most the largest's work
        return {"path": path, "fmt": fmt, "m": m, "n": n, "k": k, "group": group}
    if path == "layer":
        hidden = rng.choice((2048, 3072, 4096))
        return {"path": path, "fmt": fmt, "m": _log(rng, 1, 4096), "hidden": hidden,
                "kv": rng.choice((512, 1024, hidden)), "inter": 128 * rng.randint(32, 112),
                "group": group}
    if path == "mlp":
        return {"path": path, "m": _log(rng, 1, 8192), "hidden": rng.choice((2048, 3072, 4096)),
                "inter": 128 * rng.randint(32, 112), "group": rng.choice((64, 128))}
    if path == "moe":
        return {"path": path, "tokens": _log(rng, 1, 4096), "experts": rng.choice((16, 64, 128)),
                "topk": rng.choice((2, 4, 8)), "hidden": 128 * rng.randint(8, 24),
                "inter": 128 * rng.randint(4, 10), "group": rng.choice((64, 128)),
                "shared": rng.choice((0, 0, 1))}
    k = 128 * _log(rng, 4, 112)
    return {"path": path, "fmt": fmt, "k": k, "group": group,
            "n": 4 * _log(rng, 64, min(4096, 14_000_000 // k)) + rng.choice((0, 0, 1))}


# ------------------------------------------------------------------- inputs
class _Inputs:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(self.dev).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float16):
        return (torch.randn(shape, generator=self.gen, device=self.dev) * std).to(dtype)


def _pack(codes, rowpacked=False):
    """codes [..., N, K] in 0..15 -> int32 words [..., K/8, N] ([..., N, K/8] row-packed)."""
    c = codes.unflatten(-1, (-1, 8)).to(torch.int32)
    word = c[..., 0]
    for i in range(1, 8):
        word = word | (c[..., i] << (4 * i))
    return (word if rowpacked else word.transpose(-1, -2)).contiguous()


def _fp4(w, group, rowpacked=False):
    """W [..., N, K] -> (words, fp16 scales [..., K/g, N]): absmax / 6 per group, nearest E2M1."""
    x = w.float().unflatten(-1, (-1, group))
    amax = x.abs().amax(-1).clamp_min(1e-7)
    v = (x / amax.unsqueeze(-1) * 6.0).flatten(-2)
    mids = torch.tensor((0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0), device=w.device)
    codes = torch.bucketize(v.abs(), mids, out_int32=True) + 8 * (v < 0)
    return _pack(codes, rowpacked), (amax / 6.0).to(torch.float16).transpose(-1, -2).contiguous()


def _int4(w, group):
    """W [N, K] -> (words [K/8, N], fp16 scales [K/g, N], fp16 zero points [K/g, N])."""
    x = w.float().unflatten(-1, (-1, group))
    lo, hi = x.amin(-1), x.amax(-1)
    s = ((hi - lo) / 15.0).clamp_min(1e-7)
    z = torch.round(-lo / s)
    q = torch.round(x / s.unsqueeze(-1) + z.unsqueeze(-1)).clamp(0, 15).flatten(-2)
    half = lambda t: t.to(torch.float16).t().contiguous()  # noqa: E731
    return _pack(q.to(torch.int32)), half(s), half(z)


def _weight(inp, fmt, n, k, group, rowpacked=False):
    w = inp.normal(n, k, std=0.02, dtype=torch.float32)
    return _int4(w, group) if fmt == "int4" else _fp4(w, group, rowpacked)


def _experts(inp, e, n, k, group):
    parts = [_fp4(inp.normal(min(16, e - i), n, k, std=0.02, dtype=torch.float32), group)
             for i in range(0, e, 16)]
    return torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])


def _inputs(c, seed):
    """The case's tensors, made from the seed alone with plain torch."""
    inp, path = _Inputs(seed), c["path"]
    if path == "gemm":
        return {"w": _weight(inp, c["fmt"], c["n"], c["k"], c["group"]),
                "x": inp.normal(c["m"], c["k"])}
    if path == "layer":
        h, kv, i, g, m = c["hidden"], c["kv"], c["inter"], c["group"], c["m"]
        W = lambda n, k: _weight(inp, c["fmt"], n, k, g)  # noqa: E731
        if c["fmt"] == "fp4":
            w = {"q": W(h, h), "k": W(kv, h), "v": W(kv, h), "o": W(h, h), "gate": W(i, h),
                 "up": W(i, h), "down": W(h, i)}
            x = {n: inp.normal(m, h) for n in ("qkv", "o", "gate_up")}
        else:
            w = {"qkv": W(h + 2 * kv, h), "o": W(h, h), "gate_up": W(2 * i, h), "down": W(h, i)}
            x = {n: inp.normal(m, i if n == "down" else h)
                 for n in ("qkv", "o", "gate_up", "down")}
        return {"w": w, "x": x}
    if path == "mlp":
        h, i, g = c["hidden"], c["inter"], c["group"]
        return {"gate": _weight(inp, "fp4", i, h, g, True),
                "up": _weight(inp, "fp4", i, h, g, True),
                "down": _weight(inp, "fp4", h, i, g, True), "x": inp.normal(c["m"], h)}
    if path == "moe":
        h, i, g, e = c["hidden"], c["inter"], c["group"], c["experts"]
        s = {"gate_up": _experts(inp, e, 2 * i, h, g), "down": _experts(inp, e, h, i, g)}
        if c["shared"]:
            s["shared_gate_up"] = _weight(inp, "fp4", 2 * i, h, g)
            s["shared_down"] = _weight(inp, "fp4", h, i, g)
        s["x"] = inp.normal(c["tokens"], h)
        logits = inp.normal(c["tokens"], e, dtype=torch.float32) + \
            inp.normal(1, e, std=0.5, dtype=torch.float32)
        s["logits"] = logits.to(torch.float16)
        return s
    if path == "dequant":
        return {"w": _weight(inp, c["fmt"], c["n"], c["k"], c["group"])}
    return {"w": inp.normal(c["n"], c["k"], std=0.02)}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["path"] == "mlp":
        s["down"] = mmfp4.MMFP4Linear(*s["down"], group_size=case["group"])
    return s


# ---------------------------------------------------------------------- run
def run(s):
    c = s["case"]
    path, g = c["path"], c.get("group")
    if path == "gemm":
        gemm = mmfp4.marlin_gemm_int4 if c["fmt"] == "int4" else mmfp4.marlin_gemm_fp4
        return gemm(s["x"], *s["w"], group_size=g)
    if path == "layer":
        w, x = s["w"], s["x"]
        if c["fmt"] == "int4":
            return [mmfp4.marlin_gemm_int4(x[n], *w[n], group_size=g)
                    for n in ("qkv", "o", "gate_up", "down")]
        q, k, v = mmfp4.mmfp4_fused_qkv(x["qkv"], *w["q"], *w["k"], *w["v"], group_size=g)
        o = mmfp4.marlin_gemm_fp4(x["o"], *w["o"], group_size=g)
        act = mmfp4.mmfp4_fused_gate_up_marlin(x["gate_up"], *w["gate"], *w["up"], group_size=g)
        return [q, k, v, o, act, mmfp4.marlin_gemm_fp4(act, *w["down"], group_size=g)]
    if path == "mlp":
        act = mmfp4.mmfp4_fused_gate_up(s["x"], *s["gate"], *s["up"], group_size=g)
        return [act, s["down"](act)]
    if path == "moe":
        probs, ids = mmfp4.router_softmax_topk(s["logits"], c["topk"])
        if c["shared"]:
            out = mmfp4.moe_fused_dispatch_shared_fp4(
                s["x"], *s["shared_gate_up"], *s["shared_down"], *s["gate_up"], *s["down"],
                ids, probs, g)
        else:
            out = mmfp4.moe_mlp_fp4(s["x"], *s["gate_up"], *s["down"], ids, probs, g)
        return [probs, ids, out]
    if path == "dequant":
        deq = mmfp4.dequant_int4 if c["fmt"] == "int4" else mmfp4.dequant_fp4
        return deq(*s["w"], c["k"], c["n"], g)
    if c["fmt"] == "int4":
        return list(mmfp4.pack_u4_weights(s["w"], g))
    return list(mmfp4.quantize_fp4(s["w"], g))


# --------------------------------------------------------------------- work
def _matrix_bytes(c, n, k):
    """Packed words and the scales (and zero points) of an [n, k] matrix."""
    return n * k / 2 + 2 * n * (k // c["group"]) * (2 if c.get("fmt") == "int4" else 1)


def work(c):
    path = c["path"]
    if path == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": _matrix_bytes(c, n, k) + 2 * m * (k + n), "flops": 2 * m * n * k}
    if path in ("layer", "mlp"):
        h, i, m = c["hidden"], c["inter"], c["m"]
        mats = [(2 * i, h), (h, i)]
        if path == "layer":
            mats += [(h + 2 * c["kv"], h), (h, h)]
            acts = 3 * h + i + (h + 2 * c["kv"]) + 2 * h   # fp4: down reads its own act
            if c["fmt"] == "int4":
                acts += 2 * i
        else:
            acts = 2 * h + i
        return {"bytes": sum(_matrix_bytes(c, n, k) for n, k in mats) + 2 * m * acts,
                "flops": sum(2 * m * n * k for n, k in mats)}
    if path == "moe":
        t, e, k, h, i = c["tokens"], c["experts"], c["topk"], c["hidden"], c["inter"]
        per = _matrix_bytes(c, 2 * i, h) + _matrix_bytes(c, h, i)
        hit = e * (1 - (1 - k / e) ** t) + c["shared"]   # experts that some token visits
        return {"bytes": hit * per + 2 * t * (2 * h + e) + 10 * t * k,
                "flops": 6 * t * (k + c["shared"]) * h * i}
    n, k = c["n"], c["k"]
    return {"bytes": _matrix_bytes(c, n, k) + 2 * n * k, "flops": 0}


# ---------------------------------------------------------------- tolerance
def tolerance(c):
    # Packed words, scales, zero points and expanded weights are defined to the
    # bit.
    if c["path"] in ("dequant", "quantize"):
        return "exact"
    # fp16 results of fp32 sums: one rounding of the result (2e-4) and, above
    # 32 rows, one of each weight.  Chained products add the rounding of the
    # activation between them.
    return {"rel": 1.5e-3, "max": 2e-2}


# -------------------------------------------------------------------- exact
def _codes(words):
    """int32 words [K/8, N] -> codes [K, N]."""
    sh = torch.arange(0, 32, 4, device=words.device, dtype=torch.int32)
    return ((words.unsqueeze(1) >> sh.view(1, 8, 1)) & 15).flatten(0, 1)


def _dense(c, w, rowpacked=False):
    """A quantized matrix as float64 [K, N]."""
    words = w[0].t() if rowpacked else w[0]
    codes = _codes(words)
    s = w[1].double().repeat_interleave(c["group"], 0)
    if len(w) == 3:
        return (codes.double() - w[2].double().repeat_interleave(c["group"], 0)) * s
    return torch.tensor(E2M1, dtype=torch.float64, device=words.device)[codes.long()] * s


def _swiglu(g, u):
    return g * torch.sigmoid(g) * u


def exact(c, seed):
    s, path = _inputs(c, seed), c["path"]
    mm = lambda x, w: x.double() @ _dense(c, w)  # noqa: E731
    if path == "gemm":
        return mm(s["x"], s["w"])
    if path == "layer":
        w, x = s["w"], s["x"]
        if c["fmt"] == "int4":
            return [mm(x[n], w[n]) for n in ("qkv", "o", "gate_up", "down")]
        act = _swiglu(mm(x["gate_up"], w["gate"]), mm(x["gate_up"], w["up"]))
        return [mm(x["qkv"], w["q"]), mm(x["qkv"], w["k"]), mm(x["qkv"], w["v"]),
                mm(x["o"], w["o"]), act, mm(act, w["down"])]
    if path == "mlp":
        x = s["x"].double()
        act = _swiglu(x @ _dense(c, s["gate"], True), x @ _dense(c, s["up"], True))
        return [act, act @ _dense(c, s["down"], True)]
    if path == "moe":
        lg = s["logits"].double()
        # equal logits go to the lower expert, as the entry point documents
        ids = torch.sort(lg, dim=-1, descending=True, stable=True)[1][:, :c["topk"]]
        p = torch.softmax(lg, -1).gather(1, ids)
        p = p / p.sum(-1, keepdim=True)
        x, i = s["x"].double(), c["inter"]

        def mlp(rows, gu, dn):
            h = rows @ _dense(c, gu)
            return _swiglu(h[:, :i], h[:, i:]) @ _dense(c, dn)

        out = torch.zeros_like(x)
        if c["shared"]:
            out += mlp(x, s["shared_gate_up"], s["shared_down"])
        gu, dn = s["gate_up"], s["down"]
        for e in range(c["experts"]):
            t, slot = (ids == e).nonzero(as_tuple=True)
            if t.numel():
                out[t] += p[t, slot].unsqueeze(1) * mlp(x[t], (gu[0][e], gu[1][e]),
                                                        (dn[0][e], dn[1][e]))
        return [p, None, out]
    if path == "dequant":
        return _dense(c, s["w"])
    x = s["w"].double().unflatten(-1, (-1, c["group"]))
    if c["fmt"] == "int4":
        return [None, ((x.amax(-1) - x.amin(-1)) / 15).clamp_min(1e-7).t().contiguous(), None]
    return [None, (x.abs().amax(-1) / 6).clamp_min(1e-7 / 6).t().contiguous()]
