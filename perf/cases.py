"""The work that a program using this library gives it, as cases that can be timed and compared.

Each case is one call sequence through the public entry points of `prismwing_amd`, on inputs made
from a seed with plain torch: block-FP8 projections, the BF16 wide linear, one whole expert, the
routed-MoE layer at decode widths (with and without its router), the host-array call that takes
the reference's bindings, and the routed prefill. `exact` computes the same results in 64 bits
without the library.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mimo-prismwing_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import prismwing_amd as P  # noqa: E402

TOP_K = 8
_MODES = {"A": P.MODE_A, "B": P.MODE_B}
_DTYPES = {"f32": P.DTYPE_F32, "bf16": P.DTYPE_BF16, "f32_raw": P.DTYPE_F32_RAW}
_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f32_raw": torch.float32}
_runtime = None


def _rt() -> P.WideMoeRuntime:
    """The process's one runtime on device 0, as a serving program keeps it."""
    global _runtime
    if _runtime is None:
        _runtime = P.WideMoeRuntime.compile(0)
    return _runtime


# --------------------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: one expert-sized projection of one token (latency)
        {"name": "projection_w1", "kind": "linear", "rows": 2048, "columns": 4096, "width": 1, "mode": "A",
         "x": "bf16", "out": "bf16"},
        # attention QKV of a decode step, separate q/k/v tensors, the reference's own mode and types
        {"name": "qkv_w8", "kind": "linear", "rows": 13568, "columns": 4096, "width": 8, "mode": "B", "x": "f32",
         "out": "f32"},
        # the variant whose k tensor ends in a partial scale block, an odd batch wider than eight,
        # exact f32 activations and unrounded sums
        {"name": "qkv_ragged_w13", "kind": "linear", "rows": 13800, "columns": 4096, "width": 13, "mode": "A",
         "x": "f32", "out": "f32_raw"},
        # attention output projection (BF16 weights) of a decode step
        {"name": "oproj_w8", "kind": "bf16", "rows": 4096, "columns": 8192, "width": 8, "x": "f32", "out": "f32"},
        # the dense FP8 MLP of a non-routed layer, a decode batch of 24 rows
        {"name": "dense_mlp_w24", "kind": "expert", "hidden": 4096, "inter": 16384, "width": 24, "mode": "B",
         "x": "bf16", "out": "bf16"},
        # one token through the routed layer (single-stream decoding)
        {"name": "layer_w1", "kind": "layer", "hidden": 4096, "inter": 2048, "experts": 256, "width": 1, "mode": "A",
         "x": "bf16", "out": "bf16", "routed": False, "skew": 0.0},
        # the headline decode batch with its router in one call
        {"name": "layer_w8", "kind": "layer", "hidden": 4096, "inter": 2048, "experts": 256, "width": 8, "mode": "A",
         "x": "bf16", "out": "bf16", "routed": True, "skew": 0.0},
        # an odd serving batch, routes in hand and skewed, exact f32 activations, unrounded sums
        {"name": "layer_skewed_w19", "kind": "layer", "hidden": 4096, "inter": 2048, "experts": 256, "width": 19,
         "mode": "A", "x": "f32", "out": "f32_raw", "routed": False, "skew": 1.1},
        # the widest decode batch, FP8 activations, with its router
        {"name": "layer_w32", "kind": "layer", "hidden": 4096, "inter": 2048, "experts": 256, "width": 32, "mode": "B",
         "x": "bf16", "out": "bf16", "routed": True, "skew": 0.0},
        # the reference's own call: host arrays and per-expert bindings, eight rows, synchronous
        {"name": "execute_w8", "kind": "execute", "hidden": 4096, "inter": 2048, "experts": 256, "width": 8,
         "mode": "B", "skew": 0.0},
        # a short ragged prompt: its router, then the routed prefill
        {"name": "prefill_200", "kind": "prefill", "hidden": 4096, "inter": 2048, "experts": 256, "width": 200,
         "x": "bf16", "out": "bf16", "skew": 0.0},
        # the long prefill
        {"name": "prefill_2048", "kind": "prefill", "hidden": 4096, "inter": 2048, "experts": 256, "width": 2048,
         "x": "bf16", "out": "bf16", "skew": 0.0},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "bf16", "expert", "layer", "layer", "layer", "execute", "prefill"])
    width = _log_int(rng, 1, 32)
    c = {"kind": kind, "width": width}
    if kind in ("linear", "bf16"):
        c["rows"] = _log_int(rng, 512, 16384) + (0 if kind == "bf16" else 8 * rng.randrange(2))
        c["columns"] = 128 * _log_int(rng, 8, 64)
        if kind == "linear":
            c["mode"] = rng.choice("AB")
        c["x"] = rng.choice(["f32", "bf16"])
        c["out"] = rng.choice(["f32", "bf16", "f32_raw"])
        return c
    c["hidden"] = rng.choice([2048, 4096, 4096, 4096])
    c["inter"] = rng.choice([512, 1024, 1536, 2048, 2048, 2048])
    if kind == "expert":
        c["inter"] = rng.choice([2048, 2048, 4096, 8192, 16384])
    else:
        c["experts"] = rng.choice([64, 128, 256, 256])
        c["skew"] = rng.choice([0.0, 0.0, 1.1])
    if kind == "prefill":
        c["width"] = _log_int(rng, 33, 2048)
    else:
        c["mode"] = rng.choice("AB")
    if kind == "layer":
        c["routed"] = rng.random() < 0.5
    if kind != "execute":
        c["x"] = rng.choice(["f32", "bf16", "bf16"])
        c["out"] = rng.choice(["f32", "bf16", "bf16"])
    return c


# -------------------------------------------------------------------------------- inputs
def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFFF)


def _fp8_weight(g, count, rows, columns):
    """[count, rows, columns] e4m3 codes of N(0, 112^2) clamped to +-448, and f32 block scales that
    put the weights at about N(0, 0.02^2), each block's scale within a factor of two of that."""
    codes = torch.empty((count, rows, columns), dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 27) // (rows * columns))
    for i in range(0, count, step):
        part = codes[i:i + step]
        z = torch.randn(part.shape, generator=g, device="cuda").mul_(112.0).clamp_(-448.0, 448.0)
        part.copy_(z.to(torch.float8_e4m3fn).view(torch.uint8))
    u = torch.rand((count, (rows + 127) // 128, columns // 128), generator=g, device="cuda")
    return codes, torch.exp2(2.0 * u - 1.0).mul_(0.02 / 112.0)


def _activations(case, seed):
    """Normalised activations: N(0, 1) with a few large channels."""
    g = _gen(seed, 1)
    columns = case["columns"] if "columns" in case else case["hidden"]
    x = torch.randn((case["width"], columns), generator=g, device="cuda")
    x *= torch.where(torch.rand((columns,), generator=g, device="cuda") < 0.01, 6.0, 1.0)
    return x.to(_TORCH[case.get("x", "f32")])


def _segments(case):
    """Rows of the tensors that a projection concatenates: q, k and v, or one tensor."""
    n = case["rows"]
    return [12288, n - 12800, 512] if 12800 < n <= 13952 else [n]


def _projection_weights(case, seed):
    g = _gen(seed, 2)
    return [tuple(t[0] for t in _fp8_weight(g, 1, n, case["columns"])) for n in _segments(case)]


def _bf16_weight(case, seed):
    return torch.randn((case["rows"], case["columns"]), generator=_gen(seed, 2), device="cuda").mul_(0.02).bfloat16()


def _expert_weights(case, seed):
    n, h, i = case.get("experts", 1), case["hidden"], case["inter"]
    g = _gen(seed, 2)
    return {"gate": _fp8_weight(g, n, i, h), "up": _fp8_weight(g, n, i, h), "down": _fp8_weight(g, n, h, i)}


def _router(case, seed):
    """BF16 router weights and an f32 correction bias; skew adds a Zipf popularity to the bias."""
    g = _gen(seed, 3)
    n = case["experts"]
    w = torch.randn((n, case["hidden"]), generator=g, device="cuda").mul_(0.02).bfloat16()
    bias = torch.rand((n,), generator=g, device="cuda").mul_(0.02).sub_(0.01)
    rank = torch.randperm(n, generator=g, device="cuda").add_(1)
    return w, bias - 0.05 * case["skew"] * torch.log(rank.float())


def _routes64(case, x, seed):
    """(expert ids, weights) [width, 8] of the noaux top-8 router, in 64 bits."""
    w, bias = _router(case, seed)
    s = torch.sigmoid(x.double() @ w.double().t())
    ids = torch.topk(s + bias.double(), TOP_K, dim=1).indices
    weights = s.gather(1, ids)
    return ids, weights / weights.sum(1, keepdim=True)


def _bind_experts(case, weights):
    rt, h, i = _rt(), case["hidden"], case["inter"]
    n = case.get("experts", 1)
    torch.cuda.synchronize()

    def bound(which, rows, columns):
        codes, scales = weights[which]
        return [rt.bind_projection_device(codes[e], scales[e], rows, columns) for e in range(n)]
    return bound("gate", i, h), bound("up", i, h), bound("down", h, i)


def prepare(case, seed):
    rt, kind = _rt(), case["kind"]
    x = _activations(case, seed)
    st = {"case": case, "rt": rt, "x": x}
    out_dtype = _TORCH[case.get("out", "f32")]
    if kind == "linear":
        segs = _projection_weights(case, seed)
        if len(segs) == 1:
            st["weights"] = segs
            torch.cuda.synchronize()
            st["proj"] = rt.bind_projection_device(*segs[0], case["rows"], case["columns"])
        else:
            st["proj"] = rt.bind_segments([(w.cpu().numpy(), s.cpu().numpy()) for w, s in segs], scan_codes=False)
        st["out"] = torch.empty((case["width"], case["rows"]), dtype=out_dtype, device="cuda")
    elif kind == "bf16":
        st["weights"] = _bf16_weight(case, seed)
        torch.cuda.synchronize()
        st["proj"] = rt.bind_bf16_device(st["weights"], case["rows"], case["columns"])
        st["out"] = torch.empty((case["width"], case["rows"]), dtype=out_dtype, device="cuda")
    else:
        st["weights"] = _expert_weights(case, seed)
        st["projs"] = _bind_experts(case, st["weights"])
        st["out"] = torch.empty((case["width"], case["hidden"]), dtype=out_dtype, device="cuda")
        if kind != "execute":
            st["bank"] = rt.expert_bank(*st["projs"])
        if kind == "execute":
            ids, weights = _routes64(case, x, seed)
            st["ids"], st["route_w"] = ids.cpu().numpy(), weights.float().cpu().numpy()
            st["x"] = x.cpu().numpy()
        elif kind != "expert":
            if kind == "layer" and not case["routed"]:
                ids, weights = _routes64(case, x, seed)
                st["ids"], st["route_w"] = ids.int().contiguous(), weights.float().contiguous()
            else:
                st["router"], st["bias"] = _router(case, seed)
                st["ids"] = torch.empty((case["width"], TOP_K), dtype=torch.int32, device="cuda")
                st["route_w"] = torch.empty((case["width"], TOP_K), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------------------------- calls
def _bindings(st):
    """The reference's expert bindings of one batch, from its routes."""
    gates, ups, downs = st["projs"]
    rows = {}
    for p, (ids, weights) in enumerate(zip(st["ids"].tolist(), st["route_w"].tolist())):
        for e, w in zip(ids, weights):
            pos, rw = rows.setdefault(e, ([], []))
            pos.append(p)
            rw.append(w)
    return [P.WideExpertBinding(e, pos, rw, gates[e], ups[e], downs[e]) for e, (pos, rw) in sorted(rows.items())]


def run(st):
    c, rt, out = st["case"], st["rt"], st["out"]
    kind, width = c["kind"], c["width"]
    if kind == "execute":
        return rt.execute(st["x"], _bindings(st), mode=_MODES[c["mode"]]).output
    types = {"x_dtype": _DTYPES[c["x"]], "out_dtype": _DTYPES[c["out"]]}
    if kind == "linear":
        rt.fp8_linear_device(st["proj"], st["x"], width, out, mode=_MODES[c["mode"]], **types)
    elif kind == "bf16":
        rt.bf16_linear_device(st["proj"], st["x"], width, out, **types)
    elif kind == "expert":
        rt.expert_forward_device(st["bank"], 0, st["x"], width, out, mode=_MODES[c["mode"]], **types)
    elif kind == "layer" and c["routed"]:
        rt.moe_layer_routed_device(st["bank"], st["x"], width, st["router"], st["bias"], st["ids"], st["route_w"], out,
                                   mode=_MODES[c["mode"]], **types)
        return [out, st["ids"], st["route_w"]]
    elif kind == "layer":
        rt.moe_layer_device(st["bank"], st["x"], width, st["ids"], st["route_w"], out, mode=_MODES[c["mode"]], **types)
    else:
        rt.route_device(st["x"], width, c["hidden"], st["router"], c["experts"], st["bias"], st["ids"], st["route_w"],
                        x_dtype=types["x_dtype"])
        rt.moe_prefill_device(st["bank"], st["x"], width, st["ids"], st["route_w"], out, **types)
        return [out, st["ids"], st["route_w"]]
    return out


# ------------------------------------------------------------------- what a pass has to do
_BYTES = {"f32": 4, "bf16": 2, "f32_raw": 4}


def work(case):
    w, kind = case["width"], case["kind"]
    if kind in ("linear", "bf16"):
        r, k = case["rows"], case["columns"]
        weight = r * k * 2 if kind == "bf16" else r * k + -(-r // 128) * (k // 128) * 4
        return {"bytes": weight + w * k * _BYTES[case["x"]] + w * r * _BYTES[case["out"]], "flops": 2 * w * r * k}
    h, i = case["hidden"], case["inter"]
    expert = 3 * h * i + 3 * (h // 128) * (i // 128) * 4
    io = w * h * (_BYTES[case.get("x", "f32")] + _BYTES[case.get("out", "f32")])
    if kind == "expert":
        return {"bytes": expert + io, "flops": 6 * w * h * i}
    e = case["experts"]
    # distinct experts that uniform routes of w tokens reach, on average (skewed routes: fewer)
    used = e * (1.0 - (1.0 - TOP_K / e) ** w)
    routed = kind == "prefill" or case.get("routed", False)
    router = e * h * 2 if routed else 0
    return {"bytes": used * expert + io + w * TOP_K * 8 + router,
            "flops": 6 * w * TOP_K * h * i + (2 * w * e * h if routed else 0)}


def tolerance(case):
    """About four times the distance from `exact`: 1.7e-3 for a bf16-rounded result, 2.7e-3 where
    mode B's bf16 stages and e4m3 re-quantisation come before it, 1.5e-7 (one projection) to 2.7e-7
    (a layer) for unrounded 32-bit sums of exact products."""
    mode = case.get("mode", "A" if case["kind"] == "bf16" else "B")
    if case["kind"] in ("linear", "bf16"):
        return {"rel": 1e-6 if mode == "A" and case["out"] == "f32_raw" else 7e-3}
    if mode == "A":
        return {"rel": 1.2e-6 if case.get("out") == "f32_raw" else 7e-3}
    return {"rel": 1.1e-2}


# ------------------------------------------------------------------------ the same in 64 bits
def _dequant(codes, scales):
    w = codes.view(torch.float8_e4m3fn).float().double()
    s = scales.double().repeat_interleave(128, 0)[:w.shape[0]].repeat_interleave(128, 1)
    return w * s


def _quant(x):
    """Activations after the dynamic e4m3 quantiser (one scale per row and 128 columns), in 64 bits."""
    g = x.float().reshape(x.shape[0], -1, 128)
    # a tensor divisor: torch divides by a Python number through its reciprocal, an ulp off at times
    scale = g.abs().amax(2, keepdim=True).clamp_(min=1e-10) / torch.full((), 448.0, device="cuda")
    q = (g / scale).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn).float()
    return (q.double() * scale.double()).reshape(x.shape)


def _bf16(x):
    return x.bfloat16().double()


def _expert64(mode, x, gate, up, down):
    """One expert on rows x, unrounded in mode A, with mode B's quantisers and bf16 stages."""
    if mode == "A":
        x = x.double()
        return ((x @ gate.t()) * torch.sigmoid(x @ gate.t()) * (x @ up.t())) @ down.t()
    x = _quant(x)
    g, u = _bf16(x @ gate.t()), _bf16(x @ up.t())
    return _bf16(_quant(_bf16(_bf16(g * torch.sigmoid(g)) * u)) @ down.t())


def exact(case, seed):
    x, kind = _activations(case, seed), case["kind"]
    if kind == "linear":
        xs = _quant(x) if case["mode"] == "B" else x.double()
        return torch.cat([xs @ _dequant(w, s).t() for w, s in _projection_weights(case, seed)], 1)
    if kind == "bf16":
        return x.double() @ _bf16_weight(case, seed).double().t()
    weights = _expert_weights(case, seed)

    def expert(e):
        return [_dequant(weights[k][0][e], weights[k][1][e]) for k in ("gate", "up", "down")]
    if kind == "expert":
        return _expert64(case["mode"], x, *expert(0))
    ids, route_w = _routes64(case, x, seed)
    given = kind == "execute" or (kind == "layer" and not case["routed"])
    if given:  # the call was handed these weights as f32
        route_w = route_w.float().double()
    out = torch.zeros((case["width"], case["hidden"]), dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        rows, slots = (ids == e).nonzero(as_tuple=True)
        y = _expert64(case.get("mode", "B"), x[rows], *expert(e))
        out.index_add_(0, rows, y * route_w[rows, slots].unsqueeze(1))
    if kind == "execute":
        return out.cpu().numpy()
    return out if given else [out, None, None]
