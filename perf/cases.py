"""The work a user of this framework has it do, as measurable cases.

A case is one call of a public entry point on one set of inputs:

* ``layer``  -- ``MoeLayer.forward``: router, top-k, routed experts, combine
  and the shared expert where the layer has one, for the four packed bank
  formats, from one decoded token to a prefill batch;
* ``dense``  -- the ``fused`` backend of the registry on dense bf16 banks;
* ``linear`` -- ``fused_*_linear``, one packed projection;
* ``expert`` -- ``fused_*_expert_forward``, one packed expert.

Weights are N(0, 0.02) quantised per bank format, tokens N(0, 1) in bf16, made
here in plain torch from the seed alone; :func:`exact` dequantises the same
banks and computes the same call in 64 bits.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "freetoken-intel_amd"))

DEV = "cuda"

# The layer shapes of the benchmark configurations (INT8 per-channel, GPTQ
# int4 g128, block-FP8 with a shared expert, MXFP4 with biases), and generic
# ones beside them: other hidden and intermediate sizes, expert counts, a
# shared expert beside int4 experts, grouped INT8, MXFP4 without biases.
SHAPES = {
    "int8_e16": dict(fmt="int8", E=16, H=1024, I=512, k=2, shared=0, groups=1, oai=False),
    "gptq_e128": dict(fmt="gptq", E=128, H=2048, I=768, k=8, shared=0, groups=1, oai=False),
    "fp8_e256": dict(fmt="fp8", E=256, H=2048, I=512, k=8, shared=512, groups=1, oai=False),
    "mxfp4_e32": dict(fmt="mxfp4", E=32, H=2880, I=2880, k=4, shared=0, groups=1, oai=True),
    "gptq_e60_shared": dict(fmt="gptq", E=60, H=2048, I=1408, k=4, shared=5632, groups=1, oai=False),
    "fp8_e64": dict(fmt="fp8", E=64, H=3072, I=1024, k=6, shared=0, groups=1, oai=False),
    "int8_e64": dict(fmt="int8", E=64, H=2048, I=1024, k=4, shared=0, groups=8, oai=False),
    "mxfp4_e64": dict(fmt="mxfp4", E=64, H=2048, I=768, k=8, shared=0, groups=1, oai=False),
}
DENSE = {
    "bf16_e128": dict(E=128, H=2048, I=768, k=8),
    "bf16_e16": dict(E=16, H=1024, I=512, k=2),
}
# projections of one expert, [K, N]: gate_up and down of the layers above
LINEAR = ((2048, 768), (2048, 1536), (768, 2048), (2048, 1024), (512, 2048), (1024, 1024), (1408, 2048))
FORMATS = ("gptq", "fp8", "int8", "mxfp4")


def _layer(shape, T, name=None):
    c = dict(kind="layer", T=T, **SHAPES[shape])
    return dict(c, name=name) if name else c


def _dense(shape, T, name=None):
    c = dict(kind="dense", T=T, **DENSE[shape])
    return dict(c, name=name) if name else c


def _linear(fmt, M, K, N, dtype, name=None):
    c = dict(kind="linear", fmt=fmt, M=M, K=K, N=N, dtype=dtype)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one sequence decoding: one token a step, latency and launches
        _layer("fp8_e256", 1, "fp8_decode_1"),
        # the headline batch of the benchmark
        _layer("fp8_e256", 16, "fp8_decode_16"),
        # a server's decode batch of many sequences, a ragged count
        _layer("fp8_e256", 100, "fp8_batch_100"),
        # one prefill chunk
        _layer("fp8_e256", 2048, "fp8_prefill_2048"),
        # int4 decode, a small server batch
        _layer("gptq_e128", 16, "gptq_decode_16"),
        # a prompt of a thousand tokens through int4 experts
        _layer("gptq_e128", 1000, "gptq_prefill_1000"),
        # few large experts with biases and the clamped activation: a decode batch and a prefill chunk
        _layer("mxfp4_e32", 32, "mxfp4_decode_32"),
        _layer("mxfp4_e32", 4096, "mxfp4_prefill_4096"),
        # a small model: a few sequences, and a prompt of odd length
        _layer("int8_e16", 4, "int8_decode_4"),
        _layer("int8_e16", 777, "int8_prefill_777"),
        # unquantised experts through the backend registry, a short prompt of odd length
        _dense("bf16_e128", 333, "bf16_dense_333"),
        # one packed projection called by itself, the rows one expert gets
        _linear("gptq", 32, 2048, 768, "bf16", "gptq_linear_32"),
    ]


def _size(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    u = rng.random()
    if u < 0.65:
        shape = rng.choice(sorted(SHAPES))
        return _layer(shape, _size(rng, 1, 2048 if shape in ("gptq_e60_shared", "fp8_e64") else 4096))
    if u < 0.75:
        return _dense(rng.choice(sorted(DENSE)), _size(rng, 1, 2048))
    fmt = rng.choice(FORMATS)
    if u < 0.9:
        K, N = rng.choice(LINEAR)
        return _linear(fmt, _size(rng, 1, 1024), K, N, rng.choice(("bf16", "bf16", "bf16", "f16", "f32")))
    H, I = rng.choice(((2048, 768), (2048, 512), (1024, 512), (3072, 1024)))
    return dict(kind="expert", fmt=fmt, M=_size(rng, 1, 1024), H=H, I=I)


# ------------------------------------------------------------------ inputs in plain torch
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _quantise(fmt, w, groups=1):
    """[N, K] float32 -> the tensors of one packed projection."""
    N, K = w.shape
    if fmt == "fp8":  # e4m3, one fp32 scale per 128 x 128 block
        b = w.reshape(N // 128, 128, K // 128, 128)
        s = b.abs().amax(dim=(1, 3)).clamp_min(1e-12) / 448.0
        return [(b / s[:, None, :, None]).reshape(N, K).clamp(-448, 448).to(torch.float8_e4m3fn), s]
    if fmt == "int8":  # offset-binary bytes, four to a word, fp32 scales per row and K group
        b = w.reshape(N, groups, K // groups)
        s = b.abs().amax(dim=2).clamp_min(1e-12) / 127.0
        q = (b / s[:, :, None]).round().clamp(-127, 127).reshape(N, K) + 128
        return [q.to(torch.uint8).contiguous().view(torch.int32), s]
    if fmt == "gptq":  # int4 with zero points per 128 rows of K; stored zero = zero - 1
        b = w.t().reshape(K // 128, 128, N)
        lo, hi = b.amin(dim=1).clamp_max(0), b.amax(dim=1).clamp_min(0)
        s = ((hi - lo).clamp_min(1e-6) / 15.0).to(torch.float16)
        z = (-lo / s.float()).round().clamp(1, 15)
        q = ((b / s.float()[:, None, :]).round() + z[:, None, :]).clamp(0, 15).reshape(K // 8, 8, N).to(torch.int32)
        zz = (z - 1).to(torch.int32).reshape(K // 128, N // 8, 8)
        qw, qz = torch.zeros(K // 8, N, dtype=torch.int32, device=w.device), torch.zeros(K // 128, N // 8, dtype=torch.int32, device=w.device)
        for i in range(8):
            qw |= q[:, i] << (4 * i)
            qz |= zz[:, :, i] << (4 * i)
        return [qw, qz, s]
    b = w.reshape(N, K // 32, 32)  # mxfp4: e2m1 pairs (low nibble first), one e8m0 byte per 32
    e = torch.ceil(torch.log2(b.abs().amax(dim=2).clamp_min(1e-12) / 6.0)).clamp(-127, 127)
    v = (b * torch.exp2(-e)[:, :, None])
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device)
    q = torch.bucketize(v.abs().contiguous(), edges).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
    return [(q[..., 0::2] | (q[..., 1::2] << 4)).contiguous(), (e + 127).to(torch.uint8)]


def _dequantise(fmt, t, groups=1):
    """One packed projection -> [N, K] float64."""
    if fmt == "bf16":
        return t[0].double()
    if fmt == "fp8":
        return t[0].double() * t[1].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    if fmt == "int8":
        q = t[0].view(torch.uint8).double() - 128
        return q * t[1].double().repeat_interleave(q.shape[1] // t[1].shape[1], 1)
    if fmt == "gptq":
        sh = torch.arange(0, 32, 4, device=t[0].device, dtype=torch.int32)
        q = ((t[0][:, None, :] >> sh[None, :, None]) & 15).reshape(-1, t[0].shape[1])
        z = ((t[1][:, :, None] >> sh) & 15).reshape(t[1].shape[0], -1) + 1
        w = (q - z.repeat_interleave(128, 0)).double() * t[2].double().repeat_interleave(128, 0)
        return w.t()
    lut = torch.tensor(_E2M1 + tuple(-v for v in _E2M1), dtype=torch.float64, device=t[0].device)
    q = torch.stack((t[0] & 15, t[0] >> 4), dim=-1).long()
    v = lut[q].reshape(t[0].shape[0], -1, 32) * torch.exp2(t[1].double() - 127)[:, :, None]
    return v.reshape(t[0].shape[0], -1)


def _banks(fmt, E, N, K, groups, rnd):
    """Packed projections of E experts, stacked."""
    if fmt == "bf16":
        out = [torch.empty(E, N, K, dtype=torch.bfloat16, device=DEV)]
        for e in range(E):
            out[0][e] = rnd(N, K) * 0.02
        return out
    out = None
    for e in range(E):
        t = _quantise(fmt, rnd(N, K) * 0.02, groups)
        if out is None:
            out = [torch.empty((E, *v.shape), dtype=v.dtype, device=DEV) for v in t]
        for o, v in zip(out, t):
            o[e].view(torch.uint8).copy_(v.contiguous().view(torch.uint8))
    return out


def _inputs(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)

    kind, d = case["kind"], {}
    if kind == "linear":
        d["w"] = _banks(case["fmt"], 1, case["N"], case["K"], 1, rnd)
        d["x"] = rnd(case["M"], case["K"]).to(_DTYPES[case["dtype"]])
        return d
    H, I = case["H"], case["I"]
    if kind == "expert":
        d["w13"] = _banks(case["fmt"], 1, 2 * I, H, 1, rnd)
        d["w2"] = _banks(case["fmt"], 1, H, I, 1, rnd)
        d["x"] = rnd(case["M"], H).to(torch.bfloat16)
        return d
    E, fmt = case["E"], "bf16" if kind == "dense" else case["fmt"]
    groups = case.get("groups", 1)
    d["w13"] = _banks(fmt, E, 2 * I, H, groups, rnd)
    d["w2"] = _banks(fmt, E, H, I, groups, rnd)
    d["x"] = rnd(case["T"], H).to(torch.bfloat16)
    if kind == "dense":
        d["gating"] = rnd(case["T"], E)
        return d
    d["gate"] = (rnd(E, H) * 0.02).to(torch.bfloat16)
    if case["oai"]:
        d["gate_b"] = (rnd(E) * 0.02).to(torch.bfloat16)
        d["b13"] = (rnd(E, 2 * I) * 0.02).to(torch.bfloat16)
        d["b2"] = (rnd(E, H) * 0.02).to(torch.bfloat16)
    if case["shared"]:
        S = case["shared"]
        d["shared"] = {"w13": (rnd(2 * S, H) * 0.02).to(torch.bfloat16), "w2": (rnd(H, S) * 0.02).to(torch.bfloat16),
                       "gate": (rnd(1, H) * 0.02).to(torch.bfloat16)}
    return d


_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BANK = {"fp8": ("fp8_block", ("weight_", "scale_"), 128), "int8": ("int8_channel", ("weight_packed_", "weight_scale_"), None),
         "gptq": ("gptq_int4", ("qweight_", "qzeros_", "scales_"), 128), "mxfp4": ("mxfp4", ("blocks_", "scales_"), 32)}


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dense":
        from ftmoe.moe import create_moe_backend

        return {"case": case, "backend": create_moe_backend("fused"), "x": d["x"], "w1": d["w13"][0], "w2": d["w2"][0], "gating": d["gating"]}
    if kind in ("linear", "expert"):
        return {"case": case, **d}
    from ftmoe import MoeLayer, proj_from_bank

    fmt, names, group = _BANK[case["fmt"]]
    bank = {n + "gate_up": t for n, t in zip(names, d["w13"])}
    bank.update({n + "down": t for n, t in zip(names, d["w2"])})
    H, I = case["H"], case["I"]
    oai = case["oai"]
    layer = MoeLayer(
        w13=proj_from_bank(fmt, bank, which="gate_up", N=2 * I, K=H, group=group, bias=d.get("b13")),
        w2=proj_from_bank(fmt, bank, which="down", N=H, K=I, group=group, bias=d.get("b2")),
        num_experts=case["E"], hidden=H, inter=I, topk=case["k"], gate_w=d["gate"], gate_b=d.get("gate_b"), shared=d.get("shared"),
        route_mode="topk_softmax" if oai else "softmax_topk", act="swiglu_oai" if oai else "silu")
    return {"case": case, "layer": layer, "x": d["x"]}


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "layer":
        return state["layer"].forward(state["x"])
    if kind == "dense":
        return state["backend"].forward(state["x"], state["w1"], state["w2"], state["gating"], c["k"], True)
    fmt, x = c["fmt"], state["x"]
    if kind == "linear":
        w = [t[0] for t in state["w"]]
        if fmt == "fp8":
            from ftmoe.kernel.fused_fp8_linear import fused_fp8_linear
            return fused_fp8_linear(x, *w)
        if fmt == "gptq":
            from ftmoe.kernel.gptq_fused_linear import fused_gptq_linear
            return fused_gptq_linear(x, *w, group_size=128)
        if fmt == "int8":
            from ftmoe.kernel.fused_int8_linear import fused_int8_linear
            return fused_int8_linear(x, *w, k=c["K"])
        from ftmoe.kernel.fused_mxfp4_linear import fused_mxfp4_linear
        return fused_mxfp4_linear(x, *w)
    w = [t[0] for t in state["w13"]] + [t[0] for t in state["w2"]]
    if fmt == "fp8":
        from ftmoe.kernel.fused_fp8_linear import fused_fp8_expert_forward
        return fused_fp8_expert_forward(x, *w, intermediate=c["I"])
    if fmt == "gptq":
        from ftmoe.kernel.gptq_fused_linear import fused_gptq_expert_forward
        return fused_gptq_expert_forward(x, *w, group_size=128, intermediate=c["I"])
    if fmt == "int8":
        from ftmoe.kernel.fused_int8_linear import fused_int8_expert_forward
        return fused_int8_expert_forward(x, *w, intermediate=c["I"], k_gate_up=c["H"], k_down=c["I"])
    from ftmoe.kernel.fused_mxfp4_linear import fused_mxfp4_expert_forward
    return fused_mxfp4_expert_forward(x, *w, intermediate=c["I"])


def _weight_bytes(fmt, N, K, groups=1):
    if fmt == "bf16":
        return 2 * N * K
    if fmt == "fp8":
        return N * K + 4 * -(-N // 128) * -(-K // 128)
    if fmt == "int8":
        return N * K + 4 * N * groups
    if fmt == "gptq":
        return N * K // 2 + (K // 128) * (N // 2 + 2 * N)
    return N * K // 2 + N * K // 32


def work(case):
    """Bytes: each routed expert's banks once (the number of experts that T
    tokens hit when the routing is spread evenly), the router, the shared
    expert, tokens in and out.  Operations: the products of every routed pair,
    the shared expert and the router."""
    kind = case["kind"]
    if kind == "linear":
        es = 4 if case["dtype"] == "f32" else 2
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _weight_bytes(case["fmt"], N, K) + es * M * (K + N), "flops": 2 * M * N * K}
    H, I = case["H"], case["I"]
    if kind == "expert":
        M = case["M"]
        return {"bytes": _weight_bytes(case["fmt"], 2 * I, H) + _weight_bytes(case["fmt"], H, I) + 4 * M * H, "flops": 6 * M * H * I}
    E, k, T = case["E"], case["k"], case["T"]
    fmt, groups = ("bf16", 1) if kind == "dense" else (case["fmt"], case["groups"])
    hit = E * (1.0 - (1.0 - k / E) ** T)
    b = hit * (_weight_bytes(fmt, 2 * I, H, groups) + _weight_bytes(fmt, H, I, groups)) + 4 * T * H
    f = 6 * T * k * H * I
    if kind == "dense":
        return {"bytes": int(b + 4 * T * E), "flops": f}
    S = case["shared"]
    b += 2 * E * H + (6 * S * H + 2 * H if S else 0) + (2 * E + hit * 2 * (2 * I + H) if case["oai"] else 0)
    return {"bytes": int(b), "flops": f + 2 * T * E * H + 6 * T * S * H}


def tolerance(case):
    """About four times the error against :func:`exact` that the path shows:
    layers and experts 0.0029-0.0038 (hidden activations, router weights and
    the output in bf16, products summed in 32 bits in any order), projections
    0.0017 with a bf16 result, 2.1e-4 with an fp16 one and 5.6e-6 with an fp32
    one (activations enter the matrix cores as bf16 pairs there)."""
    if case["kind"] == "linear":
        return {"rel": {"bf16": 7e-3, "f16": 8e-4, "f32": 2.2e-5}[case["dtype"]]}
    return {"rel": 1.2e-2}


def _mlp(x, w13, w2, I, oai, b13=None, b2=None):
    gu = x @ w13.t()
    if b13 is not None:
        gu = gu + b13.double()
    g, u = gu[:, :I], gu[:, I:]
    if oai:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
        h = (u + 1.0) * g * torch.sigmoid(1.702 * g)
    else:
        h = g * torch.sigmoid(g) * u
    y = h @ w2.t()
    return y if b2 is None else y + b2.double()


def exact(case, seed):
    d = _inputs(case, seed)
    kind, x = case["kind"], d["x"].double()
    if kind == "linear":
        return x @ _dequantise(case["fmt"], [t[0] for t in d["w"]]).t()
    I = case["I"]
    if kind == "expert":
        w13, w2 = (_dequantise(case["fmt"], [t[0] for t in d[n]]) for n in ("w13", "w2"))
        return _mlp(x, w13, w2, I, False)
    fmt, oai = ("bf16", False) if kind == "dense" else (case["fmt"], case["oai"])
    logits = d["gating"].double() if kind == "dense" else x @ d["gate"].double().t()
    if "gate_b" in d:
        logits = logits + d["gate_b"].double()
    if kind == "layer":  # the router is a bf16 projection
        logits = logits.to(torch.bfloat16).double()
    key = logits if oai else torch.softmax(logits, dim=1)
    top, ids = (t[:, :case["k"]] for t in torch.sort(key, dim=1, descending=True, stable=True))  # ties: the lower id
    wts = torch.softmax(top, dim=1) if oai else top / top.sum(dim=1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(case["E"]):
        rows, col = (ids == e).nonzero(as_tuple=True)
        if rows.numel() == 0:
            continue
        w13, w2 = (_dequantise(fmt, [t[e] for t in d[n]]) for n in ("w13", "w2"))
        y = _mlp(x[rows], w13, w2, I, oai, d["b13"][e] if oai else None, d["b2"][e] if oai else None)
        out.index_add_(0, rows, y * wts[rows, col][:, None])
    if "shared" in d:
        s = {n: t.double() for n, t in d["shared"].items()}
        out += torch.sigmoid(x @ s["gate"].t()) * _mlp(x, s["w13"], s["w2"], case["shared"], False)
    return out
