"""The calls whose speed this repository is judged by: forward passes of the
MoE layer and of its decode caller, through the public entry points.

A case is one handle (a layer with its weights on the GPU) and one call on it:

  entry "layer"   moe_forward_async: x and out in device memory
  entry "decode"  moe_decode_async: n tokens of a decode step, device memory
  entry "host"    MoELayer(x, training=...): numpy in, numpy out

T tokens per call on a handle made for `cap` tokens; D -> H -> D experts, E of
them (`lsh` of them the layer's shared experts, `ns` SharedExpertGating's),
k slots of the gate; `w` the weights' type, `x` the activations'; `skew` how
uneven the expert load is ("normal": N(0, 1) router biases, "zipf": Zipf(1.1)).
"""
import ctypes
import math

import numpy as np
import torch

import mixtureofexperts_amd as moe
from mixtureofexperts_amd import _lib
from mixtureofexperts_amd._device import DeviceLayer, GateSpec

_BASE = dict(entry="layer", T=1, cap=1, D=512, H=2048, E=8, k=2, gate="topk", ns=0, lsh=0, etype="gated", act="silu",
             w="f32", x="f32", training=False, drop=False, skew="none")


def _case(name, **kw):
    c = dict(_BASE, **kw)
    c["cap"] = max(c["cap"], c["T"])
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one token of a stories42M-sized Llama2 whose FFNs became 8 experts:
        # the smallest call, three times per generated token
        _case("decode_stories42m", entry="decode", T=1, H=1376),
        # the same layer serving eight sequences at once
        _case("decode_f32_n8", entry="decode", T=8, H=1376),
        # one token of a Mixtral-8x7B-sized layer, bf16 weights, on a handle
        # that also serves prefill
        _case("decode_mixtral_n1", entry="decode", T=1, cap=4096, D=4096, H=14336, w="bf16", skew="normal"),
        # sixteen sequences decoded together on that layer
        _case("decode_mixtral_n16", entry="decode", T=16, cap=4096, D=4096, H=14336, w="bf16", skew="normal"),
        # the README's layer called from Python on host arrays
        _case("readme_host", entry="host", T=32, training=True),
        # MoEConfig's defaults (standard GELU experts, 768/3072, top-2 of 8,
        # 4096 tokens, fp32): a training batch at reference precision
        _case("default_f32", T=4096, D=768, H=3072, etype="standard", act="gelu", training=True),
        # odd sizes everywhere at reference precision: no dimension is a
        # multiple of a tile
        _case("ragged_f32", T=1037, cap=2048, D=1001, H=2731, E=12, k=3),
        # a Mixtral-8x7B layer over a full batch, skewed expert load
        _case("mixtral", T=4096, D=4096, H=14336, w="bf16", x="bf16", training=True, skew="normal"),
        # a short prompt (or a serving step's tokens) on the same layer
        _case("mixtral_48", T=48, cap=4096, D=4096, H=14336, w="bf16", x="bf16", skew="normal"),
        # fine-grained experts with fp8 weights, two always on, Zipf load
        _case("deepseek", T=8192, D=2048, H=1408, E=66, k=6, gate="shared", ns=2, w="fp8", x="bf16", training=True,
              skew="zipf"),
        # a ragged short prompt on that layer
        _case("deepseek_517", T=517, cap=8192, D=2048, H=1408, E=66, k=6, gate="shared", ns=2, w="fp8", x="bf16",
              skew="zipf"),
        # Switch: top-1 of 128 standard experts, a large training batch
        _case("switch", T=16384, D=768, H=3072, E=128, k=1, gate="switch", etype="standard", act="gelu", w="bf16",
              x="bf16", training=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _slots(c):
    if c["gate"] == "expert_choice":
        Er = c["E"] - c["lsh"]
        return c["lsh"] + min(Er, _ec_capacity(c["T"], c["k"], Er))
    return c["lsh"] + c["k"] + (c["ns"] if c["gate"] == "shared" else 0)


def _rows(c):
    """Rows the experts run: the call's (token, expert) pairs."""
    if c["gate"] == "expert_choice":
        Er = c["E"] - c["lsh"]
        return c["T"] * c["lsh"] + Er * min(c["T"], _ec_capacity(c["T"], c["k"], Er))
    return c["T"] * _slots(c)


def _mats(c):
    return 3 if c["etype"] == "gated" else 2


_WSIZE = {"f32": 4, "bf16": 2, "fp8": 1}


def draw(rng):
    while True:
        c = dict(_BASE)
        if rng.random() < 0.35:
            c.update(entry="decode", T=_log_int(rng, 1, 64), D=4 * _log_int(rng, 32, 1024),
                     H=_log_int(rng, 96, 14336), E=_log_int(rng, 4, 128), k=rng.choice((1, 2, 2, 4, 6, 8)),
                     lsh=rng.choice((0, 0, 0, 1, 2)), w=rng.choice(("f32", "bf16", "fp8")),
                     skew=rng.choice(("none", "normal")))
            c["cap"] = max(2 * c["T"], rng.choice((0, 2048)))
            if c["k"] + c["lsh"] > c["E"] or c["T"] * _slots(c) * 3 * c["D"] * c["H"] * _WSIZE[c["w"]] > 8e9:
                continue
        else:
            w = rng.choice(("f32", "bf16", "bf16", "fp8"))
            c.update(T=_log_int(rng, 1, 16384), D=_log_int(rng, 64, 4096), H=_log_int(rng, 64, 14336),
                     E=_log_int(rng, 2, 256), k=rng.choice((1, 2, 2, 3, 4, 6, 8)), w=w,
                     x=rng.choice(("f32", "bf16")) if w != "f32" else "f32",
                     gate=rng.choice(("topk", "topk", "topk", "switch", "shared", "expert_choice")),
                     etype=rng.choice(("gated", "gated", "standard")), training=rng.random() < 0.5,
                     skew=rng.choice(("none", "normal", "zipf")))
            if c["etype"] == "standard":
                c["act"] = rng.choice(("gelu", "relu"))
            if c["gate"] == "switch":
                c["k"] = 1
            if c["gate"] == "shared":
                c["ns"] = rng.choice((1, 2))
            elif rng.random() < 0.15:
                c["lsh"] = rng.choice((1, 2))
            if c["gate"] in ("topk", "switch") and c["training"] and c["lsh"] == 0:
                c["drop"] = rng.random() < 0.3
            if w == "f32" and c["T"] <= 1024 and c["gate"] == "topk" and rng.random() < 0.3:
                c["entry"], c["cap"] = "host", c["T"]
            else:
                c["cap"] = max(c["T"], rng.choice((c["T"], 2 * c["T"], 4096)))
            if c["k"] + c["ns"] + c["lsh"] > c["E"]:
                continue
            if 2 * _rows(c) * _mats(c) * c["D"] * c["H"] > (1.5e11 if w == "f32" else 2.4e12):
                continue
        if c["E"] * _mats(c) * c["D"] * c["H"] * _WSIZE[c["w"]] > (2e8 if c["entry"] == "host" else 2.9e9):
            continue
        return c


# ---- inputs --------------------------------------------------------------------

def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + part) & 0x7FFFFFFFFFFFFFFF)
    return g


def _routed(c):
    return c["E"] - c["lsh"]


def _inputs(c, seed):
    """x, the router's weight (E_router, D) and its bias (None: no bias)."""
    g = _gen(seed, 0)
    x = torch.randn(c["T"], c["D"], generator=g, device="cuda")
    if c["x"] == "bf16":
        x = x.to(torch.bfloat16)
    Er = _routed(c)
    if c["skew"] == "none":
        return x, torch.randn(Er, c["D"], generator=g, device="cuda") / c["D"] ** 0.5, None
    wr = torch.randn(Er, c["D"], generator=g, device="cuda") * 0.02
    if c["skew"] == "normal":
        return x, wr, torch.randn(Er, generator=g, device="cuda")
    ns = c["ns"]
    r = torch.arange(1, Er - ns + 1, device="cuda", dtype=torch.float32)
    return x, wr, torch.cat([torch.zeros(ns, device="cuda"), -1.1 * torch.log(r)])


def _expert(c, seed, e):
    """Expert e's matrices in (out, in) order, their fp8 scales, its biases."""
    g = _gen(seed, 1 + e)
    D, H = c["D"], c["H"]
    shapes = [(H, D), (D, H), (H, D)][:_mats(c)]
    std = (2.0 / D) ** 0.5 if c["w"] == "f32" else 0.02
    ws, ss = [], []
    for shp in shapes:
        w = torch.randn(*shp, generator=g, device="cuda") * std
        s = None
        if c["w"] == "bf16":
            w = w.to(torch.bfloat16)
        elif c["w"] == "fp8":
            s = w.abs().amax(dim=1) / 448.0
            w = (w / s[:, None]).to(torch.float8_e4m3fn)
        ws.append(w)
        ss.append(s)
    bs = [None, None]
    if c["etype"] == "standard":
        bs = [torch.randn(H, generator=g, device="cuda") * 0.02, torch.randn(D, generator=g, device="cuda") * 0.02]
    return ws, ss, bs


def _ptr(t):
    return None if t is None else t.data_ptr()


_ALPHA, _BETA, _CF = 0.01, 0.001, 1.25


def prepare(c, seed):
    c = dict(_BASE, **c)
    x, wr, br = _inputs(c, seed)
    if c["entry"] == "host":
        return _prepare_host(c, seed, x, wr, br)
    spec = {"topk": GateSpec(_lib.MOE_GATE_TOPK, c["k"], 0), "switch": GateSpec(_lib.MOE_GATE_SWITCH, 1, 0),
            "shared": GateSpec(_lib.MOE_GATE_SHARED, c["k"], c["ns"]),
            "expert_choice": GateSpec(_lib.MOE_GATE_EXPERT_CHOICE, 1, 0, float(c["k"]))}[c["gate"]]
    wcode = {"f32": _lib.MOE_F32, "bf16": _lib.MOE_BF16, "fp8": _lib.MOE_FP8_E4M3}[c["w"]]
    act = {"silu": _lib.MOE_ACT_SILU, "gelu": _lib.MOE_ACT_GELU, "relu": _lib.MOE_ACT_RELU}[c["act"]]
    dev = DeviceLayer(num_experts=c["E"],
                      expert_type=_lib.MOE_EXPERT_GATED if c["etype"] == "gated" else _lib.MOE_EXPERT_STANDARD,
                      input_dim=c["D"], hidden_dim=c["H"], output_dim=c["D"], activation=act, gate=spec,
                      weight_dtype=wcode, balance_alpha=_ALPHA, z_loss_weight=_BETA, capacity_factor=_CF,
                      drop_tokens=c["drop"], max_tokens=max(c["cap"], 2 * c["T"] if c["entry"] == "decode" else 1),
                      num_shared_experts=c["lsh"])
    L = _lib.lib()
    wr_mem = wr.t().contiguous()  # the Flux weight's memory, [D][E_router]
    _lib.check(L.moe_set_router(dev.h, _ptr(wr_mem), _ptr(br)), dev.h)
    for e in range(c["E"]):
        ws, ss, bs = _expert(c, seed, e)
        ws, ss = ws + [None] * (3 - len(ws)), ss + [None] * (3 - len(ss))
        _lib.check(L.moe_set_expert(dev.h, e, _lib.MOE_LAYOUT_LLAMA_IN_OUT, wcode, _ptr(ws[0]), _ptr(ws[1]),
                                    _ptr(ws[2]), _ptr(bs[0]), _ptr(bs[1]), _ptr(ss[0]), _ptr(ss[1]), _ptr(ss[2])),
                   dev.h)
    out = torch.zeros(c["T"], c["D"], device="cuda")
    loss = torch.zeros(1, device="cuda")
    return dict(entry=c["entry"], dev=dev, x=x, out=out, loss=loss, T=c["T"], training=int(c["training"]),
                xcode=_lib.MOE_BF16 if c["x"] == "bf16" else _lib.MOE_F32)


def _prepare_host(c, seed, x, wr, br):
    act = {"silu": moe.silu, "gelu": moe.gelu, "relu": moe.relu}[c["act"]]
    cfg = moe.MoEConfig(num_experts=c["E"], expert_type=c["etype"], input_dim=c["D"], hidden_dim=c["H"],
                        output_dim=c["D"], activation=act, gate_type=moe.TopKGating(c["k"]), top_k=c["k"],
                        balance_loss=moe.SwitchTransformerLoss(_ALPHA), z_loss_weight=_BETA, capacity_factor=_CF,
                        drop_tokens=c["drop"], num_shared_experts=c["lsh"], weight_dtype="f32", max_tokens=c["cap"])
    experts = []
    for e in range(c["E"]):
        ws, _, bs = _expert(c, seed, e)
        ws, bs = [w.cpu().numpy() for w in ws], [None if b is None else b.cpu().numpy() for b in bs]
        if c["etype"] == "gated":
            experts.append(moe.GatedExpert(c["D"], c["H"], c["D"], act, w1=ws[0], w2=ws[1], w3=ws[2]))
        else:
            experts.append(moe.StandardExpert(c["D"], c["H"], c["D"], act, w1=ws[0], w2=ws[1], b1=bs[0], b2=bs[1]))
    router = moe.Router(c["D"], _routed(c), cfg.gate_type, weight=wr.cpu().numpy(),
                        bias=None if br is None else br.cpu().numpy())
    layer = moe.MoELayer(cfg, experts=experts, router=router)
    layer.sync_weights()
    return dict(entry="host", layer=layer, x=np.ascontiguousarray(x.cpu().numpy()).T, training=c["training"])


def run(s):
    if s["entry"] == "host":
        out, loss = s["layer"](s["x"], training=s["training"])
        return [out, np.float32(loss)]
    dev = s["dev"]
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if s["entry"] == "decode":
        _lib.check(_lib.lib().moe_decode_async(dev.h, s["x"].data_ptr(), s["T"], s["out"].data_ptr(), stream), dev.h)
        return [s["out"]]
    _lib.check(_lib.lib().moe_forward_async(dev.h, s["x"].data_ptr(), s["xcode"], s["T"], s["training"],
                                            s["out"].data_ptr(), s["loss"].data_ptr(), stream), dev.h)
    return [s["out"], s["loss"]]


# ---- what a pass cannot do without ----------------------------------------------

def work(c):
    c = dict(_BASE, **c)
    T, D, H, Er = c["T"], c["D"], c["H"], _routed(c)
    rows = _rows(c)
    # experts that some token picked (even load), and those always on
    free = Er - c["ns"]
    hit = c["lsh"] + c["ns"] + (free if c["gate"] == "expert_choice" else free * (1 - (1 - c["k"] / free) ** T))
    xsize = 2 if c["x"] == "bf16" else 4
    wbytes = _mats(c) * D * H * _WSIZE[c["w"]] + (4 * (2 * H + D) if c["w"] == "fp8" else 0)
    return {"bytes": T * D * xsize + T * D * 4 + Er * D * 4 + hit * wbytes,
            "flops": 2.0 * rows * _mats(c) * D * H + 2.0 * T * Er * D}


def tolerance(c):
    return {"rel": 1e-5} if c.get("w", "f32") == "f32" or c.get("entry") == "decode" else {"rel": 1e-2}


# ---- the same in 64 bits ----------------------------------------------------------

def _ec_capacity(T, cf, E):
    return int(np.ceil(np.float32(np.float32(T) * np.float32(cf)) / np.float32(E)))


def _gating(c, logits):
    """Gates as a (T, E_router) matrix (0: not picked), the picks as a mask,
    the probabilities, and the index rows the Switch loss divides by."""
    T, E = logits.shape
    ns, k = c["ns"], c["k"]
    gates, picked = torch.zeros_like(logits), torch.zeros_like(logits, dtype=torch.bool)
    if c["gate"] == "expert_choice":
        probs = torch.softmax(logits, dim=1)
        C = _ec_capacity(T, k, E)
        top = torch.topk(logits, min(C, T), dim=0).indices
        picked.scatter_(0, top, True)
        return torch.where(picked, probs, gates), picked, probs, C
    p = torch.softmax(logits[:, ns:], dim=1)
    v, i = torch.topk(p, k, dim=1)
    v = v / v.sum(dim=1, keepdim=True)
    if c["gate"] == "shared":
        v = v * (1 - ns / (ns + k))
        gates[:, :ns], picked[:, :ns] = 1.0 / (ns + k), True
        probs = torch.cat([torch.full((T, ns), 1.0 / E, dtype=p.dtype, device=p.device), p * (1 - ns / E)], dim=1)
    else:
        probs = p
    gates.scatter_(1, i + ns, v)
    picked.scatter_(1, i + ns, True)
    if c["drop"]:  # the first `cap` tokens of each expert stay, gates renormalised
        cap = int(np.ceil(np.float32(_CF) * np.float32(T) / np.float32(E)))
        picked = picked & (picked.to(torch.int32).cumsum(dim=0) <= cap)
        gates = torch.where(picked, gates, torch.zeros_like(gates))
        s = gates.sum(dim=1, keepdim=True)
        gates = torch.where(s > 0, gates / torch.where(s > 0, s, torch.ones_like(s)), gates)
    return gates, picked, probs, (ns if c["gate"] == "shared" else 0) + k


def _loss(c, logits, picked, probs, rows):
    T, E = probs.shape
    lsh = c["lsh"]
    n = picked.sum(dim=0).double()
    f = torch.zeros(E, dtype=torch.float64, device=probs.device)
    f[lsh:] = n[: E - lsh]  # shared experts of the layer: the loss sees the shifted ids
    if c["gate"] == "expert_choice" and 0 < lsh <= E:
        f[lsh - 1] += T * rows - n.sum()
    return _ALPHA * E * (f / (T * rows) * probs.mean(dim=0)).sum() + _BETA * torch.logsumexp(logits, dim=1).square().mean()


def exact(c, seed):
    c = dict(_BASE, **c)
    x, wr, br = _inputs(c, seed)
    x = x.double()
    logits = x @ wr.double().t()
    if br is not None:
        logits = logits + br.double()
    gates, picked, probs, rows = _gating(c, logits)
    act = {"silu": torch.nn.functional.silu, "relu": torch.relu,
           "gelu": lambda a: torch.nn.functional.gelu(a, approximate="tanh")}[c["act"]]
    lsh = c["lsh"]
    out, shared = torch.zeros_like(x), torch.zeros_like(x)
    for e in range(c["E"]):
        if e < lsh:
            t, g = torch.arange(c["T"], device=x.device), None
        else:
            t = picked[:, e - lsh].nonzero()[:, 0]
            g = gates[t, e - lsh][:, None]
        if t.numel() == 0:
            continue
        ws, ss, bs = _expert(c, seed, e)
        w = [m.double() if s is None else m.to(torch.float32).double() * s.double()[:, None] for m, s in zip(ws, ss)]
        a = x[t] @ w[0].t()
        if c["etype"] == "gated":
            y = (act(a) * (x[t] @ w[2].t())) @ w[1].t()
        else:
            y = act(a + bs[0].double()) @ w[1].t() + bs[1].double()
        if g is None:
            shared += y / lsh
        else:
            out.index_add_(0, t, g * y)
    if lsh:
        out = 0.5 * shared + 0.5 * out
    if c["entry"] == "decode":
        return [out]
    loss = _loss(c, logits, picked, probs, rows) if c["training"] else torch.zeros((), dtype=torch.float64)
    if c["entry"] == "host":
        return [out.t().cpu().numpy(), float(loss)]
    return [out, loss.reshape(1)]
