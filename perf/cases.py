"""The calls that users of the MoE block make, as timed cases.

A layer's weights are generated on the device by the block's counter-based
generator (moe_layer_generate); `exact` generates the same weights in torch
and computes the block in 64 bits.  The activations and the SwiGLU output are
rounded to Q8_0 there as the block defines it (d = fp16(amax / 127),
q = rint(x * (127 / amax)), both in f32): that rounding is part of the result.

Magnitudes: nibbles uniform over the 16 codes and E8M0 exponents in
[116, 121) give weights of about 0.01 (gate and up sums of about 1);
activations are normal with a few larger channels, rounded to bf16, as a
transformer's normalised hidden states are.
"""
import importlib
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llama-sandbox_amd"))
mb = importlib.import_module("moe_block")
wl = importlib.import_module("workloads")

E_LO, E_SPAN = 116, 5
DEV = "cuda:0"
SOFTMAX, SIGMOID, SQRT_SOFTPLUS = wl.ROUTE_SOFTMAX, wl.ROUTE_SIGMOID, wl.ROUTE_SQRT_SOFTPLUS

# entry: forward (device tensors, ids and weights given), route (router logits
# given: routing and block in one call), graph (one captured graph of `layers`
# layers), host (host arrays in and out, the ggml backend's per-call boundary)
_BASE = {"entry": "forward", "T": 1, "zipf": False, "per_slot": False, "layers": 1}
_SMALL = {"H": 2048, "F": 768, "E": 32, "k": 4, "shared": False, "mode": SOFTMAX, "scale": 1.0, "clamp": 0.0}
_V3 = {"H": 7168, "F": 2048, "E": 256, "k": 8, "shared": True, "mode": SIGMOID, "scale": 1.0, "clamp": 0.0}
_V4P = {"H": 7168, "F": 3072, "E": 384, "k": 6, "shared": True, "mode": SQRT_SOFTPLUS, "scale": 2.5, "clamp": 10.0}
_MID = {"H": 5120, "F": 1536, "E": 160, "k": 6, "shared": True, "mode": SOFTMAX, "scale": 1.0, "clamp": 0.0}


def listed():
    def case(name, shape, **more):
        return {"name": name, **_BASE, **shape, **more}

    return [
        # the smallest call: one token through a small layer, routed in the same call
        case("decode_small", _SMALL, entry="route"),
        # one token through four consecutive layers, as a decode loop replays them
        case("decode_stack", _V3, entry="graph", layers=4),
        # one token across the host boundary, as llama.cpp's scheduler calls the backend: per-slot rows back
        case("decode_host", _V3, entry="host", per_slot=True),
        # small-batch decode: a few concurrent sequences
        case("batch_4", _V3, T=4, zipf=True),
        case("batch_16", _V3, T=16, zipf=True),
        case("batch_64", _V3, T=64, zipf=True),
        # a ragged batch through the backend's per-slot output on a mid-sized layer
        case("batch_37_per_slot", _MID, T=37, per_slot=True),
        # prompt chunks: balanced routing, and skewed routing with hot experts
        case("prefill_512", _V3, T=512),
        case("prefill_512_zipf", _V3, T=512, zipf=True, entry="route"),
        # the widest experts the block is used with, clamped SwiGLU, an odd chunk
        case("prefill_509_wide", _V4P, T=509, zipf=True),
        # a prompt chunk through a mid-sized layer
        case("prefill_300_mid", _MID, T=300, entry="route"),
        # the largest call: a long prompt chunk
        case("prefill_2048", _V3, T=2048),
    ]


def draw(rng):
    H, F = 128 * rng.randint(8, 56), 128 * rng.randint(4, 24)
    k = rng.randint(1, 8)
    most = int(6.1e9 / (3 * H * F / 32 * 17)) - 1  # a layer no larger than the listed ones
    E = max(2 * k, min(most, int(round(8 * 48 ** rng.random()))))
    T = int(round(1024 ** rng.random()))
    return {
        **_BASE, "H": H, "F": F, "E": E, "k": k, "T": T, "shared": rng.random() < 0.5,
        "mode": rng.choice([SOFTMAX, SIGMOID, SQRT_SOFTPLUS]), "scale": rng.choice([1.0, 2.5]),
        "clamp": rng.choice([0.0, 0.0, 10.0]), "zipf": rng.random() < 0.5, "per_slot": rng.random() < 0.25,
        "entry": rng.choice(["forward", "forward", "route", "graph"] + (["host"] if T <= 64 else [])),
    }


def _shape(case):
    return wl.LayerShape(hidden=case["H"], ffn=case["F"], n_expert=case["E"], n_used=case["k"],
                         has_shared=case["shared"], route_mode=case["mode"], scale=case["scale"],
                         clamp=case["clamp"], bf16_act=True)


def _logits(case, seed, i):
    """Router logits [T, E] of layer i: N(0, 1), with a per-expert Zipf(1.1) bias where the case is skewed."""
    rng = np.random.default_rng([int(seed), i, 1])
    lg = rng.standard_normal((case["T"], case["E"]), dtype=np.float32)
    if case["zipf"]:
        p = (np.arange(case["E"]) + 1.0) ** -1.1
        lg = lg + np.log(p / p.sum())[rng.permutation(case["E"])].astype(np.float32)
    return torch.from_numpy(np.ascontiguousarray(lg, dtype=np.float32))


def _route64(case, logits):
    """ids [T, k] and weights [T, k] (f64) of the router."""
    z = logits.double()
    if case["mode"] == SOFTMAX:
        s = torch.softmax(z, 1)
    elif case["mode"] == SIGMOID:
        s = torch.sigmoid(z)
    else:
        s = torch.sqrt(torch.where(z > 20, z, torch.log1p(torch.exp(z))))
    order = torch.sort(s, dim=1, descending=True, stable=True).indices[:, :case["k"]]
    w = torch.gather(s, 1, order)
    w = w / torch.clamp(w.sum(1, keepdim=True), min=2.0 ** -14)
    return order.to(torch.int32), w * case["scale"]


def _x(case, seed, i):
    g = torch.Generator(device=DEV).manual_seed(1000 * int(seed) + i)
    gain = torch.exp(0.5 * torch.randn(case["H"], generator=g, device=DEV))
    x = torch.randn(case["T"], case["H"], generator=g, device=DEV) * gain
    return x.to(torch.bfloat16).float()


def prepare(case, seed):
    shape, T, H, n = _shape(case), case["T"], case["H"], case["layers"]
    blk = mb.MoeBlock(0)
    blk.reserve(shape, T)
    for i in range(n):
        blk.generate_layer(i, shape, int(seed) + 1, E_LO, E_SPAN)
    out_shape = (T, case["k"], H) if case["per_slot"] else (T, H)
    s = {"case": case, "blk": blk, "flags": mb.MOE_FWD_PER_SLOT if case["per_slot"] else 0, "x": [], "ids": [],
         "wts": [], "logits": [], "out": []}
    for i in range(n):
        lg = _logits(case, seed, i)
        ids, wts = _route64(case, lg)
        s["x"].append(_x(case, seed, i))
        s["ids"].append(ids.to(DEV))
        s["wts"].append(wts.float().to(DEV))
        s["logits"].append(lg.to(DEV))
        s["out"].append(torch.empty(out_shape, dtype=torch.float32, device=DEV))
    if case["entry"] == "graph":
        torch.cuda.synchronize()
        s["graph"] = blk.graph_capture(list(range(n)), s["x"], s["ids"], s["wts"], s["out"], s["flags"])
    if case["entry"] == "host":
        s["host"] = [s[a][0].cpu().numpy() for a in ("x", "ids", "wts")]
    return s


def run(state):
    case, blk, flags = state["case"], state["blk"], state["flags"]
    x, ids, wts, out = (state[a] for a in ("x", "ids", "wts", "out"))
    if case["entry"] == "graph":
        state["graph"].launch()
        return {"out": out}
    if case["entry"] == "host":
        return {"out": blk.forward_host(0, *state["host"], flags=flags)}
    if case["entry"] == "route":
        blk.route_forward(0, x[0], state["logits"][0], ids[0], wts[0], out[0], mode=case["mode"], norm=True,
                          scale=case["scale"], flags=flags)
        return {"out": out[0], "ids": ids[0], "wts": wts[0]}
    blk.forward(0, x[0], ids[0], wts[0], out[0], flags)
    return {"out": out[0]}


def work(case):
    """The touched experts' weights, the activations in and the rows out, once each."""
    shape, T, b, f = _shape(case), case["T"], 0, 0
    sh = case["shared"] and not case["per_slot"]
    for i in range(case["layers"]):
        lg = _logits(case, 1, i)
        ids, _ = _route64(case, lg)
        b += (len(torch.unique(ids)) + int(sh)) * shape.expert_bytes
        b += 4 * T * case["H"] * (1 + (case["k"] if case["per_slot"] else 1)) + 8 * ids.numel()
        b += 4 * lg.numel() if case["entry"] == "route" else 0
        f += 6 * T * (case["k"] + int(sh)) * case["F"] * case["H"]
    return {"bytes": b, "flops": f}


def tolerance(case):
    # f32 sums of exact block products in another order move a SwiGLU value by
    # about 1e-7 of its size.  Where that crosses a Q8_0 rounding boundary one
    # code changes by 1 of at most 127, about 0.02 of a value's standard
    # deviation, in a sum over F values of each slot: 1e-4 of a token's row on
    # these layers (measured 3e-5 to 9e-5 over the listed cases), more on a
    # narrow layer with one slot
    terms = case["F"] * (1 if case["per_slot"] else case["k"] + int(case["shared"]))
    rel = max(4e-4, 0.04 / math.sqrt(terms))
    return {"rel": rel, "max": 12 * rel}


# ---- the block in 64 bits ------------------------------------------------------------

_MASK = (1 << 64) - 1


def _mix(z):
    """SplitMix64's output function on a Python int (the generator's key derivation)."""
    z = (z + 0x9E3779B97F4A7C15) & _MASK
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK
    return z ^ (z >> 31)


def _i64(v):
    v &= _MASK
    return v - (1 << 64) if v >> 63 else v


def _srl(z, n):
    return (z >> n) & ((1 << (64 - n)) - 1)


def _mix_t(z):
    z = z + _i64(0x9E3779B97F4A7C15)
    z = (z ^ _srl(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ _srl(z, 27)) * _i64(0x94D049BB133111EB)
    return z ^ _srl(z, 31)


def _matrix(seed, layer, tensor, expert, rows, K):
    """[rows, K] f64 weights of one generated expert matrix (tensor 0-2 gate, up, down; 3-5 the shared expert's)."""
    key = _mix((seed & _MASK) ^ _mix((layer << 40) ^ (tensor << 32) ^ expert))
    i = torch.arange(rows * (K // 32), dtype=torch.int64, device=DEV)
    a, b = _mix_t(2 * i + _i64(key + 1)), _mix_t(2 * i + _i64(key + 2))
    c = _mix_t(~i ^ _i64(key))
    e = E_LO + _srl(_srl(c, 32) * E_SPAN, 32)
    lut = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12], dtype=torch.float64, device=DEV)
    sh = torch.arange(0, 64, 8, dtype=torch.int64, device=DEV)
    w = torch.empty((i.numel(), 32), dtype=torch.float64, device=DEV)
    for half, v in ((0, a), (8, b)):  # byte j: element j (low nibble) and j + 16 (high nibble)
        byte = (v[:, None] >> sh) & 255
        w[:, half:half + 8] = lut[byte & 15]
        w[:, 16 + half:24 + half] = lut[byte >> 4]
    w *= torch.exp2((e - 128).double())[:, None]
    return w.view(rows, K)


def _q8(x):
    """f32 [N, K] -> its Q8_0 value in f64."""
    b = x.float().view(x.shape[0], -1, 32)
    amax = b.abs().amax(2, keepdim=True)
    m = torch.full_like(amax, 127.0)  # tensor by tensor: a scalar's division may go by the reciprocal
    inv = torch.where(amax > 0, m / amax, torch.zeros_like(amax))
    d = (amax / m).half().double()
    return (torch.round(b * inv).double() * d).view(x.shape)


def _expert(case, seed, layer, x, tensors, expert):
    H, F, L = case["H"], case["F"], case["clamp"]
    g = x @ _matrix(seed, layer, tensors, expert, F, H).T
    u = x @ _matrix(seed, layer, tensors + 1, expert, F, H).T
    if L > 1e-6:
        u, g = torch.clamp(u, -L, L), torch.clamp(g, max=L)
    h = _q8(g * torch.sigmoid(g) * u)
    return h @ _matrix(seed, layer, tensors + 2, expert, H, F).T


def exact(case, seed):
    outs, seed_w, k, H = [], int(seed) + 1, case["k"], case["H"]
    for i in range(case["layers"]):
        ids, wts = _route64(case, _logits(case, seed, i))
        given = wts.float().double() if case["entry"] != "route" else wts
        flat, w = ids.reshape(-1).to(DEV), given.reshape(-1).to(DEV)
        x = _q8(_x(case, seed, i))
        y = torch.zeros((case["T"] * k, H), dtype=torch.float64, device=DEV)
        for e in torch.unique(ids).tolist():
            p = torch.nonzero(flat == e).view(-1)
            y[p] = _expert(case, seed_w, i, x[p // k], 0, e) * w[p, None]
        y = y.view(case["T"], k, H)
        if not case["per_slot"]:
            y = y.sum(1)
            if case["shared"]:
                y = y + _expert(case, seed_w, i, x, 3, 0)
        outs.append(y)
    if case["entry"] == "graph":
        return {"out": outs}
    if case["entry"] == "route":
        return {"out": outs[0], "ids": ids, "wts": wts}
    return {"out": outs[0]}
