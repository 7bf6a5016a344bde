"""The calls whose speed this repository is held to: what a user of the EXL3
trellis quantizer has it do, through `quantize.py`'s public functions.

Twelve listed cases and `draw` cover the encoder at every bit width from one
tile to a whole layer, single Viterbi runs, the BlockLDLQ sweep from a small
ragged weight to a 17408x5120 down projection, whole `quantize_linear` and
mixed-width group calls on host weights, the block-128 incoherence transforms,
and the trellis format both ways.  Shapes are the layer shapes of this
repository's own workloads (128, 4096, 5120, 6144/1024, 17408) or generic ones.

Every result here is a sequence of whole numbers (states, packed trellis), a
value looked up from the codebook, or an fp32 sum in a fixed order, and the
encoder is specified bit for bit, so the tolerance is exact wherever the
inputs of a case fix the bits.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "exl3xpu-mixedk_amd", "quantize")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import quantize as xq  # noqa: E402

CODES = ("exl3_mul1", "exl3_mcg", "exl3_3inst", "qtip_1mad")
STATES = 1 << 16
STEPS = 256


def listed():
    """The twelve cases."""
    return [
        # One 128x128 weight's tiles at the lowest width: the smallest call a
        # harness makes (a smoke test, a block of a narrow layer).
        {"name": "encode_64_k2", "kind": "encode", "tiles": 64, "K": 2, "pivot": 128,
         "margin": 0, "code": "exl3_mul1"},
        # A ragged batch with a truncated first pass and a seeded pivot, as the
        # `quantize()` harness entry runs it.
        {"name": "encode_1003_k5", "kind": "encode", "tiles": 1003, "K": 5, "pivot": 147,
         "margin": 16, "code": "exl3_mcg"},
        # Every tile of a 4096x4096 layer without feedback, at the width the
        # headline benchmark uses.
        {"name": "encode_65536_k4", "kind": "encode", "tiles": 65536, "K": 4, "pivot": 128,
         "margin": 0, "code": "exl3_mul1"},
        # A single pinned Viterbi run over shorter sequences.
        {"name": "viterbi_2001x200_k6", "kind": "viterbi", "tiles": 2001, "steps": 200, "K": 6,
         "pinned": True, "code": "exl3_3inst"},
        # The BlockLDLQ sweep of a small ragged weight: few column chains, so
        # the time of one tile sets the pace.
        {"name": "sweep_1040x2064_k7", "kind": "sweep", "k": 1040, "n": 2064, "K": 7,
         "margin": 0, "code": "exl3_mul1"},
        # The sweep of a square attention projection at 3 bits.
        {"name": "sweep_5120x5120_k3", "kind": "sweep", "k": 5120, "n": 5120, "K": 3,
         "margin": 0, "code": "exl3_mul1"},
        # The sweep of a down projection, the longest feedback and the largest
        # weight of the workloads.
        {"name": "sweep_17408x5120_k4", "kind": "sweep", "k": 17408, "n": 5120, "K": 4,
         "margin": 0, "code": "exl3_mul1"},
        # A whole quantize_linear call on a host fp16 weight and its Gram.
        {"name": "linear_4096x4096_k4", "kind": "linear", "k": 4096, "ns": "4096", "Ks": "4",
         "channel_scales": False},
        # q/k/v of one layer at their own widths in one call, with EXL3's
        # per-channel scales: the mixed-K path.
        {"name": "group_5120_k5_k7", "kind": "linear", "k": 5120, "ns": "6144 1024 1024",
         "Ks": "5 7 7", "channel_scales": True},
        # The incoherence transform of a down projection and its inverse.
        {"name": "incoherence_17408x5120", "kind": "incoherence", "k": 17408, "n": 5120},
        # Rebuilding a layer's weight from its trellis when a model is loaded.
        {"name": "decode_17408x5120_k4", "kind": "decode", "k": 17408, "n": 5120, "K": 4,
         "code": "exl3_mul1"},
        # The format's round trip that follows every encode: pack the states,
        # unpack them again, decode.
        {"name": "roundtrip_4096x4096_k3", "kind": "roundtrip", "k": 4096, "n": 4096, "K": 3,
         "code": "exl3_mul1"},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], uniform over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["encode", "encode", "encode", "viterbi", "sweep", "sweep", "sweep",
                       "linear", "incoherence", "decode", "roundtrip"])
    K = rng.randint(2, 7)
    code = rng.choice(CODES)
    margin = rng.choice([0, 0, 16])
    if kind == "encode":
        return {"kind": kind, "tiles": _log(rng, 1, 65536), "K": K,
                "pivot": rng.choice([128, rng.randint(0, 255)]), "margin": margin, "code": code}
    if kind == "viterbi":
        return {"kind": kind, "tiles": _log(rng, 1, 16384), "steps": rng.randint(32, 256),
                "K": K, "pinned": rng.random() < 0.5, "code": code}
    if kind == "sweep":
        return {"kind": kind, "k": 16 * _log(rng, 4, 400), "n": 16 * _log(rng, 4, 400), "K": K,
                "margin": margin, "code": code}
    if kind == "linear":
        m = rng.choice([1, 1, 3])
        k = 128 * _log(rng, 2, 32)
        return {"kind": kind, "k": k,
                "ns": " ".join(str(128 * _log(rng, 1, 32 // m)) for _ in range(m)),
                "Ks": " ".join(str(rng.randint(2, 7)) for _ in range(m)),
                "channel_scales": rng.random() < 0.5}
    if kind == "incoherence":
        return {"kind": kind, "k": 128 * _log(rng, 1, 136), "n": 128 * _log(rng, 1, 40)}
    return {"kind": kind, "k": 16 * _log(rng, 1, 1088), "n": 16 * _log(rng, 1, 320), "K": K,
            "code": code}


# ------------------------------------------------------------------- inputs
def _ints(text):
    return [int(v) for v in str(text).split()]


def _gen(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(int(seed))


def _targets(steps, n, seed):
    """Targets of incoherent weights at the codebook's scale: unit-variance
    Gaussians, [steps, n] as quantize_seq_tailbite takes them."""
    return torch.randn(steps, n, generator=_gen(seed), device="cuda")


def _factor(k, seed):
    """A block-LDL factor of the kind the rotated, damped Gram of correlated
    activations gives: unit 16x16 diagonal blocks, small dense entries below
    them.  (Column norms about 0.3, as AR(1) activations give.)"""
    L = torch.randn(k, k, generator=_gen(seed + 1), device="cuda").mul_(0.3 / math.sqrt(k))
    b = torch.arange(k, device="cuda") // 16
    L.masked_fill_(b[:, None] <= b[None, :], 0.0)
    L.diagonal().fill_(1.0)
    return L


def _gram(k, seed):
    """Input Gram of 2k samples with correlation 0.5 between neighbouring
    channels (a moving average of white noise), on the host as a calibration
    run leaves it.  Every product of the sums is exact (whole numbers), so
    the Gram does not depend on the order of the reduction."""
    z = torch.randint(-8, 9, (2 * k, k + 1), generator=_gen(seed + 2), device="cuda")
    x = (z[:, 1:] + z[:, :-1]).double()
    return ((x.t() @ x) / (2 * k * 48)).float().cpu()


def prepare(case, seed):
    """What a user's program holds before the call."""
    kind = case["kind"]
    s = {"case": case}
    if "code" in case:
        s["lut"] = xq.get_lut(case["code"])
    if kind == "encode":
        s["X"] = _targets(STEPS, case["tiles"], seed)
    elif kind == "viterbi":
        s["X"] = _targets(case["steps"], case["tiles"], seed)
        s["overlap"] = torch.randint(0, 1 << (16 - case["K"]), (case["tiles"],),
                                     generator=_gen(seed + 3), device="cuda") \
            if case["pinned"] else None
    elif kind == "sweep":
        s["W"] = torch.randn(case["k"], case["n"], generator=_gen(seed), device="cuda")
        s["L"] = _factor(case["k"], seed)
    elif kind == "linear":
        s["Ws"] = [(0.02 * torch.randn(n, case["k"], generator=_gen(seed + 10 + i),
                                       device="cuda")).half().cpu()
                   for i, n in enumerate(_ints(case["ns"]))]
        s["H"] = _gram(case["k"], seed)
    elif kind == "incoherence":
        s["W"] = 0.02 * torch.randn(case["k"], case["n"], generator=_gen(seed), device="cuda")
        s["suh"] = xq.sign_vec(case["k"], seed + 4, "cuda").half()
        s["svh"] = xq.sign_vec(case["n"], seed + 5, "cuda").half()
        s["h"] = xq.hadamard128("cuda")
    else:
        tk, tn = case["k"] // 16, case["n"] // 16
        bits = torch.randint(-32768, 32768, (tk, tn, 16 * case["K"]), generator=_gen(seed),
                             device="cuda", dtype=torch.int16)
        if kind == "decode":
            s["trellis"] = bits
        else:
            s["states"] = xq.unpack_states(bits, case["K"]).view(-1, STEPS)
    return s


# --------------------------------------------------------------------- pass
def run(state):
    """One pass."""
    c = state["case"]
    kind = c["kind"]
    if kind == "encode":
        return xq.quantize_seq_tailbite(state["X"], state["lut"], c["K"], 16, pivot=c["pivot"],
                                        margin=c["margin"])
    if kind == "viterbi":
        return xq.viterbi(state["X"], state["lut"], c["K"], 16, overlap=state["overlap"])
    if kind == "sweep":
        hat, states = xq.ldlq_viterbi(state["W"], state["L"], state["lut"], c["K"], 16,
                                      margin=c["margin"])
        return {"W_hat": hat, "states": states, "trellis": xq.ldlq_viterbi.last_trellis}
    if kind == "linear":
        Ks = _ints(c["Ks"])
        if len(Ks) == 1:
            res = [xq.quantize_linear(state["Ws"][0], state["H"], K=Ks[0], device="cuda",
                                      channel_scales=c["channel_scales"])]
        else:
            res = xq.quantize_linear_group(state["Ws"], state["H"], K=Ks, device="cuda",
                                           channel_scales=c["channel_scales"])
        return [{name: r[name] for name in ("W_hat", "trellis", "suh", "svh", "Wscale")}
                for r in res]
    if kind == "incoherence":
        inner = xq.to_inner(state["W"], state["suh"], state["svh"], state["h"])
        return {"inner": inner,
                "orig": xq.from_inner(inner, state["suh"], state["svh"], state["h"])}
    if kind == "decode":
        return xq.decode_trellis(state["trellis"], state["lut"], c["K"], c["k"], c["n"])
    packed = xq.pack_states(state["states"], c["K"])
    packed = packed.view(c["k"] // 16, c["n"] // 16, -1)
    return {"trellis": packed, "states": xq.unpack_states(packed, c["K"]),
            "W": xq.decode_trellis(packed, state["lut"], c["K"], c["k"], c["n"])}


# --------------------------------------------------------------------- work
def work(case):
    """Bytes each input read and each output written once, and operations:
    a subtraction, a product, a sum and a comparison per state and step."""
    kind = case["kind"]
    if kind in ("encode", "viterbi"):
        n, t = case["tiles"], case.get("steps", STEPS)
        steps = t
        if kind == "encode":
            m, p = case["margin"], case["pivot"]
            steps += p + m if m and p + m < STEPS else STEPS
        return {"bytes": n * t * (4 + 8), "flops": 4.0 * STATES * steps * n}
    k = case["k"]
    if kind in ("sweep", "linear"):
        by = 4.0 * k * k
        fl = 0.0
        ns = _ints(case.get("ns", case.get("n")))
        for n, K in zip(ns, _ints(case.get("Ks", case.get("K")))):
            m = case.get("margin", 0)
            steps = STEPS + (128 + m if m else STEPS)
            by += (8 + 8) * k * n if kind == "sweep" else (2 + 4) * k * n
            by += k * n * K / 8
            fl += 4.0 * STATES * steps * (k * n / 256) + float(k) * k * n
        if kind == "linear":
            fl += k ** 3 / 3.0 + 2 * 2 * 128.0 * k * k + sum(
                2 * 4 * 128.0 * k * n for n in ns)
        return {"bytes": by, "flops": fl}
    n = case["n"]
    if kind == "incoherence":
        return {"bytes": 4.0 * k * n * 3, "flops": 4 * 2 * 128.0 * k * n}
    K = case["K"]
    if kind == "decode":
        return {"bytes": k * n * (K / 8 + 4.0), "flops": 1.0 * k * n}
    return {"bytes": k * n * (8.0 + K / 8 + 8.0 + 4.0), "flops": 1.0 * k * n}


def tolerance(case):
    """Whole numbers, looked-up values and fixed-order sums: exact."""
    return "exact"


# -------------------------------------------------------------------- exact
def _perm():
    """Sequence element t -> row-major position in the 16x16 tile."""
    t = np.arange(256)
    g, e = t // 8, t % 8
    return ((g % 4) * 2 + (e % 2) + 8 * ((e // 2) % 2)) * 16 + g // 4 + 8 * (e // 4)


def _codebook(code):
    """The codebook over all states, from its definition."""
    s = np.arange(STATES, dtype=np.uint64)

    def half(bits):
        return np.asarray(bits).astype(np.uint16).view(np.float16).astype(np.float64)

    def bytesum(h):
        return sum(((h >> sh) & 0xFF) for sh in (0, 8, 16, 24)).astype(np.float64)

    if code == "exl3_mul1":
        v = (1024 + bytesum((s * 0x83DCD12D) & 0xFFFFFFFF)) * half([0x1EEE]) + half([0xC931])
        return v.astype(np.float16).astype(np.float64)
    if code == "qtip_1mad":
        h = (s * 34038481 + 76625530) & 0xFFFFFFFF
        return ((bytesum(h) - 510.0) / 147.800537109375).astype(np.float32).astype(np.float64)
    h = s * 89226354 + 64248484 if code == "exl3_3inst" else s * 0xCBAC1FED
    h = ((h & 0xFFFFFFFF) & 0x8FFF8FFF) ^ 0x3B603B60
    return (half(h & 0xFFFF) + half(h >> 16)).astype(np.float16).astype(np.float64)


def _unpacked(trellis, K):
    """States [.., 256] of packed tiles: the 16-bit circular window that ends
    with symbol t's bits."""
    w = trellis.reshape(-1, 8 * K, 2).to(torch.int64) & 0xFFFF
    words = w[..., 0] | (w[..., 1] << 16)
    sh = torch.arange(31, -1, -1, device=trellis.device)
    out = torch.empty(words.shape[0], STEPS, dtype=torch.int64, device=trellis.device)
    idx = (torch.arange(STEPS, device=trellis.device)[:, None] * K + K - 16
           + torch.arange(16, device=trellis.device)) % (STEPS * K)
    wt = 1 << torch.arange(15, -1, -1, device=trellis.device)
    for a in range(0, words.shape[0], 8192):
        bits = ((words[a:a + 8192, :, None] >> sh) & 1).reshape(-1, STEPS * K)
        out[a:a + 8192] = (bits[:, idx] * wt).sum(-1)
    return out


def _decoded(states, code, k, n):
    perm = torch.from_numpy(_perm()).to(states.device)
    tile = torch.empty(states.shape, dtype=torch.float64, device=states.device)
    tile[:, perm] = torch.from_numpy(_codebook(code)).to(states.device)[states]
    return tile.view(k // 16, n // 16, 16, 16).permute(0, 2, 1, 3).reshape(k, n)


def exact(case, seed):
    """What run returns, in 64 bits by plain torch; None for encodes, whose
    results are the whole numbers that the fp32 recursion itself defines."""
    kind = case["kind"]
    if kind in ("encode", "viterbi", "sweep", "linear"):
        return None
    s = prepare(case, seed)
    if kind == "incoherence":
        h = torch.ones(1, 1, dtype=torch.float64, device="cuda")
        while h.shape[0] < 128:
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        h = h / math.sqrt(128.0)
        k, n = case["k"], case["n"]
        su, sv = s["suh"].double()[:, None], s["svh"].double()[None, :]

        def both(w):
            w = torch.matmul(h.expand(k // 128, 128, 128).contiguous(), w.view(k // 128, 128, n))
            return (w.view(-1, 128) @ h).view(k, n)

        inner = both(s["W"].double() / su / sv)
        return {"inner": inner, "orig": both(inner) * su * sv}
    if kind == "decode":
        return _decoded(_unpacked(s["trellis"], case["K"]), case["code"], case["k"], case["n"])
    return {"trellis": None, "states": None,
            "W": _decoded(s["states"], case["code"], case["k"], case["n"])}
