"""Timed cases of the engine's per-layer work on one GPU, at the shapes of the model this library serves (64 layers of
width 5120: 48 gated-delta-net layers, 16 attention layers, FFN 17408, vocabulary 248320).

Decode cases (1 to 4 tokens) replay a HIP graph of one layer's launches, as the engine does for every decode step; the
graph is recorded once per state in prepare(). Prefill cases (a batch of up to 4099 rows) call the launchers one after
another. Weights are random GGUF blocks whose super-block scales give weights of about 0.02 rms, activations are
normal with log-normal channel scales, gates decay as trained ones do (g <= 0).

exact() restates every op in float64 with plain torch. Where the op itself rounds (the int8 quantization of the
activations, the truncating integer scale rules of four weight formats, the float32 rotary angle) it rounds at the same
place, since that is what the op computes.
"""
import importlib.util
import math
import os
import re
import sys

import torch

E, FF, NQH, NKVH, KH, HV, D = 5120, 17408, 24, 4, 16, 48, 128
C = 2 * KH * D + HV * D  # conv channels: q heads, k heads, v heads
VOCAB, EPS = 248320, 1e-6
THETA = float(torch.tensor(1e7, dtype=torch.float32) ** torch.tensor(-2.0 / 64, dtype=torch.float32))
DEV = "cuda:0"
PKG = os.path.join(os.getcwd(), "qwen27-engine_amd")

# GGUF weight formats: ggml type id, bytes per 256-weight block, fp16 scale fields, rms of a random block's weights in
# units of the scale
TYPES = {"q2_k": (10, 84, (80, 82), 12.0), "q4_k": (12, 144, (0, 2), 250.0), "q6_k": (14, 210, (208,), 1367.0),
         "iq2_xxs": (16, 66, (0,), 57.0), "iq2_xs": (17, 74, (0,), 57.0), "iq3_xxs": (18, 98, (0,), 130.0),
         "iq3_s": (21, 110, (0,), 150.0), "iq2_s": (22, 82, (0,), 57.0), "iq4_xs": (23, 136, (0,), 1220.0),
         "iq1_m": (29, 56, (), 7.5)}
MIN_RATIO = {"q2_k": 1.5, "q4_k": 7.5}  # dmin / d of the two formats with a minimum
EMBED_BYTES = {"q4_k": (144, 256), "q6_k": (210, 256), "q8_0": (34, 32), "iq2_s": (82, 256)}


def _q27():
    name = "qwen27_engine_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(PKG, "__init__.py"), submodule_search_locations=[PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name].ops


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one token's residual add + norm + quantization, launched by itself (128 of them per step)
        {"name": "residual_norm_t1", "kind": "residual_norm", "T": 1},
        # plain decoding: a gated-delta-net layer's mixer for one token, Q4_K projections
        {"name": "gdn_layer_t1_q4k", "kind": "gdn_layer", "T": 1, "type": "q4_k"},
        # verification of a 4-token draft: an attention layer's projections and Q/K/V preparation at 150k context
        {"name": "attn_layer_t4_q4k", "kind": "attn_layer", "T": 4, "type": "q4_k"},
        # the feed-forward block, two thirds of the weights: plain decoding and verification, 3-bit weights
        {"name": "ffn_t1_iq3s", "kind": "ffn", "T": 1, "type": "iq3_s", "down": "iq3_s"},
        {"name": "ffn_t4_iq3s", "kind": "ffn", "T": 4, "type": "iq3_s", "down": "iq3_s"},
        # the same with an odd number of tokens and the mixed low-bit formats of the smallest files
        {"name": "ffn_t3_iq2xs", "kind": "ffn", "T": 3, "type": "iq2_xs", "down": "iq4_xs"},
        # the output head: the largest matrix of a decode step
        {"name": "head_t4_q6k", "kind": "proj", "T": 4, "type": "q6_k", "N": VOCAB, "K": E},
        # token embedding of a prompt batch and the first norm
        {"name": "embed_2052_iq2s", "kind": "embed", "T": 2052, "type": "iq2_s"},
        # prompt batches: the gated-delta-net mixer (full batch, and the ragged rest of a prompt), the element-wise part
        # of the FFN, and an attention layer's preparation for a 64 x 64 image grid after 3 text tokens
        {"name": "gdn_prefill_2048", "kind": "gdn_prefill", "T": 2048},
        {"name": "gdn_prefill_333", "kind": "gdn_prefill", "T": 333},
        {"name": "ffn_prefill_2048", "kind": "ffn_prefill", "T": 2048},
        {"name": "attn_prefill_4099", "kind": "attn_prefill", "T": 4099, "image": True},
    ]


def draw(rng):
    kind = rng.choice(["residual_norm", "gdn_layer", "attn_layer", "ffn", "ffn", "proj", "proj", "embed", "gdn_prefill",
                       "gdn_prefill", "ffn_prefill", "attn_prefill"])
    types = sorted(TYPES)

    def rows(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    case = {"kind": kind, "T": rng.randint(1, 4)}
    if kind == "residual_norm":
        case["T"] = rows(1, 64)
    elif kind in ("gdn_layer", "attn_layer"):
        case["type"] = rng.choice(types)
    elif kind == "ffn":
        case["type"], case["down"] = rng.choice(types), rng.choice(types)
    elif kind == "proj":
        case["type"], case["N"], case["K"] = rng.choice(types), 8 * rows(32, 4096), 256 * rows(2, 80)
    elif kind == "embed":
        case["T"], case["type"] = rows(5, 2052), rng.choice(sorted(EMBED_BYTES))
    elif kind == "gdn_prefill":
        case["T"] = rows(5, 2048)
    elif kind == "ffn_prefill":
        case["T"] = rows(5, 2048)
    else:
        case["T"], case["image"] = rows(5, 4099), rng.random() < 0.3
    return case


# ---------------------------------------------------------------- inputs
class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed) * 2 + 1)

    def n(self, *shape, std=1.0, mean=0.0):
        return torch.randn(shape, device=DEV, generator=self.g) * std + mean

    def u(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return torch.rand(shape, device=DEV, generator=self.g, dtype=dtype) * (hi - lo) + lo

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=self.g)


def _put_half(blocks, off, h):
    blocks[:, off:off + 2] = h.to(torch.float16).view(torch.uint8).view(-1, 2)


def _weights(r, type_, N, K, rms=0.02):
    """N raw GGUF rows of K weights, uint8 [N * K / 256][block bytes]."""
    _, bb, offs, unit = TYPES[type_]
    B = r.bytes(N * (K // 256), bb)
    d = (rms / unit) * torch.exp2(r.u(B.shape[0], lo=-0.5, hi=0.5))
    if offs:
        _put_half(B, offs[0], d)
    if len(offs) > 1:
        _put_half(B, offs[1], d * MIN_RATIO[type_])
    if type_ == "iq1_m":  # its fp16 scale is the four top nibbles of the scale words
        h = d.to(torch.float16).view(torch.int16).to(torch.int32) & 0xFFFF
        for k in range(4):
            B[:, 49 + 2 * k] = (B[:, 49 + 2 * k] & 0x0F) | (((h >> (4 * k)) & 0xF) << 4).to(torch.uint8)
    return B


def _rows(r, T, n):
    """Residual-stream rows: normal values, log-normal channel scales."""
    return (r.n(T, n) * torch.exp(r.n(n, std=0.5))).reshape(-1)


def _gates(r):
    return {"ssm_a": -torch.exp(r.n(HV, std=0.7, mean=-1.0)), "dt_bias": r.n(HV)}


def _rope3(T):
    """(t, h, w) positions of 3 text tokens followed by an image of 64 columns."""
    rows = [(p, p, p) for p in range(min(3, T))] + [(3, 3 + i // 64, 3 + i % 64) for i in range(max(0, T - 3))]
    return torch.tensor(rows, dtype=torch.int32, device=DEV).reshape(-1)


def _inputs(case, seed):
    """Everything a pass reads, from the seed alone ("w_*": raw GGUF rows)."""
    r, T, kind = _Rand(seed), case["T"], case["kind"]
    i32 = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)  # noqa: E731
    s = {}
    if kind in ("residual_norm", "gdn_layer", "attn_layer", "ffn", "ffn_prefill"):
        s["x"], s["partial"], s["norm_w"] = _rows(r, T, E), r.n(T * E), r.n(E, std=0.1, mean=1.0)
    if kind == "ffn":
        s["w_gate"], s["w_up"] = _weights(r, case["type"], FF, E), _weights(r, case["type"], FF, E)
        s["w_down"] = _weights(r, case["down"], E, FF)
    elif kind == "gdn_layer":
        s["w_qkv"], s["w_z"] = _weights(r, case["type"], C, E), _weights(r, case["type"], HV * D, E)
        s["w_out"] = _weights(r, case["type"], E, HV * D)
        s["wa"], s["wb"] = (r.n(HV * E, std=0.02).to(torch.bfloat16) for _ in range(2))
        s["out_norm"] = r.n(D, std=0.1, mean=1.0)
    elif kind == "attn_layer":
        s["w_q"], s["w_k"] = _weights(r, case["type"], NQH * 512, E), _weights(r, case["type"], NKVH * 256, E)
        s["w_v"], s["w_o"] = _weights(r, case["type"], NKVH * 256, E), _weights(r, case["type"], E, NQH * 256)
        s["attn_out"] = r.n(T * NQH * 256)
        s["pos0"], s["n_ctx"] = i32(150000), 180224
    elif kind == "proj":
        s["w"] = _weights(r, case["type"], case["N"], case["K"])
        s["xq"] = torch.clamp(torch.round(r.n(T * case["K"], std=45.0)), -127, 127).to(torch.int8)
        s["xd"] = r.u(T * case["K"] // 32, lo=0.01, hi=0.04).to(torch.float16).float()
    elif kind == "embed":
        bb, bv = EMBED_BYTES[case["type"]]
        s["table"] = r.bytes(VOCAB * (E // bv), bb)
        unit = 74.0 if case["type"] == "q8_0" else TYPES[case["type"]][3]
        d = (0.02 / unit) * torch.exp2(r.u(s["table"].shape[0], lo=-0.5, hi=0.5))
        _put_half(s["table"], 208 if case["type"] == "q6_k" else 0, d)
        if case["type"] == "q4_k":
            _put_half(s["table"], 2, d * MIN_RATIO["q4_k"])
        rank = torch.arange(1, VOCAB + 1, dtype=torch.float64, device=DEV) ** -1.1  # token frequencies (Zipf)
        cdf = torch.cumsum(rank, 0)
        ranks = torch.clamp(torch.searchsorted(cdf / cdf[-1], r.u(T, dtype=torch.float64)), max=VOCAB - 1)
        s["ids"] = torch.randperm(VOCAB, device=DEV, generator=r.g)[ranks].to(torch.int32)
        s["norm_w"] = r.n(E, std=0.1, mean=1.0)
    elif kind == "gdn_prefill":
        s["qkv"], s["z"] = r.n(T * C), r.n(T * HV * D)
        s["a"], s["b"] = r.n(T * HV, std=2.0), r.n(T * HV, std=2.0)
        s["out_norm"] = r.n(D, std=0.1, mean=1.0)
    elif kind == "ffn_prefill":
        s["g"], s["u"] = r.n(T * FF, std=2.0), r.n(T * FF, std=2.0)
    elif kind == "attn_prefill":
        s["qg"], s["k"], s["v"] = r.n(T * NQH * 512), r.n(T * NKVH * 256), r.n(T * NKVH * 256)
        s["attn_out"] = r.n(T * NQH * 256)
        s["n_ctx"] = 16384
        s["pos0"] = i32(0 if case["image"] else 9001)
        s["rope3"] = _rope3(T) if case["image"] else None
    if kind in ("gdn_layer", "gdn_prefill"):
        s.update(_gates(r))
        s["conv_w"], s["planes"] = r.n(C * 4, std=0.5), r.n(4 * C * 3)
        s["states"] = r.n(4 * HV * D * D, std=0.1)
        s["plane"] = i32(T - 1 if kind == "gdn_layer" else 0)
    if kind in ("attn_layer", "attn_prefill"):
        s["q_norm"], s["k_norm"] = r.n(256, std=0.1, mean=1.0), r.n(256, std=0.1, mean=1.0)
    return s


# ---------------------------------------------------------------- a pass
def _buffers(case, s):
    T, kind = case["T"], case["kind"]
    z = lambda n, dt=torch.float32: torch.zeros(n, dtype=dt, device=DEV)  # noqa: E731

    def q8(name, n, xs):
        s[name + "q"], s[name + "d"] = z(n, torch.int8), z(n // 32)
        s[name + "s"] = z(n // 16) if xs else None

    if kind in ("residual_norm", "gdn_layer", "attn_layer", "ffn", "embed", "ffn_prefill"):
        q8("n", T * E, kind in ("embed", "ffn_prefill"))
        s["h"] = z(T * E) if kind in ("gdn_layer", "embed") else None
    if kind == "ffn":
        s["yg"], s["yu"], s["y"] = z(T * FF), z(T * FF), z(T * E)
        q8("m", T * FF, False)
    elif kind == "gdn_layer":
        s["qkv"], s["z"], s["a"], s["b"], s["y"] = z(T * C), z(T * HV * D), z(T * HV), z(T * HV), z(T * E)
    elif kind == "attn_layer":
        s["qg"], s["k"], s["v"], s["y"] = z(T * NQH * 512), z(T * NKVH * 256), z(T * NKVH * 256), z(T * E)
        q8("m", T * NQH * 256, False)
    elif kind == "proj":
        s["y"] = z(T * case["N"])
    elif kind == "embed":
        s["x"] = z(T * E)
    elif kind == "ffn_prefill":
        q8("m", T * FF, True)
    elif kind == "attn_prefill":
        q8("m", T * NQH * 256, True)
    if kind in ("gdn_layer", "gdn_prefill"):
        s["conv"], s["g"], s["beta"], s["o"] = z(T * C), z(T * HV), z(T * HV), z(T * HV * D)
        q8("m", T * HV * D, kind == "gdn_prefill")
    if kind in ("attn_layer", "attn_prefill"):
        s["qn"] = z(T * NQH * 256)
        nb = _q27().kv_cache_bytes(NKVH, s["n_ctx"], True)
        s["kc"], s["vc"] = z(nb, torch.uint8), z(nb, torch.uint8)


def _launch(case, s):
    """The launches of one pass, in the engine's order."""
    o, T, kind = _q27(), case["T"], case["kind"]
    scale = 1.0 / math.sqrt(D)
    q, k, v = (s["conv"], s["conv"][KH * D:], s["conv"][2 * KH * D:]) if "conv" in s else (None, None, None)
    if kind in ("residual_norm", "gdn_layer", "attn_layer", "ffn"):
        o.sum_norm_q8(s["x"], s["partial"], E, T, None, s["norm_w"], EPS, s["h"], s["nq"], s["nd"])
    if kind == "ffn":
        o.qgemv(s["gate"], s["nq"], s["nd"], s["yg"], T)
        o.qgemv(s["up"], s["nq"], s["nd"], s["yu"], T)
        o.swiglu_q8(s["yg"], s["yu"], s["mq"], s["md"], T * FF)
        o.qgemv(s["down"], s["mq"], s["md"], s["y"], T)
    elif kind == "gdn_layer":
        o.gemv_bf16_pair(s["wa"], s["wb"], s["h"], s["a"], s["b"], HV, E, T)
        o.qgemv(s["wqkv"], s["nq"], s["nd"], s["qkv"], T)
        o.qgemv(s["wz"], s["nq"], s["nd"], s["z"], T)
        o.gdn_conv_l2(s["qkv"], s["conv_w"], s["planes"], s["plane"], s["conv"], C, T, True, 2 * KH, EPS, s["a"], s["b"],
                      s["ssm_a"], s["dt_bias"], s["g"], s["beta"], HV)
        o.gdn_step(q, k, v, C, s["g"], s["beta"], s["states"], s["plane"], s["o"], HV, KH, T, scale, True)
        o.gated_rmsnorm_q8(s["o"], s["out_norm"], s["z"], s["mq"], s["md"], T * HV, EPS)
        o.qgemv(s["wout"], s["mq"], s["md"], s["y"], T)
    elif kind == "attn_layer":
        o.qgemv(s["wq"], s["nq"], s["nd"], s["qg"], T)
        o.qgemv(s["wk"], s["nq"], s["nd"], s["k"], T)
        o.qgemv(s["wv"], s["nq"], s["nd"], s["v"], T)
        o.attn_prep(s["qg"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["qn"], s["kc"], s["vc"], s["pos0"], T, EPS, THETA,
                    NQH, NKVH, s["n_ctx"], True)
        o.quantize_q8_1(s["attn_out"], s["mq"], s["md"], NQH * 256, T)
        o.qgemv(s["wo"], s["mq"], s["md"], s["y"], T)
    elif kind == "proj":
        o.qgemv(s["mat"], s["xq"], s["xd"], s["y"], T)
    elif kind == "embed":
        getattr(o, "get_rows_" + case["type"])(s["table"], s["row_bytes"], s["ids"], T, s["x"], E)
        o.rmsnorm_q8(s["x"], s["norm_w"], s["h"], s["nq"], s["nd"], E, T, EPS, None, s["ns"])
    elif kind == "gdn_prefill":
        o.gdn_conv_prefill(s["qkv"], s["conv_w"], s["planes"], s["plane"], s["conv"], C, T, 2 * KH, EPS, s["a"], s["b"],
                           s["ssm_a"], s["dt_bias"], s["g"], s["beta"], HV)
        o.gdn_step(q, k, v, C, s["g"], s["beta"], s["states"], s["plane"], s["o"], HV, KH, T, scale, False, None, True)
        o.gated_rmsnorm_q8(s["o"], s["out_norm"], s["z"], s["mq"], s["md"], T * HV, EPS, None, s["ms"])
    elif kind == "ffn_prefill":
        o.sum_norm_rows(s["x"], s["partial"], E, T, None, s["norm_w"], EPS, None, s["nq"], s["nd"], s["ns"])
        o.swiglu_q8(s["g"], s["u"], s["mq"], s["md"], T * FF, None, s["ms"])
    elif kind == "attn_prefill":
        o.attn_prep(s["qg"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["qn"], s["kc"], s["vc"], s["pos0"], T, EPS, THETA,
                    NQH, NKVH, s["n_ctx"], True, None, None, 0, s["rope3"])
        o.quantize_q8_1(s["attn_out"], s["mq"], s["md"], NQH * 256, T, None, s["ms"])


OUTPUTS = {
    "residual_norm": ["x", "nq", "nd"],
    "gdn_layer": ["x", "h", "nq", "nd", "a", "b", "qkv", "z", "conv", "planes", "g", "beta", "o", "states", "mq", "md", "y"],
    "attn_layer": ["x", "nq", "nd", "qg", "k", "v", "qn", "kc", "vc", "mq", "md", "y"],
    "ffn": ["x", "nq", "nd", "yg", "yu", "mq", "md", "y"],
    "proj": ["y"],
    "embed": ["x", "h", "nq", "nd", "ns"],
    "gdn_prefill": ["conv", "planes", "g", "beta", "o", "states", "mq", "md", "ms"],
    "ffn_prefill": ["x", "nq", "nd", "ns", "mq", "md", "ms"],
    "attn_prefill": ["qn", "kc", "vc", "mq", "md", "ms"],
}
GRAPHED = ("gdn_layer", "attn_layer", "ffn", "proj")
UPDATED = ("x", "planes", "states")  # inputs that a pass also writes


def _shape(case, name):
    """(type, N, K) of the weight matrix `name`."""
    if case["kind"] == "proj":
        return case["type"], case["N"], case["K"]
    t = case["down"] if name == "w_down" else case["type"]
    return (t,) + {"w_gate": (FF, E), "w_up": (FF, E), "w_down": (E, FF), "w_qkv": (C, E), "w_z": (HV * D, E),
                   "w_out": (E, HV * D), "w_q": (NQH * 512, E), "w_k": (NKVH * 256, E), "w_v": (NKVH * 256, E),
                   "w_o": (E, NQH * 256)}[name]


def prepare(case, seed):
    s = _inputs(case, seed)
    for name in [n for n in s if n == "w" or n.startswith("w_")]:
        t, N, K = _shape(case, name)
        to = {"w": "mat", "w_gate": "gate", "w_up": "up", "w_down": "down"}.get(name, name.replace("_", ""))
        s[to] = _q27().qmat_upload(s.pop(name), TYPES[t][0], N, K)
    if "table" in s:
        s["row_bytes"] = E // EMBED_BYTES[case["type"]][1] * s["table"].shape[1]
    _buffers(case, s)
    s["case"] = case
    if case["kind"] in GRAPHED:
        kept = {n: s[n].clone() for n in UPDATED if n in s}
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _launch(case, s)  # loads the kernels before they are recorded
        side.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=side):
            _launch(case, s)
        for n, t in kept.items():
            s[n].copy_(t)
        torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    if "graph" in s:
        s["graph"].replay()
    else:
        _launch(case, s)
    return {n: s[n] for n in OUTPUTS[case["kind"]]}


# ---------------------------------------------------------------- what a pass cannot do without
def _norm_work(T, h, xs):
    n = T * E
    return 3 * 4 * n + 4 * E + n + n // 8 + (4 * n if h else 0) + (n // 4 if xs else 0), 6 * n


def work(case):
    T, kind = case["T"], case["kind"]
    b = f = 0

    def gemv(t, N, K):
        nonlocal b, f
        b += N * (K // 256) * TYPES[t][1] + T * (K + K // 8) + 4 * T * N
        f += 2 * N * K * T

    if kind in ("residual_norm", "gdn_layer", "attn_layer", "ffn", "ffn_prefill"):
        nb, nf = _norm_work(T, kind == "gdn_layer", kind == "ffn_prefill")
        b, f = b + nb, f + nf
    if kind == "ffn":
        gemv(case["type"], FF, E), gemv(case["type"], FF, E), gemv(case["down"], E, FF)
        b, f = b + T * FF * 9 + T * FF // 8, f + 8 * T * FF
    elif kind in ("gdn_layer", "gdn_prefill"):
        if kind == "gdn_layer":
            gemv(case["type"], C, E), gemv(case["type"], HV * D, E), gemv(case["type"], E, HV * D)
            b, f = b + 2 * HV * E * 2 + 4 * T * (E + 2 * HV), f + 4 * HV * E * T
        planes = T if kind == "gdn_layer" else 1
        b += T * (2 * C + 4 * HV) * 4 + C * 16 + (1 + planes) * C * 12  # conv, gates, window state
        b += T * (C + HV * D + 2 * HV) * 4 + (1 + planes) * HV * D * D * 4  # recurrence
        b += T * HV * D * 9 + T * HV * D // 8 + (T * HV * D // 4 if kind == "gdn_prefill" else 0)  # gated norm
        f += T * C * 14 + 7 * T * HV * D * D + 12 * T * HV * D
    elif kind in ("attn_layer", "attn_prefill"):
        if kind == "attn_layer":
            gemv(case["type"], NQH * 512, E), gemv(case["type"], NKVH * 256, E), gemv(case["type"], NKVH * 256, E)
            gemv(case["type"], E, NQH * 256)
        b += T * (NQH * 256 * 8 + NKVH * 256 * 8 + 2 * NKVH * 272)
        b += T * NQH * 256 * 5 + T * NQH * 256 // 8 + (T * NQH * 64 if kind == "attn_prefill" else 0)
        f += T * (NQH + NKVH) * 256 * 8 + T * NQH * 256 * 4
    elif kind == "proj":
        gemv(case["type"], case["N"], case["K"])
    elif kind == "embed":
        bb, bv = EMBED_BYTES[case["type"]]
        b += T * (4 * E + E // bv * bb + 4)  # gather
        b += T * (4 * E + 4 * E + E + E // 8 + E // 4) + 4 * E
        f += 10 * T * E
    elif kind == "ffn_prefill":
        b, f = b + T * FF * 9 + T * FF // 8 + T * FF // 4, f + 10 * T * FF
    return {"bytes": b, "flops": f}


def tolerance(case):
    # Float outputs agree with float64 to 2.4e-7 (sums of 32-bit floats). Two rounded outputs set the bars of the
    # blocks that quantize: a value within float32 rounding of a tie may go one unit either way (one in a few hundred
    # thousand; "differ"), a block scale one fp16 step (5e-4 of the value, one scale in a few thousand), and in a decode
    # block one such unit moves the projection after it by about 1e-4 of its norm.
    if case["kind"] in ("gdn_layer", "attn_layer", "ffn"):
        return {"rel": 5e-4, "max": 1e-2, "differ": 5e-4}
    if case["kind"] == "proj":
        return {"rel": 1e-6, "max": 4e-5}
    return {"rel": 5e-5, "max": 2e-3, "differ": 2e-4}


# ---------------------------------------------------------------- float64 restatement
_tables = {}


def _table(name):
    """A codebook of the GGUF formats (data)."""
    if name not in _tables:
        text = "\n".join(x for x in open(os.path.join(PKG, "csrc", name + ".inc")) if not x.lstrip().startswith("//"))
        vals = [int(v, 0) for v in re.findall(r"-?0x[0-9a-fA-F]+|-?\d+", re.sub(r"(?<=[0-9a-fA-F])[uU][lL]*", "", text))]
        vals = [v - (1 << 64) if v >= 1 << 63 else v for v in vals]
        _tables[name] = torch.tensor(vals, dtype=torch.int64, device=DEV)
    return _tables[name]


def _half(B, off):
    return (B[:, off:off + 2].contiguous().view(torch.float16).to(torch.float64)).reshape(-1, 1)


def _bytes_of(v, n):
    """Bytes 0 .. n - 1 of int64 values, as a last axis."""
    return torch.stack([(v >> (8 * j)) & 0xFF for j in range(n)], -1)


def _signed(mag, signs):
    """mag [..., 8] negated where the sign byte has a bit."""
    return torch.stack([torch.where((signs >> j) & 1 != 0, -mag[..., j], mag[..., j]) for j in range(8)], -1)


def _ksigns(v):
    p = v ^ (v >> 4)
    p = p ^ (p >> 2)
    p = p ^ (p >> 1)
    return v | ((p & 1) << 7)


def _dequant(type_, raw):
    """Raw blocks -> (q, sc, d, m): weight = d * sc * q - m with q [n][256] and sc [n][16 or 8] before the super-block
    scale d [n][1], m [n][256] or 0."""
    n = raw.shape[0]
    B = raw.to(torch.int64)
    at = lambda off, cnt: B[:, off:off + cnt]  # noqa: E731
    m = 0
    if type_ == "q4_k":
        d, sc6 = _half(raw, 0), at(4, 12)
        sc = torch.cat([sc6[:, :4] & 63, (sc6[:, 8:] & 15) | ((sc6[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([sc6[:, 4:8] & 63, (sc6[:, 8:] >> 4) | ((sc6[:, 4:8] >> 6) << 4)], 1)
        qs = at(16, 128).view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 256)
        m = (_half(raw, 2) * mn).repeat_interleave(32, 1)
    elif type_ == "q2_k":
        d, sc = _half(raw, 80), at(0, 16) & 15
        qs = at(16, 64).view(n, 2, 1, 32)
        q = torch.cat([(qs >> (2 * j)) & 3 for j in range(4)], 2).reshape(n, 256)
        m = (_half(raw, 82) * (at(0, 16) >> 4)).repeat_interleave(16, 1)
    elif type_ == "q6_k":
        d, sc = _half(raw, 208), raw[:, 192:208].contiguous().view(torch.int8).to(torch.int64)
        ql, qh = at(0, 128).view(n, 2, 2, 32), at(128, 64).view(n, 2, 32)
        parts = [(ql[:, :, j & 1] >> (4 * (j >> 1)) & 15) | ((qh >> (2 * j) & 3) << 4) for j in range(4)]
        q = (torch.stack(parts, 2) - 32).reshape(n, 256)
    elif type_ == "iq4_xs":
        d, lv = _half(raw, 0), _table("iq4nl_values")
        hi = B[:, 2:3] | (B[:, 3:4] << 8)
        sc = torch.stack([((B[:, 4 + s // 2] >> (4 * (s & 1))) & 15 | ((hi[:, 0] >> (2 * s)) & 3) << 4) - 32 for s in range(8)], 1)
        qs = at(8, 128).view(n, 8, 1, 16)
        q = lv[torch.cat([qs & 15, qs >> 4], 2)].reshape(n, 256)
    elif type_ == "iq3_s":
        d, s4 = _half(raw, 0), at(106, 4)
        sc = 1 + 2 * torch.stack([s4 & 15, s4 >> 4], 2).reshape(n, 8)
        qh = at(66, 8).view(n, 8, 1)
        sh = 8 - torch.arange(8, device=DEV)
        idx = at(2, 64).view(n, 8, 8) | ((qh << sh) & 256)
        q = _signed(_bytes_of(_table("iq3s_grid")[idx], 4).view(n, 32, 8), at(74, 32)).reshape(n, 256)
    elif type_ in ("iq2_xxs", "iq3_xxs"):
        d = _half(raw, 0)
        w = at(2, 64).view(n, 8, 8) if type_ == "iq2_xxs" else at(66, 32).view(n, 8, 4)
        a = w[:, :, -4:]
        aux = a[..., 0] | (a[..., 1] << 8) | (a[..., 2] << 16) | (a[..., 3] << 24)
        sg = _ksigns(torch.stack([(aux >> (7 * p)) & 127 for p in range(4)], 2))
        sc = aux >> 28
        if type_ == "iq2_xxs":
            mag = _bytes_of(_table("iq2xxs_grid")[w[:, :, :4]], 8)
        else:
            mag = _bytes_of(_table("iq3xxs_grid")[at(2, 64).view(n, 8, 4, 2)], 4).reshape(n, 8, 4, 8)
        q = _signed(mag, sg).reshape(n, 256)
    elif type_ in ("iq2_xs", "iq2_s"):
        d = _half(raw, 0)
        s8 = at(66 if type_ == "iq2_xs" else 74, 8)
        sc = torch.stack([s8 & 15, s8 >> 4], 2).reshape(n, 16)
        if type_ == "iq2_xs":
            v = at(2, 64).view(n, 8, 4, 2)
            v = v[..., 0] | (v[..., 1] << 8)
            idx, sg, grid = v & 511, _ksigns(v >> 9), _table("iq2xs_grid")
        else:
            sh = 8 - 2 * torch.arange(4, device=DEV)
            idx = at(2, 32).view(n, 8, 4) | ((at(66, 8).view(n, 8, 1) << sh) & 0x300)
            sg, grid = at(34, 32).view(n, 8, 4), _table("iq2s_grid")
        q = _signed(_bytes_of(grid[idx], 8), sg).reshape(n, 256)
    else:  # iq1_m
        w = at(48, 8).view(n, 4, 2)
        w = w[..., 0] | (w[..., 1] << 8)
        dh = (w[:, 0] >> 12) | ((w[:, 1] >> 8) & 0xF0) | ((w[:, 2] >> 4) & 0xF00) | (w[:, 3] & 0xF000)
        d = dh.to(torch.int16).view(torch.float16).to(torch.float64).view(n, 1)
        sc = 2 * torch.stack([(w[:, s // 4] >> (6 * ((s // 2) % 2) + 3 * (s & 1))) & 7 for s in range(16)], 1) + 1
        h = at(32, 16)
        h = torch.stack([h & 15, h >> 4], 2).view(n, 32)
        g = _table("iq1s_grid")[at(0, 32) | ((h & 7) << 8)]
        nib = torch.cat([torch.stack([(g >> (8 * j)) & 15 for j in range(4)], -1),
                         torch.stack([(g >> (8 * j + 4)) & 15 for j in range(4)], -1)], -1)
        q = (nib.to(torch.float64) + torch.where(h & 8 != 0, -1.125, -0.875).to(torch.float64).unsqueeze(-1)).reshape(n, 256)
    return q, sc, d, m


def _scale_value(type_, sc):
    """The factor of a sub-block scale in the dequantized weight."""
    sc = sc.to(torch.float64)
    return {"iq2_xxs": (sc + 0.5) * 0.25, "iq2_xs": (sc + 0.5) * 0.25, "iq2_s": (sc + 0.5) * 0.25,
            "iq3_xxs": (sc + 0.5) * 0.5}.get(type_, sc)


def _weights64(type_, raw):
    if type_ == "q8_0":
        return raw[:, 2:34].contiguous().view(torch.int8).to(torch.float64) * _half(raw, 0)
    q, sc, d, m = _dequant(type_, raw)
    return d * _scale_value(type_, sc).repeat_interleave(256 // sc.shape[1], 1) * q - m


def _gemv64(type_, raw, N, K, xq, xd, T):
    """[T][N]: the products of the weights with the int8 activations times their scales. Four formats round each
    sub-block's scaled integer sum towards zero (their integer scale rules)."""
    nb = K // 256
    x, dx = xq.view(T, K).to(torch.float64), xd.view(T, K // 32).to(torch.float64)
    y = torch.empty(T, N, dtype=torch.float64, device=DEV)
    step = max(8, (1 << 26) // K)
    for r0 in range(0, N, step):
        n = min(step, N - r0)
        B = raw[r0 * nb:(r0 + n) * nb]
        if type_ not in ("iq2_xxs", "iq2_xs", "iq2_s", "iq3_xxs"):
            W = _weights64(type_, B).view(n, K)
            y[:, r0:r0 + n] = (x * dx.repeat_interleave(32, 1)) @ W.t()
            continue
        q, sc, d, _ = _dequant(type_, B)
        A = q.to(torch.float64).view(n, K // 16, 16).transpose(0, 1).contiguous()  # [K / 16][n][16]
        P = torch.bmm(A, x.view(T, K // 16, 16).permute(1, 2, 0).contiguous()).view(K // 32, 2, n, T)
        s0, s1 = P[:, 0], P[:, 1]
        per = lambda v: v.view(n, K // 32, -1).permute(1, 0, 2)  # noqa: E731
        sc = per(sc.to(torch.float64).view(n, nb, 8, -1).reshape(n, K // 32, -1))
        if type_ == "iq2_xxs":
            v = torch.trunc((s0 + s1) * (2 * sc + 1) / 8)
        elif type_ == "iq3_xxs":
            v = torch.trunc((sc * (s0 + s1) + torch.trunc((s0 + s1) / 2)) / 2)
        else:
            v = torch.trunc((s0 * sc[..., :1] + s1 * sc[..., 1:] + torch.trunc((s0 + s1) / 2)) / 4)
        dd = per(d.view(n, nb, 1).expand(n, nb, 8).reshape(n, K // 32))
        y[:, r0:r0 + n] = (v * dd * dx.t().unsqueeze(1)).sum(0).t()
    return y


def _q8(y):
    """The int8 quantization of rows in blocks of 32: (q, fp16 scale, sums per 16)."""
    v = y.reshape(-1, 32)
    d = v.abs().amax(1, keepdim=True) / 127
    t = torch.where(d > 0, v / torch.where(d > 0, d, 1.0), 0.0)
    return (torch.sign(t) * torch.floor(t.abs() + 0.5)).reshape(-1), d.float().half().double().reshape(-1), y.reshape(-1, 16).sum(1)


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _gdn64(case, s, snapshots, out):
    """conv + SiLU + L2 norm + gates, the delta rule, the gated norm."""
    T = case["T"]
    f64 = lambda n: s[n].double()  # noqa: E731
    p0 = int(s["plane"].item())
    planes = f64("planes").view(4, C, 3).clone()
    x = torch.cat([planes[p0].t(), f64("qkv").view(T, C)])
    w = f64("conv_w").view(C, 4)
    y = sum(x[j:j + T] * w[:, j] for j in range(4))
    y = (y * torch.sigmoid(y)).view(T, C // D, D)
    y[:, :2 * KH] /= torch.sqrt((y[:, :2 * KH] ** 2).sum(-1, keepdim=True) + EPS)
    if snapshots:
        for t in range(T):
            planes[t] = x[t + 1:t + 4].t()
    else:
        planes[1 if p0 == 0 else 0] = x[T:T + 3].t()
    beta = torch.sigmoid(f64("b").view(T, HV))
    g = torch.nn.functional.softplus(f64("a").view(T, HV) + f64("dt_bias"), threshold=1e9) * f64("ssm_a")
    states = f64("states").view(4, HV, D, D).clone()  # [value column][key]
    S, eg, o = states[p0].clone(), torch.exp(g), torch.empty(T, HV, D, dtype=torch.float64, device=DEV)
    head = torch.arange(HV, device=DEV) % KH
    q, k, v = y[:, :KH][:, head], y[:, KH:2 * KH][:, head], y[:, 2 * KH:]
    for t in range(T):
        S = S * eg[t].view(HV, 1, 1)
        delta = (v[t] - torch.bmm(S, k[t].unsqueeze(2)).squeeze(2)) * beta[t].view(HV, 1)
        S = S + delta.unsqueeze(2) * k[t].unsqueeze(1)
        o[t] = torch.bmm(S, q[t].unsqueeze(2)).squeeze(2)
        if snapshots:
            states[t] = S
    if not snapshots:
        states[1 if p0 == 0 else 0] = S
    o = o / math.sqrt(D)
    z = f64("z").view(T, HV, D)
    m = _rms64(o, s["out_norm"]) * z * torch.sigmoid(z)
    out.update(conv=y, planes=planes, g=g, beta=beta, o=o, states=states)
    out["mq"], out["md"], out["ms"] = _q8(m.reshape(-1))


def _prep64(case, s):
    T = case["T"]
    q = _rms64(s["qg"].double().view(T, NQH, 512)[..., :256], s["q_norm"])
    pos = s["pos0"] + torch.arange(T, dtype=torch.int32, device=DEV)
    p3 = s["rope3"].view(T, 3) if s.get("rope3") is not None else pos.view(T, 1).expand(T, 3)
    j = torch.arange(32)
    freq = (torch.tensor(THETA, dtype=torch.float32) ** j.float()).to(DEV)
    ang = (p3[:, (j % 3).to(DEV)].float() * freq).double().unsqueeze(1)  # the angle is a float32 product
    sn, cs = torch.sin(ang), torch.cos(ang)
    a, b = q[..., :32], q[..., 32:64]
    return torch.cat([a * cs - b * sn, a * sn + b * cs, q[..., 64:]], -1)


def exact(case, seed):
    s, T, kind, out = _inputs(case, seed), case["T"], case["kind"], {}

    def gemv(name, q, d):
        t, N, K = _shape(case, name)
        return _gemv64(t, s[name], N, K, q, d, T)

    if kind in ("residual_norm", "gdn_layer", "attn_layer", "ffn", "ffn_prefill"):
        x = s["x"].double().view(T, E) + s["partial"].double().view(T, E)
        h = _rms64(x, s["norm_w"])
        out["x"], out["h"] = x, h
        out["nq"], out["nd"], out["ns"] = _q8(h.reshape(-1))
    if kind == "ffn":
        out["yg"], out["yu"] = gemv("w_gate", out["nq"], out["nd"]), gemv("w_up", out["nq"], out["nd"])
        out["mq"], out["md"], _ = _q8((out["yg"] * torch.sigmoid(out["yg"]) * out["yu"]).reshape(-1))
        out["y"] = gemv("w_down", out["mq"], out["md"])
    elif kind == "gdn_layer":
        out["a"], out["b"] = (out["h"] @ s[n].double().view(HV, E).t() for n in ("wa", "wb"))
        out["qkv"], out["z"] = gemv("w_qkv", out["nq"], out["nd"]), gemv("w_z", out["nq"], out["nd"])
        s.update({n: out[n].reshape(-1) for n in ("a", "b", "qkv", "z")})
        _gdn64(case, s, True, out)
        out["y"] = gemv("w_out", out["mq"], out["md"])
    elif kind == "attn_layer":
        for n in ("q", "k", "v"):
            out["qg" if n == "q" else n] = gemv("w_" + n, out["nq"], out["nd"])
        s["qg"] = out["qg"]
        out["qn"] = _prep64(case, s)
        out["mq"], out["md"], _ = _q8(s["attn_out"].double())
        out["y"] = gemv("w_o", out["mq"], out["md"])
    elif kind == "proj":
        out["y"] = gemv("w", s["xq"], s["xd"])
    elif kind == "embed":
        rows = s["table"].view(VOCAB, -1)[s["ids"].long()].view(-1, s["table"].shape[1])
        out["x"] = _weights64(case["type"], rows).view(T, E)
        out["h"] = _rms64(out["x"], s["norm_w"])
        out["nq"], out["nd"], out["ns"] = _q8(out["h"].reshape(-1))
    elif kind == "gdn_prefill":
        _gdn64(case, s, False, out)
    elif kind == "ffn_prefill":
        g, u = s["g"].double(), s["u"].double()
        out["mq"], out["md"], out["ms"] = _q8(g * torch.sigmoid(g) * u)
    elif kind == "attn_prefill":
        out["qn"] = _prep64(case, s)
        out["mq"], out["md"], out["ms"] = _q8(s["attn_out"].double())
    # the int8 values, the fp16 scales and the cache bytes are rounded outputs; the floats have a 64-bit value
    whole = ("nq", "nd", "mq", "md", "kc", "vc")
    return {n: None if n in whole else out[n].reshape(-1) for n in OUTPUTS[kind]}
