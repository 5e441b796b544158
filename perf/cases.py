"""The work that users of this framework have it do, as cases that can be timed and compared.

Every case goes through the public modules and functions: ``HelixLinear.forward`` (decode GEMV
and prefill GEMM, eager or captured in a HIP graph), ``chunked_scan``, ``HelixMamba2Mixer``
(prefill and single-token step), ``HelixMoeExperts``, ``HelixDecoder`` and the CDNAv3 encoder.
Weights follow the benchmark recipe: sorted Gaussian codebook, indices close to
Binomial(255, 1/2), group-128 affine, 0.1 % sidecar of +-U(4, 8) sigma outliers.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path
from statistics import NormalDist

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "helix-substrate_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from helix_substrate.decoder import QWEN25_3B, QWEN25_7B, DecoderConfig, HelixDecoder  # noqa: E402
from helix_substrate.generate_sidecars_v3 import find_outliers_percentile  # noqa: E402
from helix_substrate.helix_linear import HelixLinear  # noqa: E402
from helix_substrate.hxq_encoder import (build_kmeans_codebook, chunked_assign,  # noqa: E402
                                         fit_group_affine)
from helix_substrate.index_packing import pack_12bit  # noqa: E402
from helix_substrate.mamba2_mixer import HelixMamba2Mixer  # noqa: E402
from helix_substrate.moe import HelixMoeExperts  # noqa: E402
from helix_substrate.ssm_scan import chunked_scan  # noqa: E402

DEV = "cuda"
GROUP = 128
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SHAPES = {"3b": QWEN25_3B, "7b": QWEN25_7B}


def listed():
    return [
        # one projection called eagerly on one fp32 token: what a call costs at least
        {"name": "linear_token_f32", "kind": "linear", "m": 1, "k": 2048, "n": 2048,
         "dtype": "f32", "fmt": "u8", "bias": False},
        # the seven projections of a Qwen2.5-7B layer on one bf16 token, replayed from a HIP
        # graph as a serving loop does
        {"name": "layer_token_graph_bf16", "kind": "layer", "m": 1, "shape": "7b",
         "dtype": "bf16"},
        # continuous-batching decode: sixteen sequences share the gate projection
        {"name": "linear_batch16_bf16", "kind": "linear", "m": 16, "k": 3584, "n": 18944,
         "dtype": "bf16", "fmt": "u8", "bias": False},
        # a short prompt on a 12-bit pair codebook whose sizes fit no tile
        {"name": "linear_ragged_pairs_f16", "kind": "linear", "m": 45, "k": 2050, "n": 5006,
         "dtype": "f16", "fmt": "p12", "bias": True},
        # prefill of an ordinary prompt, gate/up of Qwen2.5-7B
        {"name": "linear_prefill_bf16", "kind": "linear", "m": 2048, "k": 3584, "n": 18944,
         "dtype": "bf16", "fmt": "u8", "bias": False},
        # prefill of a long prompt (or a batch of prompts), down of Qwen2.5-7B
        {"name": "linear_prefill_long_bf16", "kind": "linear", "m": 8192, "k": 18944,
         "n": 3584, "dtype": "bf16", "fmt": "u8", "bias": False},
        # the selective scan of a Mamba2-1.3B layer over a training-sized batch
        {"name": "scan_bf16", "kind": "scan", "batch": 8, "len": 2048, "heads": 64, "p": 64,
         "state": 128, "groups": 1, "dtype": "bf16", "h0": False},
        # a whole Mamba2-1.3B mixer on two prompts of a length that is no multiple of the chunk
        {"name": "mixer_prompt_bf16", "kind": "mixer", "batch": 2, "len": 1000,
         "d_model": 2048, "heads": 64, "p": 64, "state": 128, "dtype": "bf16"},
        # an OLMoE-shaped expert layer while four sequences decode
        {"name": "moe_decode4_bf16", "kind": "moe", "tokens": 4, "hidden": 2048,
         "inter": 1024, "experts": 64, "top_k": 8, "dtype": "bf16"},
        # the same layer on a prompt
        {"name": "moe_prompt512_bf16", "kind": "moe", "tokens": 512, "hidden": 2048,
         "inter": 1024, "experts": 64, "top_k": 8, "dtype": "bf16"},
        # a greedy decode step of the Qwen2.5-3B-shaped model, one launch per token
        {"name": "decoder_step_3b", "kind": "decoder", "shape": "3b", "layers": 36, "pos": 255},
        # encoding one gate projection: codebook, indices, sidecar and affine
        {"name": "encode_gate_f32", "kind": "encode", "rows": 11008, "cols": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "layer", "scan", "mixer",
                       "mixer_step", "moe", "decoder", "encode"])
    if kind == "linear":
        fmt = rng.choice(["u8", "u8", "u8", "p12", "vq2", "wide"])
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        m, n, k = _log(rng, 1, 8192), _log(rng, 256, 18944), _log(rng, 256, 18944)
        if rng.random() < 0.3:
            k = 2 * (k // 2)
            affine = False
        else:
            k = GROUP * max(1, k // GROUP)
            affine = fmt in ("u8", "wide")
        if fmt == "p12":
            n = 2 * ((n + 1) // 2)   # the packing holds an even number of pairs
        most = 8192 * 18944 * 3584 / (16 if dtype == "f32" else 1.5)
        m = max(1, min(m, int(most / (n * k))))
        return {"kind": "linear", "m": m, "k": k, "n": n, "dtype": dtype,
                "fmt": fmt, "bias": rng.random() < 0.5, "affine": affine}
    if kind == "layer":
        return {"kind": "layer", "m": _log(rng, 1, 64), "shape": rng.choice(["3b", "7b"]),
                "dtype": rng.choice(["bf16", "f16"])}
    if kind == "scan":
        batch = rng.choice([1, 2, 4, 8])
        return {"kind": "scan", "batch": batch, "len": _log(rng, 65, 16384 // batch),
                "heads": rng.choice([16, 24, 64]), "p": rng.choice([32, 64]),
                "state": rng.choice([64, 128]), "groups": rng.choice([1, 2]),
                "dtype": rng.choice(["bf16", "bf16", "f16"]), "h0": rng.random() < 0.5}
    if kind == "mixer":
        batch = rng.choice([1, 2, 4])
        return {"kind": "mixer", "batch": batch, "len": _log(rng, 17, 8192 // batch),
                "d_model": rng.choice([1024, 2048]), "heads": rng.choice([32, 64]), "p": 64,
                "state": rng.choice([64, 128]), "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "mixer_step":
        return {"kind": "mixer_step", "batch": _log(rng, 1, 64), "d_model": 2048, "heads": 64,
                "p": 64, "state": 128, "dtype": "bf16"}
    if kind == "moe":
        return {"kind": "moe", "tokens": _log(rng, 1, 2048), "hidden": 2048, "inter": 1024,
                "experts": rng.choice([16, 32, 64]), "top_k": rng.choice([2, 4, 8]),
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "decoder":
        shape = rng.choice(["3b", "7b"])
        return {"kind": "decoder", "shape": shape, "layers": rng.randint(2, 20),
                "pos": _log(rng, 1, 500)}
    return {"kind": "encode", "rows": _log(rng, 256, 11008),
            "cols": GROUP * _log(rng, 2, 16)}


# ------------------------------------------------------------------------ inputs
def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(seed * 7919 + salt)


def _codebook(k, sigma):
    nd = NormalDist()
    return torch.tensor([nd.inv_cdf((i + 0.5) / k) * sigma for i in range(k)],
                        dtype=torch.float32, device=DEV)


_CB = {}


def _cb(k, sigma):
    if (k, sigma) not in _CB:
        _CB[k, sigma] = _codebook(k, sigma)
    return _CB[k, sigma].clone()


def _normal_levels(shape, top, g):
    """Integers 0..top, normal around the middle (Binomial(255, 1/2) at top = 255)."""
    half = top / 2.0
    x = torch.randn(shape, generator=g, device=DEV).mul_(half / 16.0).add_(half).round_()
    return x.clamp_(0, top)


def _weights(n, k, g, sigma=0.02, fmt="u8", affine=True, bias=False):
    """One compressed matrix [n, k]: a dict of device tensors."""
    w = {"n": n, "k": k, "fmt": fmt, "bias": None, "scale": None, "offset": None}
    if fmt in ("p12", "vq2"):
        w["codebook"] = torch.randn(4096, 2, generator=g, device=DEV) * sigma
        w["indices"] = torch.randint(0, 4096, (n, k // 2), generator=g, device=DEV)
    elif fmt == "wide":
        w["codebook"] = _cb(1024, sigma)
        w["indices"] = _normal_levels((n, k), 1023, g).to(torch.int16)
    else:
        w["codebook"] = _cb(256, sigma)
        w["indices"] = _normal_levels((n, k), 255, g).to(torch.uint8)
    if affine and fmt in ("u8", "wide"):
        w["scale"] = torch.empty(n, k // GROUP, device=DEV).uniform_(0.95, 1.05, generator=g)
        w["offset"] = torch.randn(n, k // GROUP, generator=g, device=DEV) * 1e-4
    nnz = max(1, n * k // 1000)
    step = n * k // nnz          # one outlier in each run of `step` weights
    w["pos"] = (torch.arange(nnz, device=DEV) * step
                + torch.randint(0, step, (nnz,), generator=g, device=DEV))
    sign = torch.randint(0, 2, (nnz,), generator=g, device=DEV) * 2.0 - 1.0
    mag = torch.empty(nnz, device=DEV).uniform_(4.0, 8.0, generator=g) * sigma
    w["val"] = (sign * mag).half().float()
    if bias:
        w["bias"] = torch.randn(n, generator=g, device=DEV) * 0.02
    return w


def _linear(w):
    idx = w["indices"]
    if w["fmt"] == "p12":
        idx = pack_12bit(idx)
    return HelixLinear(w["k"], w["n"], w["codebook"], idx, w["pos"], w["val"], bias=w["bias"],
                       vector_dim=2 if w["fmt"] in ("p12", "vq2") else 1,
                       group_scale=w["scale"], group_offset=w["offset"],
                       group_size=GROUP).to(DEV)


def _dense(w):
    """The weights that the compressed form stands for, in 64 bits."""
    W = w["codebook"].double()[w["indices"].long()].reshape(w["n"], w["k"])
    if w["scale"] is not None:
        W = W.view(w["n"], -1, GROUP) * w["scale"].double().unsqueeze(-1)
        W = (W + w["offset"].double().unsqueeze(-1)).reshape(w["n"], w["k"])
    W.view(-1)[w["pos"]] = w["val"].double()
    return W


def _apply(x, w):
    y = x.double() @ _dense(w).t()
    return y if w["bias"] is None else y + w["bias"].double()


def _bytes(n, k, fmt="u8", affine=True):
    b = n * k * {"u8": 1.0, "wide": 2.0, "vq2": 1.0, "p12": 0.75}[fmt] + 8 * (n * k // 1000)
    return b + (8 * n * (k // GROUP) if affine and fmt in ("u8", "wide") else 0)


def _layer_shapes(c):
    h, i, d = c.hidden, c.intermediate, c.head_dim
    return {"q": (c.n_heads * d, h), "k": (c.n_kv_heads * d, h), "v": (c.n_kv_heads * d, h),
            "o": (h, c.n_heads * d), "gate": (i, h), "up": (i, h), "down": (h, i)}


def _layer_inputs(case, seed):
    g = _gen(seed)
    c = SHAPES[case["shape"]]
    ws = {p: _weights(n, k, g, bias=p in "qkv") for p, (n, k) in _layer_shapes(c).items()}
    rand = lambda k: torch.randn(case["m"], k, generator=g, device=DEV).to(DTYPES[case["dtype"]])
    xs = {"attn": rand(c.hidden), "heads": rand(c.n_heads * c.head_dim), "mlp": rand(c.hidden),
          "act": rand(c.intermediate)}
    return ws, xs


_LAYER_X = {"q": "attn", "k": "attn", "v": "attn", "o": "heads", "gate": "mlp", "up": "mlp",
            "down": "act"}


def _linear_inputs(case, seed):
    g = _gen(seed)
    w = _weights(case["n"], case["k"], g, fmt=case["fmt"], affine=case.get("affine", True),
                 bias=case["bias"])
    x = torch.randn(case["m"], case["k"], generator=g, device=DEV).to(DTYPES[case["dtype"]])
    return w, x


def _scan_inputs(case, seed):
    g = _gen(seed)
    b, L, H, P, N, G = (case[k] for k in ("batch", "len", "heads", "p", "state", "groups"))
    dt = DTYPES[case["dtype"]]
    n = lambda *s: torch.randn(*s, generator=g, device=DEV)
    return {"h0": n(b, H, P, N) * 0.1 if case["h0"] else None,
            "dt": torch.nn.functional.softplus(n(b, L, H) * 0.5 - 2.0),
            "A": -torch.exp(torch.rand(H, generator=g, device=DEV) * math.log(16.0)),
            "x": n(b, L, H, P).to(dt), "B": (n(b, L, G, N) / math.sqrt(N)).to(dt),
            "C": (n(b, L, G, N) / math.sqrt(N)).to(dt),
            "D": torch.rand(H, 1, generator=g, device=DEV) + 0.5}


def _mixer_inputs(case, seed):
    g = _gen(seed)
    H, P, N, dm = case["heads"], case["p"], case["state"], case["d_model"]
    inner, conv = H * P, H * P + 2 * N
    u = lambda *s: torch.rand(*s, generator=g, device=DEV)
    step = torch.exp(u(H) * (math.log(0.1) - math.log(1e-3)) + math.log(1e-3))
    m = {"in": _weights(2 * inner + 2 * N + H, dm, g), "out": _weights(dm, inner, g),
         "conv_w": u(conv, 4) - 0.5, "conv_b": u(conv) - 0.5,
         "dt_bias": step + torch.log(-torch.expm1(-step)), "A_log": torch.log(u(H) * 15 + 1),
         "D": torch.ones(H, device=DEV),
         "norm": 1.0 + 0.1 * torch.randn(inner, generator=g, device=DEV)}
    shape = (case["batch"], dm) if case["kind"] == "mixer_step" else (case["batch"], case["len"], dm)
    x = torch.randn(shape, generator=g, device=DEV).to(DTYPES[case["dtype"]])
    state = None
    if case["kind"] == "mixer_step":
        state = (torch.randn(case["batch"], conv, 4, generator=g, device=DEV),
                 torch.randn(case["batch"], H, P, N, generator=g, device=DEV) * 0.1)
    return m, x, state


def _moe_inputs(case, seed):
    g = _gen(seed)
    E, h, i = case["experts"], case["hidden"], case["inter"]
    banks = {}
    for name, n, k in (("gate", i, h), ("up", i, h), ("down", h, i)):
        w = _weights(E * n, k, g)   # all experts at once, then cut by rows
        idx, sc, so = (w[t].view(E, n, -1) for t in ("indices", "scale", "offset"))
        cuts = torch.searchsorted(w["pos"], torch.arange(E + 1, device=DEV) * (n * k)).tolist()
        banks[name] = [{"indices": idx[e], "codebook": w["codebook"], "group_scale": sc[e],
                        "group_offset": so[e], "group_size": GROUP,
                        "sidecar_positions": w["pos"][cuts[e]:cuts[e + 1]] - e * n * k,
                        "sidecar_values": w["val"][cuts[e]:cuts[e + 1]]} for e in range(E)]
    x = torch.randn(case["tokens"], h, generator=g, device=DEV).to(DTYPES[case["dtype"]])
    logits = torch.randn(case["tokens"], E, generator=g, device=DEV)
    return banks, x, logits


def _decoder_inputs(case, seed):
    g = _gen(seed)
    c = SHAPES[case["shape"]]
    cfg = DecoderConfig(c.hidden, case["layers"], c.n_heads, c.n_kv_heads, c.head_dim,
                        c.intermediate, c.vocab, c.rope_theta, c.rms_eps, 512)
    layers = []
    for _ in range(cfg.n_layers):
        L = {p: _weights(n, k, g, bias=p in "qkv") for p, (n, k) in _layer_shapes(cfg).items()}
        L["in_norm"] = 1.0 + 0.1 * torch.randn(cfg.hidden, generator=g, device=DEV)
        L["post_norm"] = 1.0 + 0.1 * torch.randn(cfg.hidden, generator=g, device=DEV)
        kv = torch.randn(2, case["pos"], cfg.n_kv_heads, cfg.head_dim, generator=g, device=DEV)
        L["kv"] = kv.to(torch.bfloat16)   # what earlier tokens left in the cache
        layers.append(L)
    embed = (torch.randn(cfg.vocab, cfg.hidden, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    norm = 1.0 + 0.1 * torch.randn(cfg.hidden, generator=g, device=DEV)
    tok = torch.randint(0, cfg.vocab, (1,), generator=g, device=DEV).to(torch.int32)
    pos = torch.tensor([case["pos"]], dtype=torch.int32, device=DEV)
    return cfg, layers, embed, norm, tok, pos


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        return {"kind": kind, "mod": _linear(w), "x": x}
    if kind == "layer":
        ws, xs = _layer_inputs(case, seed)
        mods = {p: _linear(w) for p, w in ws.items()}
        call = lambda: {p: m(xs[_LAYER_X[p]]) for p, m in mods.items()}
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            call()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        return {"kind": kind, "mods": mods, "xs": xs, "graph": graph, "out": out}
    if kind == "scan":
        return {"kind": kind, **_scan_inputs(case, seed)}
    if kind in ("mixer", "mixer_step"):
        m, x, state = _mixer_inputs(case, seed)
        mod = HelixMamba2Mixer(_linear(m["in"]), _linear(m["out"]), m["conv_w"], m["conv_b"],
                               m["dt_bias"], m["A_log"], m["D"], m["norm"],
                               num_heads=case["heads"], head_dim=case["p"],
                               ssm_state_size=case["state"]).to(DEV)
        return {"kind": kind, "mod": mod, "x": x, "from": state,
                "state": mod.new_state(case["batch"], DEV)}
    if kind == "moe":
        banks, x, logits = _moe_inputs(case, seed)
        mod = HelixMoeExperts.from_layers(banks["gate"], banks["up"], banks["down"],
                                          top_k=case["top_k"])
        return {"kind": kind, "mod": mod, "x": x, "logits": logits}
    if kind == "decoder":
        cfg, layers, embed, norm, tok, pos = _decoder_inputs(case, seed)
        dec = HelixDecoder(cfg, [{k: _linear(v) if isinstance(v, dict) else v
                                  for k, v in L.items() if k != "kv"} for L in layers],
                           embed, norm)
        for L, kc, vc in zip(layers, dec.kc, dec.vc):
            kc[:case["pos"]], vc[:case["pos"]] = L["kv"][0], L["kv"][1]
        dec.persistent_init()
        return {"kind": kind, "dec": dec, "tok": tok, "pos": pos}
    w = torch.randn(case["rows"], case["cols"], generator=_gen(seed), device=DEV) * 0.02
    return {"kind": kind, "w": w}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["mod"](state["x"])
    if kind == "layer":
        state["graph"].replay()
        return state["out"]
    if kind == "scan":
        y, h = chunked_scan(state["h0"], state["dt"], state["A"], state["x"], state["B"],
                            state["C"], state["D"])
        return {"y": y, "h": h}
    if kind == "mixer":
        y = state["mod"](state["x"], state["state"])
        return {"y": y, "conv": state["state"][0], "ssm": state["state"][1]}
    if kind == "mixer_step":
        for t, f in zip(state["state"], state["from"]):
            t.copy_(f)
        y = state["mod"].step(state["x"], state["state"])
        return {"y": y, "conv": state["state"][0], "ssm": state["state"][1]}
    if kind == "moe":
        return state["mod"](state["x"], state["logits"])
    if kind == "decoder":
        dec = state["dec"]
        dec.tok.copy_(state["tok"])
        dec.pos.copy_(state["pos"])
        dec.step_persistent()
        return {"logits": dec.logits, "k_first": dec.kc[0], "v_first": dec.vc[0],
                "k_last": dec.kc[-1], "v_last": dec.vc[-1]}
    w = state["w"]
    cb = build_kmeans_codebook(w.reshape(-1))
    idx = chunked_assign(w.reshape(-1), cb).view(w.shape)
    pos, val = find_outliers_percentile(w)
    scale, offset = fit_group_affine(w, idx, cb, GROUP, pos)
    return {"codebook": cb, "indices": idx, "positions": pos, "values": val, "scale": scale,
            "offset": offset}


# ------------------------------------------------------------------- what it takes
def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": _bytes(n, k, case["fmt"], case.get("affine", True)) + m * (n + k) * e,
                "flops": 2 * m * n * k}
    if kind == "layer":
        m, s = case["m"], _layer_shapes(SHAPES[case["shape"]])
        return {"bytes": sum(_bytes(n, k) + 2 * m * (n + k) for n, k in s.values()),
                "flops": sum(2 * m * n * k for n, k in s.values())}
    if kind == "scan":
        b, L, H, P, N, G = (case[k] for k in ("batch", "len", "heads", "p", "state", "groups"))
        return {"bytes": b * L * (H * P * 6 + H * 4 + 4 * G * N)
                + (2 if case["h0"] else 1) * 4 * b * H * P * N,
                "flops": 5 * b * L * H * P * N}
    if kind in ("mixer", "mixer_step"):
        b, L = case["batch"], case.get("len", 1)
        H, P, N, dm = case["heads"], case["p"], case["state"], case["d_model"]
        inner, width = H * P, 2 * H * P + 2 * N + H
        states = 4 * b * (4 * (inner + 2 * N) + H * P * N) * (2 if kind == "mixer_step" else 1)
        return {"bytes": _bytes(width, dm) + _bytes(dm, inner) + 4 * b * L * dm + states,
                "flops": b * L * (2 * width * dm + 2 * dm * inner + 5 * H * P * N)}
    if kind == "moe":
        T, E, h, i, k = (case[x] for x in ("tokens", "experts", "hidden", "inter", "top_k"))
        used = E * (1.0 - (1.0 - k / E) ** T)   # experts that random routing reaches
        return {"bytes": used * 3 * _bytes(i, h) + 4 * T * h + 4 * T * E,
                "flops": 6 * T * k * h * i}
    if kind == "decoder":
        c = SHAPES[case["shape"]]
        s = _layer_shapes(c)
        kv = 4 * c.n_kv_heads * c.head_dim * (case["pos"] + 1)
        return {"bytes": case["layers"] * (sum(_bytes(n, k) for n, k in s.values()) + kv)
                + c.vocab * (c.hidden * 2 + 4),
                "flops": 2 * case["layers"] * sum(n * k for n, k in s.values())
                + 2 * c.vocab * c.hidden}
    n = case["rows"] * case["cols"]
    return {"bytes": 5 * n + 8 * n // GROUP + 12 * (n // 500), "flops": 20 * n}


def tolerance(case):
    # about four times what the paths show against exact(): 16-bit results carry one rounding
    # of the output and one of the weights (bf16 2.4e-3, fp16 2.2e-4; experts and the mixer a
    # few more, 4.8e-3), fp32 ones the order of their sums (up to 8.8e-7), the scan its operands'
    # 16-bit mantissas (2.5e-6), a decoder step the roundings of every layer before (3.2e-3)
    kind = case["kind"]
    if kind == "encode":
        return "exact"
    if kind == "scan":
        return {"rel": 1e-5}
    if kind == "decoder":
        return {"rel": 0.013}
    if kind == "linear" and case["dtype"] == "f32":
        return {"rel": 4e-6}
    if case["dtype"] == "f16":
        return {"rel": 0.001 if kind in ("linear", "layer") else 0.002}
    return {"rel": 0.01}


# ------------------------------------------------------------------- in 64 bits
def _scan64(h, dt, A, x, B, C, D):
    rep = dt.shape[2] // B.shape[2]
    dt, A, x, D = dt.double(), A.double(), x.double(), D.double().reshape(-1, 1)
    B, C = (t.double().repeat_interleave(rep, dim=2) for t in (B, C))
    ys = []
    for t in range(dt.shape[1]):
        h = h * torch.exp(A * dt[:, t])[..., None, None]
        h = h + (dt[:, t, :, None] * x[:, t]).unsqueeze(-1) * B[:, t].unsqueeze(2)
        ys.append((h @ C[:, t].unsqueeze(-1)).squeeze(-1) + D * x[:, t])
    return torch.stack(ys, dim=1), h


def _mixer64(case, m, x, state):
    one = case["kind"] == "mixer_step"
    H, P, N = case["heads"], case["p"], case["state"]
    inner = H * P
    proj = _apply(x.unsqueeze(1) if one else x, m["in"])
    b, L, _ = proj.shape
    gate, xbc, dt = proj.split([inner, inner + 2 * N, H], dim=-1)
    if one:
        past = torch.cat([state[0].double()[:, :, 1:], xbc.transpose(1, 2)], dim=2)
        h = state[1].double()
    else:
        past = torch.nn.functional.pad(xbc.transpose(1, 2), (3, 0))
        h = torch.zeros(b, H, P, N, dtype=torch.float64, device=DEV)
    conv = torch.stack([(past[:, :, t:t + 4] * m["conv_w"].double()).sum(-1)
                        for t in range(L)], dim=1) + m["conv_b"].double()
    xs, B, C = torch.nn.functional.silu(conv).split([inner, N, N], dim=-1)
    dt = torch.nn.functional.softplus(dt + m["dt_bias"].double())
    y, h = _scan64(h, dt, -torch.exp(m["A_log"].double()), xs.reshape(b, L, H, P),
                   B.reshape(b, L, 1, N), C.reshape(b, L, 1, N), m["D"])
    z = y.reshape(b, L, inner) * torch.nn.functional.silu(gate)
    z = z * torch.rsqrt(z.square().mean(-1, keepdim=True) + 1e-5) * m["norm"].double()
    out = _apply(z, m["out"])
    return {"y": out[:, 0] if one else out, "conv": past[:, :, -4:].contiguous(), "ssm": h}


def _expert64(L):
    n, k = L["indices"].shape
    return {"codebook": L["codebook"], "indices": L["indices"], "n": n, "k": k, "bias": None,
            "scale": L["group_scale"], "offset": L["group_offset"],
            "pos": L["sidecar_positions"], "val": L["sidecar_values"]}


def _moe64(case, banks, x, logits):
    w, ids = torch.softmax(logits.double(), dim=-1).topk(case["top_k"], dim=-1)
    y = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    for e in range(case["experts"]):
        t, s = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            g, u = (_apply(x[t], _expert64(banks[b][e])) for b in ("gate", "up"))
            o = _apply(torch.nn.functional.silu(g) * u, _expert64(banks["down"][e]))
            y.index_add_(0, t, o * w[t, s].unsqueeze(1))
    return y


def _decoder64(case, seed):
    cfg, layers, embed, norm, tok, pos = _decoder_inputs(case, seed)
    D, nh, nkv, p = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads, case["pos"]
    rms = lambda v, w: (v * torch.rsqrt(v.square().mean(-1, keepdim=True) + cfg.rms_eps)
                        * w.double())
    ang = p * torch.exp(-math.log(cfg.rope_theta) * torch.arange(0, D, 2, device=DEV).double() / D)
    cos, sin = torch.cat([ang, ang]).cos(), torch.cat([ang, ang]).sin()
    rope = lambda v: v * cos + torch.cat([-v[..., D // 2:], v[..., :D // 2]], dim=-1) * sin
    x = embed[tok.long()].double()
    caches = {}
    for li, L in enumerate(layers):
        h = rms(x, L["in_norm"])
        q, k, v = (_apply(h, L[n]) for n in "qkv")
        q, k, v = rope(q.view(nh, D)), rope(k.view(nkv, D)), v.view(nkv, D)
        K, V = (torch.cat([c.double(), t.unsqueeze(0)]) for c, t in zip(L["kv"], (k, v)))
        for end, at in (("first", 0), ("last", len(layers) - 1)):
            if li == at:
                for n, c in (("k_", K), ("v_", V)):
                    full = torch.zeros(cfg.max_seq, nkv, D, dtype=torch.float64, device=DEV)
                    full[:p + 1] = c
                    caches[n + end] = full
        K, V = (c.repeat_interleave(nh // nkv, dim=1) for c in (K, V))
        a = torch.softmax((K * q).sum(-1) / math.sqrt(D), dim=0)
        x = x + _apply((a.unsqueeze(-1) * V).sum(0).reshape(1, -1), L["o"])
        h = rms(x, L["post_norm"])
        g, u = _apply(h, L["gate"]), _apply(h, L["up"])
        x = x + _apply(torch.nn.functional.silu(g) * u, L["down"])
    h = rms(x, norm).squeeze(0)
    logits = torch.cat([part.double() @ h for part in embed.split(32768)])
    return {"logits": logits, **caches}


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        return _apply(x, w)
    if kind == "layer":
        ws, xs = _layer_inputs(case, seed)
        return {p: _apply(xs[_LAYER_X[p]], w) for p, w in ws.items()}
    if kind == "scan":
        s = _scan_inputs(case, seed)
        h = s["h0"].double() if s["h0"] is not None else torch.zeros(
            case["batch"], case["heads"], case["p"], case["state"], dtype=torch.float64,
            device=DEV)
        y, h = _scan64(h, s["dt"], s["A"], s["x"], s["B"], s["C"], s["D"])
        return {"y": y, "h": h}
    if kind in ("mixer", "mixer_step"):
        return _mixer64(case, *_mixer_inputs(case, seed))
    if kind == "moe":
        return _moe64(case, *_moe_inputs(case, seed))
    if kind == "decoder":
        return _decoder64(case, seed)
    return None   # the encoder's results are whole numbers or must be equal bit for bit
