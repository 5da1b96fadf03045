"""Cases of ordinary use of this framework, for timing and for comparing outputs.

A case is a dict of plain values whose "kind" says which path it takes:

* gemv    the drop-in host-pointer product of the reference (q4_k_gemv! ..):
          numpy arrays in and out, one token;
* gemm    one device product (gemm_q_ex), packed or GGUF layout;
* layer   one decoder layer's matmuls with plain calls: RMSNorm + [q; k; v],
          o added into the residual, the fused MLP (no attention: q feeds o);
* step    a whole verify forward of chained matmuls, the LM head and the
          accept, captured once in a HIP graph and replayed, as a serving
          loop runs it;
* accept  rejection-sampling verify of a batch of steps over full-vocabulary
          logits (standard or reference mode), or the greedy verify;
* tree    the accept walk over a draft tree;
* sample  the draft-side sampler;
* pack    the one-time repacking of a weight matrix at model load.

Weights are random GGUF blocks whose dequantized entries have mean ~0 and
standard deviation ~gain / sqrt(K), as trained projections have, so that
activations keep their size from layer to layer. Logits of the samplers fall
off with the rank as a language model's do (exponent 1.6, noise on top).
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "inferno.jl_amd"))

import inferno_hip as ih  # noqa: E402
from inferno_hip import quantized_kernels as qk  # noqa: E402

Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K}
BLOCK = {"q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}  # elements, bytes
VOCAB = 151936
EPS = 1e-6
T_ACCEPT = 0.8


def listed():
    return [
        # the smallest call: the reference's own GEMV signature, one token, host
        # arrays (a small model's projection; the time is latency)
        {"name": "gemv_host_q4k_3072x1024", "kind": "gemv", "qtype": "q4_k", "n": 3072, "k": 1024},
        # a ragged product straight from a GGUF file's bytes, no repacking: a
        # Q8_0 adapter-like matrix, a row count and a K off every tile, more
        # tokens than one token tile
        {"name": "gemm_q8_0_2050x2080_m11", "kind": "gemm", "qtype": "q8_0", "m": 11, "n": 2050, "k": 2080,
         "prec": "f32", "packed": False, "act": "plain", "gain": 1.0},
        # a verify batch (1 accepted + 4 drafted tokens) through a layer of a small model
        {"name": "layer_h2048_m5", "kind": "layer", "proj": "q4_k", "m": 5, "h": 2048, "f": 6144, "prec": "f32"},
        # the same through a layer of a 9B-class model
        {"name": "layer_h4096_m5", "kind": "layer", "proj": "q4_k", "m": 5, "h": 4096, "f": 12288, "prec": "f32"},
        # a 64-node draft tree through that layer, half-precision operands (the default at 16 tokens and more)
        {"name": "layer_h4096_m64", "kind": "layer", "proj": "q4_k", "m": 64, "h": 4096, "f": 12288, "prec": "auto"},
        # the LM head over six verify steps' rows at once, fp32-accurate
        {"name": "lm_head_151936x2048_m30", "kind": "gemm", "qtype": "q6_k", "m": 30, "n": VOCAB, "k": 2048,
         "prec": "f32", "packed": True, "act": "plain", "gain": 2.5},
        # the largest: a full verify step of a 9B-class model, replayed from a graph
        {"name": "verify_step_32x4096_m5", "kind": "step", "layers": 32, "m": 5, "h": 4096, "f": 12288, "v": VOCAB},
        # 64 concurrent sequences' accept, k = 4
        {"name": "accept_s64_k4", "kind": "accept", "mode": "standard", "steps": 64, "k": 4, "v": VOCAB},
        # the accept walk over a 64-node tree
        {"name": "tree_accept_n64", "kind": "tree", "n": 64, "v": VOCAB},
        # drafting for 64 sequences with a nucleus
        {"name": "sample_r64_top_p", "kind": "sample", "rows": 64, "v": VOCAB, "t": 0.8, "top_k": 0, "top_p": 0.9,
         "min_p": 0.0},
        # drafting one token with the usual interactive settings
        {"name": "sample_r1_top_k_p", "kind": "sample", "rows": 1, "v": VOCAB, "t": 0.7, "top_k": 40, "top_p": 0.95,
         "min_p": 0.0},
        # model load: the down projection of a 9B-class model brought to the packed layout
        {"name": "pack_q6k_4096x12288", "kind": "pack", "qtype": "q6_k", "n": 4096, "k": 12288},
    ]


def _spread(rng, lo, hi, step=1):
    """A whole number in [lo, hi], spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    kind = rng.choice(["gemv", "gemm", "gemm", "layer", "layer", "step", "accept", "tree", "sample", "sample", "pack"])
    qtype = rng.choice(list(TYPES))
    unit = BLOCK[qtype][0]
    if kind == "gemv":
        return {"kind": kind, "qtype": qtype, "n": _spread(rng, 256, 12288), "k": _spread(rng, 512, 8192, unit)}
    if kind == "gemm":
        prec = rng.choice(["f32", "half", "auto"])
        n = _spread(rng, 200, 32000)
        if qtype == "q6_k" and rng.random() < 0.4:
            n = VOCAB
        return {"kind": kind, "qtype": qtype, "m": _spread(rng, 1, 32 if prec == "f32" else 64), "n": n,
                "k": _spread(rng, 1024, 4096 if n == VOCAB else 12288, unit), "prec": prec,
                "packed": rng.random() < 0.75, "act": rng.choice(["plain", "rmsnorm"]), "gain": 2.5 if n == VOCAB else 1.0}
    if kind == "layer":
        h = _spread(rng, 1024, 5120, 1024)
        m = _spread(rng, 1, 64)
        return {"kind": kind, "proj": rng.choice(["q4_k", "q4_k", "q5_k"]), "m": m, "h": h,
                "f": int(rng.uniform(2.5, 3.5) * h) // 256 * 256, "prec": "auto" if m >= 16 else "f32"}
    if kind == "step":
        m = rng.randint(2, 8)
        h = rng.choice([1024, 2048, 3072, 4096])
        return {"kind": kind, "layers": _spread(rng, 2, 24), "m": m, "h": h, "f": int(rng.uniform(2.5, 3.0) * h) // 256 * 256,
                "v": _spread(rng, 32000, VOCAB)}
    if kind == "accept":
        return {"kind": kind, "mode": rng.choice(["standard", "standard", "reference", "greedy"]),
                "steps": _spread(rng, 1, 64), "k": rng.randint(1, 8), "v": _spread(rng, 32000, 262144)}
    if kind == "tree":
        return {"kind": kind, "n": rng.randint(6, 64), "v": _spread(rng, 32000, 262144)}
    if kind == "sample":
        setting = rng.choice(["greedy", "plain", "top_k", "top_p", "min_p", "top_k_p", "top_p_min_p", "big_k"])
        return {"kind": kind, "rows": _spread(rng, 1, 64), "v": _spread(rng, 32000, 262144),
                "t": 0.0 if setting == "greedy" else rng.choice([0.7, 0.8, 1.0]),
                "top_k": rng.choice([20, 40, 50]) if setting in ("top_k", "top_k_p") else 500 if setting == "big_k" else 0,
                "top_p": rng.choice([0.9, 0.95]) if "top_p" in setting or setting == "top_k_p" else 1.0,
                "min_p": 0.05 if "min_p" in setting else 0.0}
    return {"kind": "pack", "qtype": qtype, "n": _spread(rng, 512, 24576), "k": _spread(rng, 1024, 12288, unit)}


# ---------------------------------------------------------------- inputs

def _device(case):
    return "cpu" if case["kind"] == "gemv" else "cuda"


def _gen(seed, case):
    return torch.Generator(device=_device(case)).manual_seed(int(seed) * 7919 + 17)


def _bytes(g, n, dev):
    return torch.randint(-2**63, 2**63 - 1, ((n + 7) // 8,), generator=g, device=dev, dtype=torch.int64).view(torch.uint8)[:n]


def _k4_scales(sc, mn):
    """The 12 packed bytes of eight 6-bit scales and mins (GGUF Q4_K / Q5_K)."""
    lo = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    mid = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    hi = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return torch.cat([lo, mid, hi], 1)


def _fp16_bytes(v):
    return v.to(torch.float16).view(-1, 1).view(torch.uint8)


def _weights(g, qtype, n, k, gain, dev):
    """An [n x k] matrix of GGUF blocks (uint8), entries of mean ~0 and sd ~gain / sqrt(k)."""
    qe, nb = BLOCK[qtype]
    blocks = n * (k // qe)
    out = torch.empty((blocks, nb), dtype=torch.uint8, device=dev)
    sd = gain / math.sqrt(k)
    at = 0
    while at < blocks:  # (in parts: the temporaries stay small)
        b = min(blocks - at, 1 << 20)
        o = out[at:at + b]
        u = 0.8 + 0.4 * torch.rand(b, generator=g, device=dev)
        if qtype in ("q4_k", "q5_k"):
            sc = (32 + (_bytes(g, b * 8, dev).view(b, 8) & 31)).to(torch.uint8)
            mid = 7.5 if qtype == "q4_k" else 15.5
            d = u * (sd / (48.5 * (4.61 if qtype == "q4_k" else 9.23)))
            o[:, 0:2] = _fp16_bytes(d)
            o[:, 2:4] = _fp16_bytes(mid * d)
            o[:, 4:16] = _k4_scales(sc, sc)
            o[:, 16:] = _bytes(g, b * (nb - 16), dev).view(b, nb - 16)
        elif qtype == "q6_k":
            o[:, :192] = _bytes(g, b * 192, dev).view(b, 192)
            r = _bytes(g, b * 16, dev).view(b, 16)
            sc = (32 + (r & 31).to(torch.int16)) * (1 - 2 * (r >> 7).to(torch.int16))
            o[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
            o[:, 208:210] = _fp16_bytes(u * (sd / (48.5 * 18.5)))
        else:
            o[:, 0:2] = _fp16_bytes(u * (sd / 73.3))
            q = _bytes(g, b * 32, dev).view(b, 32)
            o[:, 2:] = torch.where(q == 128, torch.zeros_like(q), q)
        at += b
    return out.view(-1)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=g.device)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=g.device)


def _lm_logits(g, rows, v):
    """Rows of logits as a language model gives them: -1.6 log(rank), noise, a random order."""
    base = -1.6 * torch.log(torch.arange(1, v + 1, device=g.device, dtype=torch.float32))
    out = torch.empty((rows, v), device=g.device)
    for r in range(rows):
        out[r] = base[torch.randperm(v, generator=g, device=g.device)]
    return out + 0.7 * _normal(g, rows, v)


def _draft(g, target, t):
    """Draft logits around the target's and tokens drawn from their softmax at t."""
    drf = target + 1.5 * _normal(g, *target.shape)
    p = torch.softmax(drf / t, -1).view(-1, drf.shape[-1])
    tok = torch.multinomial(p, 1, generator=g).view(drf.shape[:-1]).to(torch.int32)
    return drf, tok


def _flags(case, packed=True):
    return {"f32": ih.GEMM_F32, "half": ih.GEMM_HALF, "auto": ih.GEMM_AUTO}[case["prec"]] | (ih.GEMM_PACKED if packed else 0)


def _layer_shapes(case):
    h = case["h"]
    nq, nkv = h, h // 4
    return h, nq, nkv, case["f"]


def _layer_weights(g, case, proj):
    """One layer's GGUF matrices and norm weights: qkv, o, gate_up, down, and the two norms."""
    h, nq, nkv, f = _layer_shapes(case)
    return {"qkv": _weights(g, proj, nq + 2 * nkv, h, 1.0, "cuda"), "o": _weights(g, proj, h, nq, 0.5, "cuda"),
            "gu": _weights(g, proj, 2 * f, h, 1.0, "cuda"), "down": _weights(g, "q6_k", h, f, 0.8, "cuda"),
            "attn_norm": 1.0 + 0.1 * _normal(g, h), "ffn_norm": 1.0 + 0.1 * _normal(g, h)}


def _inputs(case, seed):
    """The inputs of a case, from the seed alone (the step's layers: _step_layers)."""
    g, kind = _gen(seed, case), case["kind"]
    if kind in ("gemv", "gemm"):
        dev, m = _device(case), case.get("m", 1)
        d = {"w": _weights(g, case["qtype"], case["n"], case["k"], case.get("gain", 1.0), dev),
             "x": _normal(g, m, case["k"])}
        if case.get("act") == "rmsnorm":
            d["norm"] = 1.0 + 0.1 * _normal(g, case["k"])
        return d
    if kind == "layer":
        d = _layer_weights(g, case, case["proj"])
        d["x"] = _normal(g, case["m"], case["h"])
        return d
    if kind == "pack":
        return {"w": _weights(g, case["qtype"], case["n"], case["k"], 1.0, "cuda")}
    if kind == "accept":
        s, k, v = case["steps"], case["k"], case["v"]
        tgt = _lm_logits(g, s * (k + 1), v).view(s, k + 1, v)
        drf, tok = _draft(g, tgt[:, :k].contiguous(), T_ACCEPT)
        if case["mode"] == "greedy":  # a draft that mostly agrees with the target's argmax
            tok = torch.where(_uniform(g, s, k) < 0.8, tgt[:, :k].argmax(-1).to(torch.int32), tok)
        return {"tgt": tgt, "drf": drf, "tok": tok, "ua": _uniform(g, s, k), "ur": _uniform(g, s), "ub": _uniform(g, s)}
    if kind == "tree":
        n, v = case["n"], case["v"]
        tgt = _lm_logits(g, n, v)
        drf = tgt + 1.5 * _normal(g, n, v)
        parent = torch.tensor([-1] + [(i - 1) // 4 for i in range(1, n)], dtype=torch.int32, device="cuda")
        p = torch.softmax(drf[parent.long().clamp(min=0)], -1)
        return {"tgt": tgt, "drf": drf, "tok": torch.multinomial(p, 1, generator=g).view(n).to(torch.int32),
                "parent": parent, "u": _uniform(g, n)}
    if kind == "sample":
        return {"logits": _lm_logits(g, case["rows"], case["v"]), "u": _uniform(g, case["rows"])}
    m, k, v = case["m"], case["m"] - 1, case["v"]  # step
    return {"x": _normal(g, m, case["h"]), "drf": 2.5 * _normal(g, 1, k, v),
            "tok": torch.randint(0, v, (1, k), generator=g, device="cuda", dtype=torch.int32),
            "ua": _uniform(g, 1, k), "ur": _uniform(g, 1), "ub": _uniform(g, 1), "norm": 1.0 + 0.1 * _normal(g, case["h"])}


def _step_layers(case, seed):
    """The step's layers one after the other, then the LM head."""
    g = _gen(seed + 1000003, case)
    for _ in range(case["layers"]):
        yield _layer_weights(g, case, "q4_k")
    yield {"head": _weights(g, "q6_k", case["v"], case["h"], 2.5, "cuda")}


# ---------------------------------------------------------------- the calls

def prepare(case, seed):
    kind, s = case["kind"], _inputs(case, seed)
    s["case"] = case
    if kind == "gemv":
        s["w"], s["x"] = s["w"].numpy(), s["x"].view(-1).numpy()
        s["out"] = np.zeros(case["n"], dtype=np.float32)
    elif kind == "gemm":
        qt, m, n, k = TYPES[case["qtype"]], case["m"], case["n"], case["k"]
        s["flags"] = _flags(case, case["packed"])
        if case["packed"]:
            s["w"] = ih.pack_weights(qt, s["w"], n, k)
        s["out"] = torch.empty((m, n), device="cuda")
        s["ws"] = torch.empty(qk.gemm_ws_bytes(qt, m, n, k, s["flags"]), dtype=torch.uint8, device="cuda")
    elif kind == "layer":
        _prepare_layer(case, s)
    elif kind == "step":
        _prepare_step(case, seed, s)
    elif kind == "accept" and case["mode"] != "greedy":
        nb = C.c_size_t()
        ih._lib.check(ih.load().ihip_spec_accept_ex_ws_bytes(case["steps"], case["k"], case["v"], 0, 1.0, 0.0, C.byref(nb)))
        s["ws"] = torch.empty(max(nb.value, 16), dtype=torch.uint8, device="cuda")
        s["out_tok"] = torch.zeros((case["steps"], case["k"] + 1), dtype=torch.int32, device="cuda")
        s["out_n"] = torch.zeros(case["steps"], dtype=torch.int32, device="cuda")
    elif kind == "sample":
        s["ws"] = torch.empty(ih.sample_ws_bytes(case["rows"], case["v"]), dtype=torch.uint8, device="cuda")
        s["out"] = torch.empty(case["rows"], dtype=torch.int32, device="cuda")
    elif kind == "pack":
        s["out"] = torch.empty(ih.packed_bytes(TYPES[case["qtype"]], case["n"], case["k"]), dtype=torch.uint8, device="cuda")
    return s


def _prepare_layer(case, s):
    h, nq, nkv, f = _layer_shapes(case)
    qt, m, fl = TYPES[case["proj"]], case["m"], _flags(case)
    for key, t, n, k in (("qkv", qt, nq + 2 * nkv, h), ("o", qt, h, nq), ("gu", qt, 2 * f, h), ("down", Q6_K, h, f)):
        s[key] = ih.pack_weights(t, s[key], n, k)
    s["flags"], s["res"] = fl, torch.empty((m, h), device="cuda")
    s["qkv_out"] = torch.empty((m, nq + 2 * nkv), device="cuda")
    ws = max(qk.gemm_ws_bytes(qt, m, nq + 2 * nkv, h, fl), qk.gemm_ws_bytes(qt, m, h, nq, fl | ih.GEMM_ACCUM),
             ih.mlp_ws_bytes(qt, Q6_K, m, h, f, fl))
    s["ws"] = torch.empty(ws, dtype=torch.uint8, device="cuda")


def _run_layer(case, s):
    h, nq, nkv, f = _layer_shapes(case)
    qt, fl, x, qkv = TYPES[case["proj"]], s["flags"], s["res"], s["qkv_out"]
    x.copy_(s["x"])  # (the residual is updated in place)
    ih.gemm_q_ex(qt, s["qkv"], x, nq + 2 * nkv, h, act=ih.ACT_RMSNORM, norm_w=s["attn_norm"], eps=EPS, flags=fl,
                 out=qkv, ws=s["ws"])
    ih.gemm_q_ex(qt, s["o"], qkv[:, :nq], h, nq, flags=fl | ih.GEMM_ACCUM, out=x, ws=s["ws"])
    ih.mlp_forward_(qt, s["gu"], Q6_K, s["down"], x, h, f, norm_w=s["ffn_norm"], eps=EPS, flags=fl, ws=s["ws"])
    return {"qkv": qkv, "x": x}


def _prepare_step(case, seed, s):
    """The chained verify step and its graph (at most 8 tokens, fp32-accurate)."""
    h, nq, nkv, f = _layer_shapes(case)
    m, k, v = case["m"], case["m"] - 1, case["v"]
    layers = []
    for w in _step_layers(case, seed):
        if "head" in w:
            head = ih.pack_weights(Q6_K, w["head"], v, h)
            break
        layers.append({"qkv": ih.pack_weights(Q4_K, w["qkv"], nq + 2 * nkv, h), "o": ih.pack_weights(Q4_K, w["o"], h, nq),
                       "gu": ih.pack_weights_gated(Q4_K, w["gu"], f, h), "down": ih.pack_weights(Q6_K, w["down"], h, f),
                       "attn_norm": w["attn_norm"], "ffn_norm": w["ffn_norm"]})
    fl = ih.GEMM_F32 | ih.GEMM_PACKED
    nb = max(qk.gemm_ws_bytes(Q4_K, m, nq + 2 * nkv, h, fl), qk.gemm_ws_bytes(Q4_K, m, 2 * f, h, fl),
             qk.gemm_ws_bytes(Q4_K, m, h, nq, fl), qk.gemm_ws_bytes(Q6_K, m, h, f, fl), qk.gemm_ws_bytes(Q6_K, m, v, h, fl))
    ws, ws_o, ws_down = (torch.zeros(nb, dtype=torch.uint8, device="cuda") for _ in range(3))
    x, qkv = torch.empty((m, h), device="cuda"), torch.empty((m, nq + 2 * nkv), device="cuda")
    hid, logits = torch.empty((m, f), device="cuda"), torch.empty((m, v), device="cuda")
    op_q, ts_q, _ = ih.chain_buffers(nq)
    op_x, ts_x, ssq_x = ih.chain_buffers(h, ssq=True)
    op_h, _, _ = ih.chain_buffers(f, tiles_per_unit=32)
    o_in, gu_in = ih.chain_in(op_q, ts_q, 16), ih.chain_in(op_x, ts_x, 16, tile_ssq=ssq_x, eps=EPS)
    down_in = ih.chain_in(op_h, None, 32)
    qkv_out = ih.chain_out(ih.EPI_STATS, qkv, Q4_K, op_q, ts_q, stat_rows=nq)
    o_out = [ih.chain_out(ih.EPI_RESID, x, Q4_K, op_x, ts_x, norm_w=lw["ffn_norm"], tile_ssq=ssq_x) for lw in layers]
    gu_out = ih.chain_out(ih.EPI_GATE, hid, Q6_K, op_h)
    parts = ih.gemm_partials(Q6_K, m, h, f, fl, ws_down)
    nws = C.c_size_t()
    ih._lib.check(ih.load().ihip_spec_accept_ex_ws_bytes(1, k, v, 0, 1.0, 0.0, C.byref(nws)))
    acc_ws = torch.empty(max(nws.value, 16), dtype=torch.uint8, device="cuda")
    out_tok = torch.zeros((1, k + 1), dtype=torch.int32, device="cuda")
    out_n = torch.zeros(1, dtype=torch.int32, device="cuda")

    def step():
        x.copy_(s["x"])
        for i, lw in enumerate(layers):
            ih.gemm_q_chain(Q4_K, lw["qkv"], nq + 2 * nkv, h, m, x=x, act=ih.ACT_RMSNORM, norm_w=lw["attn_norm"], eps=EPS,
                            add=parts if i else None, ws=ws, cout=qkv_out)
            ih.gemm_q_chain(Q4_K, lw["o"], h, nq, m, cin=o_in, ws=ws_o, cout=o_out[i])
            ih.gemm_q_chain(Q4_K, lw["gu"], 2 * f, h, m, cin=gu_in, ws=ws, cout=gu_out)
            ih.gemm_q_chain(Q6_K, lw["down"], h, f, m, cin=down_in, flags=fl | ih.GEMM_DEFER, ws=ws_down)
        ih.gemm_q_ex(Q6_K, head, x, v, h, act=ih.ACT_RMSNORM, norm_w=s["norm"], eps=EPS, flags=fl, out=logits, ws=ws,
                     add=parts)
        ih.spec_accept(logits.view(1, m, v), s["drf"], s["tok"], T_ACCEPT, s["ua"], s["ur"], s["ub"], out_tok=out_tok,
                       out_n=out_n, ws=acc_ws)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    s["graph"], s["keep"] = graph, (layers, head, ws, ws_o, ws_down, x, qkv, hid, op_q, ts_q, op_x, ts_x, ssq_x, op_h,
                                    acc_ws, o_in, gu_in, down_in, qkv_out, o_out, gu_out)
    s["outputs"] = {"logits": logits, "x": x, "tok": out_tok, "n": out_n}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        qk.GEMV_BY_QTYPE[TYPES[case["qtype"]]](s["out"], s["w"], s["x"], case["k"], case["n"])
        return s["out"]
    if kind == "gemm":
        norm = s.get("norm")
        return ih.gemm_q_ex(TYPES[case["qtype"]], s["w"], s["x"], case["n"], case["k"],
                            act=ih.ACT_PLAIN if norm is None else ih.ACT_RMSNORM, norm_w=norm, eps=EPS, flags=s["flags"],
                            out=s["out"], ws=s["ws"])
    if kind == "layer":
        return _run_layer(case, s)
    if kind == "step":
        s["graph"].replay()
        return s["outputs"]
    if kind == "accept":
        if case["mode"] == "greedy":
            return ih.greedy_verify(s["tgt"], s["tok"])
        mode = ih.MODE_STANDARD if case["mode"] == "standard" else ih.MODE_REFERENCE
        s["out_tok"].zero_()  # (a step writes the tokens it returns and leaves the rest of its row)
        return ih.spec_accept(s["tgt"], s["drf"], s["tok"], T_ACCEPT, s["ua"], s["ur"], s["ub"], mode=mode,
                              out_tok=s["out_tok"], out_n=s["out_n"], ws=s["ws"])
    if kind == "tree":
        return ih.tree_accept(s["tgt"], s["drf"], s["tok"], s["parent"], 1.0, s["u"])
    if kind == "sample":
        return ih.softmax_sample(s["logits"], s["u"], temperature=case["t"], top_p=case["top_p"], top_k=case["top_k"],
                                 min_p=case["min_p"], out=s["out"], ws=s["ws"])
    return ih.pack_weights(TYPES[case["qtype"]], s["w"], case["n"], case["k"], out=s["out"])


# ---------------------------------------------------------------- what a pass needs

def _matrix(qtype, n, k):
    qe, nb = BLOCK[qtype]
    return n * (k // qe) * nb


def _layer_work(case, proj):
    h, nq, nkv, f = _layer_shapes(case)
    m = case["m"]
    params = h * (nq + 2 * nkv) + h * nq + 3 * h * f
    return (_matrix(proj, nq + 2 * nkv, h) + _matrix(proj, h, nq) + _matrix(proj, 2 * f, h) + _matrix("q6_k", h, f) + 8 * h,
            2 * m * params)


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        m, n, k = case.get("m", 1), case["n"], case["k"]
        return {"bytes": _matrix(case["qtype"], n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "layer":
        nb, fl = _layer_work(case, case["proj"])
        h, nq, nkv, _ = _layer_shapes(case)
        return {"bytes": nb + 4 * case["m"] * (2 * h + nq + 2 * nkv), "flops": fl}
    if kind == "step":
        nb, fl = _layer_work(case, "q4_k")
        m, v, h = case["m"], case["v"], case["h"]
        return {"bytes": case["layers"] * nb + _matrix("q6_k", v, h) + 4 * (m * (2 * h + v) + (m - 1) * v),
                "flops": case["layers"] * fl + 2 * m * v * h}
    if kind == "accept":
        s, k, v = case["steps"], case["k"], case["v"]
        rows = s * (k + 1) + (0 if case["mode"] == "greedy" else s * k)
        return {"bytes": 4 * rows * v, "flops": (2 if case["mode"] == "greedy" else 8) * rows * v}
    if kind == "tree":
        return {"bytes": 8 * case["n"] * case["v"], "flops": 16 * case["n"] * case["v"]}
    if kind == "sample":
        return {"bytes": 4 * case["rows"] * case["v"], "flops": 8 * case["rows"] * case["v"]}
    qe, nb = BLOCK[case["qtype"]]
    n, k = case["n"], case["k"]
    return {"bytes": _matrix(case["qtype"], n, k) + (n + 15) // 16 * 16 * ((k + 255) // 256) * (256 // qe) * nb, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind in ("accept", "tree", "sample"):
        return {"rel": 0.0, "differ": 0.01}  # (whole values: the draws are exact but for ties)
    if kind == "gemv":
        return {"rel": 1e-6, "max": 1e-5}
    half = case.get("prec") == "half" or (case.get("prec") == "auto" and case["m"] >= 16)
    if kind == "gemm":
        return {"rel": 1.5e-3, "max": 1e-2} if half else {"rel": 1e-6, "max": 1e-5}
    if kind == "layer":
        return {"rel": 2e-3, "max": 2e-2} if half else {"rel": 1e-6, "max": 1e-5}
    return {"rel": 4e-6, "max": 4e-5, "differ": 0.01}


# ---------------------------------------------------------------- the same in 64 bits

def _dequant(qtype, w, n, k):
    """GGUF blocks -> [n, k] in float64, by the format's definition."""
    qe, nb = BLOCK[qtype]
    b = w.view(-1, nb)
    f16 = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if qtype in ("q4_k", "q5_k"):
        s = b[:, 4:16].to(torch.int16)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        qs = b[:, nb - 128:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32).to(torch.int16)  # sub-block 2c: low nibbles, 2c + 1: high
        if qtype == "q5_k":
            sh = torch.arange(8, device=w.device, dtype=torch.uint8).view(1, 8, 1)
            q = q + (((b[:, 16:48].view(-1, 1, 32) >> sh) & 1).to(torch.int16) << 4)
        out = (f16(0) * sc).unsqueeze(-1) * q.double() - (f16(2) * mn).unsqueeze(-1)
    elif qtype == "q6_k":
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # half, quarter (low l, low l + 32, high l, high l + 32), 32
        sh = torch.tensor([0, 2, 4, 6], device=w.device, dtype=torch.uint8).view(1, 1, 4, 1)
        q = (lo | (((qh >> sh) & 3) << 4)).to(torch.int16) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        out = (f16(208) * sc).unsqueeze(-1) * q.reshape(-1, 16, 16).double()
    else:
        out = f16(0) * b[:, 2:].contiguous().view(torch.int8).double()
    return out.reshape(n, k)


def _product(x, qtype, w, n, k):
    """x W^T in float64, a few thousand rows at a time."""
    qe, nb = BLOCK[qtype]
    row = k // qe * nb
    step = max(1, (1 << 24) // k)
    return torch.cat([x @ _dequant(qtype, w[r * row:min(n, r + step) * row], min(n, r + step) - r, k).t().contiguous()
                      for r in range(0, n, step)], 1)


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _layer64(x, w, case, proj):
    h, nq, nkv, f = _layer_shapes(case)
    qkv = _product(_norm64(x, w["attn_norm"]), proj, w["qkv"], nq + 2 * nkv, h)
    x = x + _product(qkv[:, :nq].contiguous(), proj, w["o"], h, nq)
    gu = _product(_norm64(x, w["ffn_norm"]), proj, w["gu"], 2 * f, h)
    return qkv, x + _product(torch.nn.functional.silu(gu[:, :f]) * gu[:, f:], "q6_k", w["down"], h, f)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("accept", "tree", "sample", "pack"):
        return None
    s = _inputs(case, seed)
    x = s["x"].double()
    if kind == "gemv":
        return _product(x, case["qtype"], s["w"], case["n"], case["k"]).view(-1).numpy()
    if kind == "gemm":
        if "norm" in s:
            x = _norm64(x, s["norm"])
        return _product(x, case["qtype"], s["w"], case["n"], case["k"])
    if kind == "layer":
        qkv, x = _layer64(x, s, case, case["proj"])
        return {"qkv": qkv, "x": x}
    for w in _step_layers(case, seed):
        if "head" in w:
            logits = _product(_norm64(x, s["norm"]), "q6_k", w["head"], case["v"], case["h"])
        else:
            x = _layer64(x, w, case, "q4_k")[1]
    return {"logits": logits, "x": x, "tok": None, "n": None}
