"""Performance cases: the work a program gives this framework, through its public entry points.

Five kinds of case:
  step   one token (or one small batch of rows) through the projections of some layers whose
         weights are resident: one qmm.gemm_batch call, as a decode loop issues it;
  proj   one projection (qmm.gemm), or a gate / up pair that shares its activations (qmm.gemm_batch);
  dequant  a packed matrix unpacked to floating point (qmm.dequantize);
  layer  a whole transformer layer over the device KV cache (TransformerLayer.forward_with_weights),
         decode (one row) or prefill (many rows);
  attn   grouped-query attention over the KV cache (qmm_gqa_attention_cached): a chunk of new rows
         against a long context.

Weights are Gaussian rows quantized to GGUF blocks on the GPU; activations are Gaussian.  `exact`
recomputes each case in float64 with plain torch from the same packed bytes.
"""

import itertools
import math
import os
import sys

import torch

_REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_REPO, "gfx1150-inference_amd"))

import gguf  # noqa: E402
import layer as layer_mod  # noqa: E402
import qmm  # noqa: E402

TYPES = {"f16": 1, "q4_0": 2, "q8_0": 8, "q4_k": 12, "q6_k": 14}
QK = {"f16": 1, "q4_0": 32, "q8_0": 32, "q4_k": 256, "q6_k": 256}
BB = {"f16": 2, "q4_0": 18, "q8_0": 34, "q4_k": 144, "q6_k": 210}
DTYPES = {"f16": torch.float16, "f32": torch.float32, "bf16": torch.bfloat16}
EB = {"f16": 2, "f32": 4, "bf16": 2}

# Layers' quantization mixes: (type of every projection but down, type of down).
MIXES = {"q4_k_m": ("q4_k", "q6_k"), "q4_k": ("q4_k", "q4_k"), "q6_k": ("q6_k", "q6_k"), "q8_0": ("q8_0", "q8_0"),
         "q4_0": ("q4_0", "q4_0")}


def listed():
    return [
        # the smallest call a program makes: one 4096 x 4096 Q4_0 projection of one fp32 row (the
        # basic benchmark configuration), where launch and call overhead count most
        {"name": "gemv_q4_0_4096_m1", "kind": "proj", "type": "q4_0", "mats": 1, "M": 1, "N": 4096, "K": 4096, "a": "f32", "c": "f32"},
        # single-user decode of an 8B Q4_K_M model: every projection of 4 layers, one token
        {"name": "step_8b_q4_k_m_m1", "kind": "step", "mix": "q4_k_m", "layers": 4, "M": 1, "hidden": 4096, "inter": 14336, "kv": 1024, "io": "f16"},
        # decode of a 70B Q4_K_M model for four users (or four speculated tokens)
        {"name": "step_70b_q4_k_m_m4", "kind": "step", "mix": "q4_k_m", "layers": 2, "M": 4, "hidden": 8192, "inter": 28672, "kv": 1024, "io": "f16"},
        # decode of an 8B Q8_0 model for a batch of eight
        {"name": "step_8b_q8_0_m8", "kind": "step", "mix": "q8_0", "layers": 4, "M": 8, "hidden": 4096, "inter": 14336, "kv": 1024, "io": "f16"},
        # the logits of one token: the 8B Q6_K output head, fp32 logits
        {"name": "lm_head_q6_k_m1", "kind": "proj", "type": "q6_k", "mats": 1, "M": 1, "N": 128256, "K": 4096, "a": "f16", "c": "f32"},
        # a short prompt, or a large decode batch, of a ragged row count on one 70B projection
        {"name": "proj_70b_q4_k_m31", "kind": "proj", "type": "q4_k", "mats": 1, "M": 31, "N": 28672, "K": 8192, "a": "f16", "c": "f16"},
        # prefill of 512 tokens: the 8B gate and up projections
        {"name": "gate_up_8b_q4_k_m512", "kind": "proj", "type": "q4_k", "mats": 2, "M": 512, "N": 14336, "K": 4096, "a": "f16", "c": "f16"},
        # prefill of a ragged 777 tokens: the 8B down projection of a Q8_0 model, fp32 activations
        {"name": "down_8b_q8_0_m777", "kind": "proj", "type": "q8_0", "mats": 1, "M": 777, "N": 4096, "K": 14336, "a": "f32", "c": "f32"},
        # unpacking a 70B projection for a dense product
        {"name": "dequant_70b_q4_k_f16", "kind": "dequant", "type": "q4_k", "N": 28672, "K": 8192, "c": "f16"},
        # one decode step of one 8B layer at a context of 4000 tokens
        {"name": "layer_8b_decode_ctx4000", "kind": "layer", "mix": "q4_k_m", "seq": 1, "pos": 4000, "hidden": 4096, "inter": 14336, "heads": 32,
         "kv_heads": 8, "head_dim": 128},
        # a 1023-token prompt through one 70B layer
        {"name": "layer_70b_prefill_1023", "kind": "layer", "mix": "q4_k_m", "seq": 1023, "pos": 0, "hidden": 8192, "inter": 28672, "heads": 64,
         "kv_heads": 8, "head_dim": 128},
        # a chunk of 40 new tokens (a follow-up question) attending over a long conversation
        {"name": "attn_8b_q40_ctx12000", "kind": "attn", "q": 40, "pos": 12000, "heads": 32, "kv_heads": 8, "head_dim": 128},
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer multiple of `step` in [lo, hi], spread over its logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step * 0.999)))
    return max(lo, min(hi, int(v) // step * step))


def _work_size(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _draw_one(rng):
    kind = rng.choice(["step", "step", "proj", "proj", "proj", "dequant", "layer", "layer", "attn", "attn"])
    if kind == "step":
        mix = rng.choice(sorted(MIXES))
        return {"kind": kind, "mix": mix, "layers": rng.choice([1, 2]), "M": _log_int(rng, 1, 16), "hidden": _log_int(rng, 2048, 8192, 256),
                "inter": _log_int(rng, 5632, 28672, 256), "kv": rng.choice([512, 1024, 2048]), "io": rng.choice(["f16", "f16", "f32"])}
    if kind == "proj":
        t = rng.choice(sorted(TYPES))
        k_step = 256 if QK[t] == 256 else 32
        return {"kind": kind, "type": t, "mats": rng.choice([1, 1, 2]), "M": _log_int(rng, 1, 1100), "N": _log_int(rng, 1000, 30000),
                "K": _log_int(rng, 2048, 16384, k_step), "a": rng.choice(["f16", "f16", "f32"]), "c": rng.choice(["f16", "f32"])}
    if kind == "dequant":
        t = rng.choice([t for t in sorted(TYPES) if t != "f16"])
        return {"kind": kind, "type": t, "N": _log_int(rng, 1000, 28672), "K": _log_int(rng, 2048, 8192, 256), "c": rng.choice(["f16", "f16", "bf16", "f32"])}
    head_dim = rng.choice([64, 128, 128])
    kv_heads = rng.choice([4, 8])
    heads = kv_heads * rng.choice([1, 4, 8])
    if kind == "layer":
        seq = rng.choice([1, 1, _log_int(rng, 2, 1000)])
        return {"kind": kind, "mix": rng.choice(sorted(MIXES)), "seq": seq, "pos": rng.choice([0, _log_int(rng, 1, 6000)]), "hidden": _log_int(rng, 2048, 8192, 256),
                "inter": _log_int(rng, 5632, 28672, 256), "heads": heads * 128 // head_dim, "kv_heads": kv_heads, "head_dim": head_dim}
    return {"kind": kind, "q": _log_int(rng, 1, 1024), "pos": _log_int(rng, 16, 16000), "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim}


def draw(rng):
    most = max(_work_size(c) for c in listed())
    while True:
        case = _draw_one(rng)
        if _work_size(case) <= most:
            return case


# ---- packed weights --------------------------------------------------------------------------
def _nibbles(lo, hi):
    return (lo | (hi << 4)).to(torch.uint8)


def _f16_bytes(v):
    """[..., 1] fp32 -> the 2 bytes of its fp16 value."""
    return v.to(torch.float16).contiguous().view(torch.uint8)


def _quantize(t, x):
    """Packed GGUF blocks of fp32 rows x [n, K] (plain round-to-nearest quantizers)."""
    n, K = x.shape
    if t == "q8_0":
        b = x.view(n, -1, 32)
        d = (b.abs().amax(-1, keepdim=True) / 127).half().float()
        q = torch.round(b / d.clamp_min(1e-8)).clamp(-127, 127).to(torch.int8)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], -1).view(n, -1)
    if t == "q4_0":
        b = x.view(n, -1, 32)
        at = b.abs().argmax(-1, keepdim=True)
        d = (b.gather(-1, at) / -8).half().float()
        inv = torch.where(d == 0, torch.zeros_like(d), 1 / d)
        q = torch.floor(b * inv + 8.5).clamp(0, 15).to(torch.int32)
        return torch.cat([_f16_bytes(d), _nibbles(q[..., :16], q[..., 16:])], -1).view(n, -1)
    if t == "q4_k":
        b = x.view(n, -1, 8, 32)
        lo = b.amin(-1).clamp_max(0)
        sc = (b.amax(-1) - lo) / 15
        d = (sc.amax(-1, keepdim=True) / 63).half().float().clamp_min(1e-7)
        dm = ((-lo).amax(-1, keepdim=True) / 63).half().float().clamp_min(1e-7)
        s = torch.round(sc / d).clamp(0, 63).to(torch.int32)
        m = torch.round(-lo / dm).clamp(0, 63).to(torch.int32)
        step = (d * s).unsqueeze(-1).clamp_min(1e-9)
        q = torch.round((b + (dm * m).unsqueeze(-1)) / step).clamp(0, 15).to(torch.int32)
        head = torch.cat([(s[..., :4] | (s[..., 4:] >> 4) << 6), (m[..., :4] | (m[..., 4:] >> 4) << 6), (s[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1).to(torch.uint8)
        qs = _nibbles(q[..., 0::2, :], q[..., 1::2, :]).flatten(-2)
        return torch.cat([_f16_bytes(d), _f16_bytes(dm), head, qs], -1).view(n, -1)
    if t == "q6_k":
        b = x.view(n, -1, 16, 16)
        sc = b.abs().amax(-1) / 31
        d = (sc.amax(-1, keepdim=True) / 127).half().float().clamp_min(1e-7)
        s = torch.round(sc / d).clamp(1, 127)
        q = (torch.round(b / (d * s).unsqueeze(-1)).clamp(-32, 31).to(torch.int32) + 32).view(n, -1, 2, 4, 32)
        ql = torch.cat([_nibbles(q[..., 0, :] & 15, q[..., 2, :] & 15), _nibbles(q[..., 1, :] & 15, q[..., 3, :] & 15)], -1).flatten(-2)
        qh = ((q[..., 0, :] >> 4) | (q[..., 1, :] >> 4) << 2 | (q[..., 2, :] >> 4) << 4 | (q[..., 3, :] >> 4) << 6).to(torch.uint8).flatten(-2)
        return torch.cat([ql, qh, s.to(torch.int8).view(torch.uint8), _f16_bytes(d)], -1).view(n, -1)
    raise ValueError(t)


def _f16_field(b):
    return b.contiguous().view(torch.float16).double()


def _unpack(t, w, N, K):
    """float64 [N, K] of a packed matrix."""
    if t == "f16":
        return w.view(N, K).double()
    b = w.view(N, K // QK[t], BB[t])
    if t == "q8_0":
        return (_f16_field(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).view(N, K)
    if t == "q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double() - 8
        return (_f16_field(b[..., :2]) * q).view(N, K)
    if t == "q4_k":
        d, dm, h = _f16_field(b[..., 0:2]), _f16_field(b[..., 2:4]), b[..., 4:16].to(torch.int32)
        s = torch.cat([h[..., :4] & 63, (h[..., 8:] & 15) | (h[..., :4] >> 6) << 4], -1).double()
        m = torch.cat([h[..., 4:8] & 63, (h[..., 8:] >> 4) | (h[..., 4:8] >> 6) << 4], -1).double()
        qs = b[..., 16:].reshape(N, -1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], -2).view(N, -1, 8, 32).double()
        return ((d * s).unsqueeze(-1) * q - (dm * m).unsqueeze(-1)).view(N, K)
    ql, qh = b[..., :128].reshape(N, -1, 2, 2, 32), b[..., 128:192].reshape(N, -1, 2, 32)
    q = torch.stack([(ql[..., 0, :] & 15) | (qh & 3) << 4, (ql[..., 1, :] & 15) | (qh >> 2 & 3) << 4, (ql[..., 0, :] >> 4) | (qh >> 4 & 3) << 4,
                     (ql[..., 1, :] >> 4) | (qh >> 6) << 4], -2).reshape(N, -1, 16, 16).double() - 32
    s = b[..., 192:208].contiguous().view(torch.int8).double()
    return ((_f16_field(b[..., 208:210]) * s).unsqueeze(-1) * q).view(N, K)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weight(t, N, K, g):
    """A packed N x K matrix of Gaussian weights of variance 1 / K."""
    out = torch.empty((N, K), dtype=torch.float16, device="cuda") if t == "f16" else torch.empty((N, K // QK[t] * BB[t]), dtype=torch.uint8, device="cuda")
    rows = max(1, (1 << 25) // K)
    for r in range(0, N, rows):
        x = torch.randn((min(rows, N - r), K), generator=g, device="cuda") * (K ** -0.5)
        out[r:r + rows] = x.half() if t == "f16" else _quantize(t, x)
    return out if t == "f16" else out.view(-1)


def _acts(M, K, dtype, g):
    return torch.randn((M, K), generator=g, device="cuda").to(DTYPES[dtype])


def _desc(d, t, A, W, C, N, K):
    d.ggml_type, d.A, d.a_dtype, d.W, d.C, d.c_dtype = TYPES[t], A.data_ptr(), qmm._dtype_code(A.dtype), W.data_ptr(), C.data_ptr(), qmm._dtype_code(C.dtype)
    d.M, d.N, d.K = A.shape[0], N, K


# ---- cases -----------------------------------------------------------------------------------
def _step_groups(c):
    """One layer's projections by the activations they read: [(K, [(type, N), ...]), ...]."""
    main, down = MIXES[c["mix"]]
    h, f, kv = c["hidden"], c["inter"], c["kv"]
    return [(h, [(main, h), (main, kv), (main, kv)]), (h, [(main, h)]), (h, [(main, f), (main, f)]), (f, [(down, h)])]


def _step_tensors(c, seed):
    """[(A, [(type, N, K, W), ...]), ...] over the layers."""
    g = _gen(seed)
    return [(_acts(c["M"], K, c["io"], g), [(t, N, K, _weight(t, N, K, g)) for t, N in mats]) for _ in range(c["layers"]) for K, mats in _step_groups(c)]


def _proj_tensors(c, seed):
    g = _gen(seed)
    return _acts(c["M"], c["K"], c["a"], g), [_weight(c["type"], c["N"], c["K"], g) for _ in range(c["mats"])]


_PROJ = (("wq", "attn_q"), ("wk", "attn_k"), ("wv", "attn_v"), ("wo", "attn_output"), ("wg", "ffn_gate"), ("wu", "ffn_up"), ("wd", "ffn_down"))


def _layer_dims(c):
    h, f, q, kv = c["hidden"], c["inter"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    main, down = MIXES[c["mix"]]
    return {"attn_q": (main, q, h), "attn_k": (main, kv, h), "attn_v": (main, kv, h), "attn_output": (main, h, q), "ffn_gate": (main, f, h),
            "ffn_up": (main, f, h), "ffn_down": (down, h, f)}


def _layer_tensors(c, seed):
    g = _gen(seed)
    x = _acts(c["seq"], c["hidden"], "f16", g)
    norms = [1 + 0.1 * torch.randn(c["hidden"], generator=g, device="cuda") for _ in range(2)]
    ws = {n: _weight(t, N, K, g) for n, (t, N, K) in _layer_dims(c).items()}
    past = [_acts(c["pos"], c["kv_heads"] * c["head_dim"], "f16", g) for _ in range(2)]
    return x, norms, ws, past


def _attn_tensors(c, seed):
    g = _gen(seed)
    kv = c["kv_heads"] * c["head_dim"]
    past = [_acts(c["pos"], kv, "f16", g) for _ in range(2)]
    return _acts(c["q"], c["heads"] * c["head_dim"], "f16", g), _acts(c["q"], kv, "f16", g), _acts(c["q"], kv, "f16", g), past


# The KV pool is one per device; each prepared state takes a layer of it of its own (the pool's
# layers are handed out in turn, more of them than states live at once).
_POOL_LAYERS = 8
_pool_layer = itertools.count()


def _attend(q, k, v, out, idx, start, c):
    qmm.check(qmm.lib().qmm_gqa_attention_cached(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), idx, q.shape[0], start, c["heads"],
                                                 c["kv_heads"], c["head_dim"], 0.0, 1, torch.cuda.current_stream().cuda_stream))


def _kv_state(c, rows, past):
    """A pool for `rows` positions and a layer of it that already holds the past keys and values."""
    pool = layer_mod.DeviceKVCache(_POOL_LAYERS, rows, c["kv_heads"], c["head_dim"])
    idx = next(_pool_layer) % _POOL_LAYERS
    if c["pos"]:
        q = torch.zeros((c["pos"], c["heads"] * c["head_dim"]), dtype=torch.float16, device="cuda")
        _attend(q, past[0], past[1], torch.empty_like(q), idx, 0, c)
        torch.cuda.synchronize()
    return pool, idx


def prepare(case, seed):
    c = case
    if c["kind"] == "step":
        groups = _step_tensors(c, seed)
        outs = [[torch.empty((c["M"], N), dtype=DTYPES[c["io"]], device="cuda") for _, N, _, _ in mats] for _, mats in groups]
        descs = (qmm.GemmDesc * sum(len(m) for _, m in groups))()
        i = 0
        for (A, mats), cs in zip(groups, outs):
            for (t, N, K, W), C in zip(mats, cs):
                _desc(descs[i], t, A, W, C, N, K)
                i += 1
        return {"kind": "step", "keep": groups, "descs": descs, "outs": outs}
    if c["kind"] == "proj":
        A, ws = _proj_tensors(c, seed)
        s = {"kind": "proj", "mats": c["mats"], "type": TYPES[c["type"]], "A": A, "W": ws, "N": c["N"], "K": c["K"], "out": DTYPES[c["c"]]}
        if c["mats"] > 1:
            s["outs"] = [torch.empty((c["M"], c["N"]), dtype=s["out"], device="cuda") for _ in ws]
            s["descs"] = (qmm.GemmDesc * len(ws))()
            for d, W, C in zip(s["descs"], ws, s["outs"]):
                _desc(d, c["type"], A, W, C, c["N"], c["K"])
        return s
    if c["kind"] == "dequant":
        return {"kind": "dequant", "type": TYPES[c["type"]], "W": _weight(c["type"], c["N"], c["K"], _gen(seed)), "n": c["N"] * c["K"], "out": DTYPES[c["c"]]}
    if c["kind"] == "layer":
        x, norms, ws, past = _layer_tensors(c, seed)
        pool, idx = _kv_state(c, c["pos"] + c["seq"], past)
        cfg = layer_mod.LlamaLayerConfig(hidden_size=c["hidden"], intermediate_size=c["inter"], num_heads=c["heads"], num_kv_heads=c["kv_heads"],
                                         head_dim=c["head_dim"], rope_freq_base=500000.0)
        p = f"blk.{idx}."
        lw = {}
        for n, (t, N, K) in _layer_dims(c).items():
            lw[f"{p}{n}.weight"] = (gguf.GGUFTensorInfo(f"{p}{n}.weight", (K, N), gguf.GGMLType(TYPES[t]), 0, 0, N * K, ws[n].numel()), ws[n])
        for n, v in zip(("attn_norm", "ffn_norm"), norms):
            lw[f"{p}{n}.weight"] = (gguf.GGUFTensorInfo(f"{p}{n}.weight", (c["hidden"],), gguf.GGMLType.F32, 0, 0, c["hidden"], 4 * c["hidden"]), v)
        return {"kind": "layer", "layer": layer_mod.TransformerLayer(cfg), "x": x, "lw": lw, "idx": idx, "pos": c["pos"], "pool": pool}
    q, k, v, past = _attn_tensors(c, seed)
    pool, idx = _kv_state(c, c["pos"] + c["q"], past)
    return {"kind": "attn", "q": q, "k": k, "v": v, "out": torch.empty_like(q), "idx": idx, "pos": c["pos"], "pool": pool, "case": dict(c)}


def run(state):
    s = state
    if s["kind"] == "step":
        qmm.gemm_batch(s["descs"])
        return s["outs"]
    if s["kind"] == "proj":
        if s["mats"] == 1:
            return qmm.gemm(s["type"], s["A"], s["W"][0], s["N"], s["K"], out_dtype=s["out"])
        qmm.gemm_batch(s["descs"])
        return s["outs"]
    if s["kind"] == "dequant":
        return qmm.dequantize(s["type"], s["W"], s["n"], out_dtype=s["out"])
    if s["kind"] == "layer":
        return s["layer"].forward_with_weights(s["x"], s["lw"], s["idx"], s["pos"], s["pool"])[0]
    _attend(s["q"], s["k"], s["v"], s["out"], s["idx"], s["pos"], s["case"])
    return s["out"]


def _wbytes(t, N, K):
    return N * (K // QK[t]) * BB[t]


def _visible(q, pos):
    """Sum over the new rows of the keys each one sees."""
    return q * pos + q * (q + 1) // 2


def work(case):
    c = case
    if c["kind"] == "step":
        b = f = 0
        for K, mats in _step_groups(c):
            b += c["M"] * K * EB[c["io"]] + sum(_wbytes(t, N, K) + c["M"] * N * EB[c["io"]] for t, N in mats)
            f += sum(2 * c["M"] * N * K for _, N in mats)
        return {"bytes": b * c["layers"], "flops": f * c["layers"]}
    if c["kind"] == "proj":
        one = _wbytes(c["type"], c["N"], c["K"]) + c["M"] * c["N"] * EB[c["c"]]
        return {"bytes": c["M"] * c["K"] * EB[c["a"]] + c["mats"] * one, "flops": 2 * c["mats"] * c["M"] * c["N"] * c["K"]}
    if c["kind"] == "dequant":
        return {"bytes": _wbytes(c["type"], c["N"], c["K"]) + c["N"] * c["K"] * EB[c["c"]], "flops": 0}
    q_len = c["seq"] if c["kind"] == "layer" else c["q"]
    kv = c["kv_heads"] * c["head_dim"]
    attn_flops = 4 * c["heads"] * c["head_dim"] * _visible(q_len, c["pos"])
    if c["kind"] == "layer":
        dims = _layer_dims(c).values()
        b = sum(_wbytes(t, N, K) for t, N, K in dims) + 2 * c["seq"] * c["hidden"] * 2 + 8 * c["hidden"] + 4 * kv * (c["pos"] + c["seq"])
        return {"bytes": b, "flops": 2 * c["seq"] * sum(N * K for _, N, K in dims) + attn_flops}
    # past keys and values read, the new ones read and written into the cache, queries and outputs
    return {"bytes": 4 * kv * (c["pos"] + 2 * c["q"]) + 4 * c["q"] * c["heads"] * c["head_dim"], "flops": attn_flops}


def tolerance(case):
    c = case
    if c["kind"] == "dequant":
        return "exact"  # a packed value has one nearest output value
    if c["kind"] in ("step", "proj"):
        types, a, out = ((set(MIXES[c["mix"]]), c["io"], c["io"]) if c["kind"] == "step" else ({c["type"]}, c["a"], c["c"]))
        if a == "f32":
            return {"rel": 1.6e-3}  # fp32 activations are rounded to fp16
        if c["M"] > 16 and types - {"f16"}:
            # matrix-core operands are fp16: packed weights (and the K-quants' scales) are rounded
            return {"rel": 3e-3 if types & {"q4_k", "q6_k"} else 1.6e-3}
        if out == "f16":
            return {"rel": 1.2e-3}  # one rounding to fp16
        # exact operands and fp32 sums; Q6_K products of scale and code may be rounded to fp16
        return {"rel": 6e-4 if "q6_k" in types else 5e-5}
    if c["kind"] == "attn":
        return {"rel": 1.2e-3}  # fp16 probabilities in the matrix product, fp16 output
    # a dozen roundings to fp16 in a row: norms, projections, rotation, probabilities, SwiGLU, residuals
    return {"rel": 3e-3}


# ---- float64 -----------------------------------------------------------------------------------
def _mm(a, t, w, N, K):
    """a [M, K] float64 @ dequant(w)^T, in row blocks of the weight."""
    rows = max(1, (1 << 27) // K)
    wb = w.view(N, -1)
    return torch.cat([a @ _unpack(t, wb[r:r + rows].contiguous(), min(rows, N - r), K).t() for r in range(0, N, rows)], 1)


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.half().double()


def _rope64(x, heads, d, pos):
    S = x.shape[0]
    x = x.view(S, heads, d)
    inv = 1.0 / 500000.0 ** (torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    ang = (pos + torch.arange(S, device="cuda", dtype=torch.float64))[:, None] * inv
    cs, sn = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cs - b * sn, a * sn + b * cs], -1).view(S, heads, d)


def _attn64(q, k, v, pos):
    """q [S, H, D], k / v [L, KVH, D] -> [S, H * D], causal from position pos."""
    S, H, D = q.shape
    L, KVH, _ = k.shape
    hide = torch.arange(L, device="cuda")[None, :] > (pos + torch.arange(S, device="cuda"))[:, None]
    out = torch.empty_like(q)
    for h in range(H):
        kk, vv = k[:, h // (H // KVH)], v[:, h // (H // KVH)]
        s = (q[:, h] @ kk.t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ vv.contiguous()
    return out.reshape(S, H * D)


def exact(case, seed):
    c = case
    if c["kind"] == "step":
        return [[_mm(A.double(), t, W, N, K) for t, N, K, W in mats] for A, mats in _step_tensors(c, seed)]
    if c["kind"] == "proj":
        A, ws = _proj_tensors(c, seed)
        r = [_mm(A.double(), c["type"], W, c["N"], c["K"]) for W in ws]
        return r[0] if c["mats"] == 1 else r
    if c["kind"] == "dequant":
        return _unpack(c["type"], _weight(c["type"], c["N"], c["K"], _gen(seed)), c["N"], c["K"]).view(-1)
    if c["kind"] == "attn":
        q, k, v, past = _attn_tensors(c, seed)
        kk, vv = (torch.cat([p, n]).double().view(-1, c["kv_heads"], c["head_dim"]) for p, n in zip(past, (k, v)))
        return _attn64(q.double().view(c["q"], c["heads"], c["head_dim"]), kk, vv, c["pos"])
    x, norms, ws, past = _layer_tensors(c, seed)
    dims = _layer_dims(c)

    def project(a, name):
        return _mm(a, dims[name][0], ws[name], dims[name][1], dims[name][2])

    H, KVH, D, pos = c["heads"], c["kv_heads"], c["head_dim"], c["pos"]
    x = x.double()
    n = _norm64(x, norms[0])
    q, k = _rope64(project(n, "attn_q"), H, D, pos), _rope64(project(n, "attn_k"), KVH, D, pos)
    k = torch.cat([past[0].double().view(-1, KVH, D), k])
    v = torch.cat([past[1].double(), project(n, "attn_v")]).view(-1, KVH, D)
    h = x + project(_attn64(q, k, v, pos), "attn_output")
    n = _norm64(h, norms[1])
    gate = project(n, "ffn_gate")
    return h + project(gate * torch.sigmoid(gate) * project(n, "ffn_up"), "ffn_down")
