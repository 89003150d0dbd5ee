"""Measured cases of the decode hot path, through its public entry points.

A case is a dict of plain values whose "op" names the path:

  project    resident Q2/Q4 projections (HipMatrix.dispatch), 1..8 rows
  mlp        residual + norm -> gate|up -> SwiGLU -> down blocks on registered
             weights, 1 row (plain decode) or 2..8 rows (draft verification)
  gdn_step   the crate's one-token gated-delta recurrence
  gdn_core   the decode layer's conv + gates + recurrence, with a state
             snapshot per verify row
  gdn_scan   chunked gated-delta prefill of a prompt
  attention  grouped-query attention over the paged mixed Q2/Q4 cache
  sample     top-k / top-p sampling of one logits row
  accept     rejection-sampling acceptance of k drafts
  decode     a decode step of the engine (4 layers of the 27B dimensions)

Inputs are made on the GPU from the seed. `exact` evaluates the same inputs in
float64 with plain torch.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ctox-llm_amd"))

import ctox_hip  # noqa: E402
from ctox_hip.engine import Engine, EngineConfig  # noqa: E402
from ctox_hip.paged_kv import DevicePagedKvCache  # noqa: E402

DEV = "cuda"
EPS = 1e-6
Q2, Q4 = 0, 1
BLOCK_BYTES = {Q2: 18, Q4: 34}
LEVELS = {Q2: 3, Q4: 15}  # value = scale * (2 code - LEVELS) / LEVELS
_backend = None


def hip():
    """The process's backend handle, as a serving program holds one per GPU."""
    global _backend
    if _backend is None:
        _backend = ctox_hip.HipBackend(0)
    return _backend


def listed():
    return [
        # One token's selection at the crate's sampler defaults over the 27B vocabulary: the smallest
        # device call of a plain decode step, after every token.
        {"name": "sample_k40", "op": "sample", "vocab": 151936, "top_k": 40, "temperature": 0.8, "top_p": 0.95},
        # The acceptance of the four drafts of a speculative step at T = 0.7.
        {"name": "accept_k4", "op": "accept", "vocab": 151936, "drafts": 4, "temperature": 0.7},
        # The Backend-level recurrence of one decoded token, 32 value heads: a call of a few microseconds.
        {"name": "gdn_step_h32", "op": "gdn_step", "heads": 32, "key_dim": 128, "value_dim": 128},
        # The FFN down projections of eight decoder layers for one decoded token (Q2 weights, long rows).
        {"name": "down_q2_row1", "op": "project", "dtype": Q2, "rows": 5120, "columns": 17408, "batch": 1,
         "layers": 8, "silu": False, "bias": False},
        # The q|k|v projections of four attention layers for the widest draft verification (8 rows, Q4).
        {"name": "qkv_q4_rows8", "op": "project", "dtype": Q4, "rows": 14336, "columns": 5120, "batch": 8,
         "layers": 4, "silu": False, "bias": False},
        # Four MLP blocks of a plain decode step: half of a token's weight bytes pass here.
        {"name": "mlp_row1", "op": "mlp", "hidden": 5120, "inter": 17408, "batch": 1, "layers": 4},
        # The same blocks under the five-row verification of four drafts.
        {"name": "mlp_rows5", "op": "mlp", "hidden": 5120, "inter": 17408, "batch": 5, "layers": 4},
        # The token mixer core of one layer in the five-row verification, every row's state kept.
        {"name": "gdn_core_rows5", "op": "gdn_core", "rows": 5, "heads": 48, "key_heads": 16},
        # A 4096-token prompt through one layer's recurrence, chunk 64.
        {"name": "gdn_prefill_4096", "op": "gdn_scan", "tokens": 4096, "heads": 32, "key_heads": 32, "chunk": 64},
        # A full-attention layer's cache read at a 32k context: plain decode, and the five-row verification.
        {"name": "attention_32k_row1", "op": "attention", "tokens": 32768, "page": 16, "rows": 1, "heads": 24,
         "kv_heads": 4},
        {"name": "attention_32k_rows5", "op": "attention", "tokens": 32768, "page": 16, "rows": 5, "heads": 24,
         "kv_heads": 4},
        # The engine's decode step on four layers (three GatedDeltaNet, one attention) and the LM head:
        # the whole call as a serving loop makes it, launches and the host's read of the status included.
        {"name": "decode_4layers_32k", "op": "decode", "layers": 4, "context": 32768},
    ]


def _log_int(rng, lo, hi, multiple=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple)) * multiple))


def draw(rng):
    op = rng.choice(["sample", "accept", "gdn_step", "project", "project", "mlp", "gdn_core", "gdn_scan", "gdn_scan",
                     "attention", "attention", "decode"])
    if op == "sample":
        return {"op": op, "vocab": _log_int(rng, 500, 151936), "top_k": _log_int(rng, 1, 256),
                "temperature": round(rng.uniform(0.4, 1.3), 3), "top_p": round(rng.uniform(0.7, 1.0), 3)}
    if op == "accept":
        return {"op": op, "vocab": _log_int(rng, 4096, 151936), "drafts": rng.randint(1, 7),
                "temperature": round(rng.uniform(0.5, 1.0), 3)}
    if op == "gdn_step":
        return {"op": op, "heads": rng.randint(4, 64), "key_dim": rng.choice([64, 96, 128]),
                "value_dim": rng.choice([48, 64, 128])}
    if op == "project":
        dtype = rng.choice([Q2, Q4])
        rows, columns = _log_int(rng, 64, 17408), _log_int(rng, 256, 17408, 64)
        return {"op": op, "dtype": dtype, "rows": rows, "columns": columns, "batch": rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8]),
                "layers": max(1, min(8, 250_000_000 // (rows * columns))), "silu": rng.random() < 0.3,
                "bias": rng.random() < 0.3}
    if op == "mlp":
        return {"op": op, "hidden": _log_int(rng, 512, 5120, 64), "inter": _log_int(rng, 1024, 17408, 64),
                "batch": rng.choice([1, 1, 2, 3, 4, 5, 5, 8]), "layers": rng.randint(1, 4)}
    if op == "gdn_core":
        heads, key_heads = rng.choice([(48, 16), (32, 16), (16, 16), (24, 8)])
        return {"op": op, "rows": rng.randint(1, 5), "heads": heads, "key_heads": key_heads}
    if op == "gdn_scan":
        heads, key_heads = rng.choice([(48, 16), (48, 16), (32, 16), (32, 32), (8, 8)])
        return {"op": op, "tokens": _log_int(rng, 40, 3200), "heads": heads, "key_heads": key_heads,
                "chunk": rng.choice([64, 64, 64, 48, 32])}
    if op == "attention":
        heads, kv_heads = rng.choice([(24, 4), (24, 4), (16, 4), (8, 2)])
        return {"op": op, "tokens": _log_int(rng, 40, 32768), "page": rng.choice([16, 16, 16, 128, 32, 8]),
                "rows": rng.choice([1, 1, 2, 3, 4, 5]), "heads": heads, "kv_heads": kv_heads}
    return {"op": op, "layers": 4, "context": _log_int(rng, 300, 30000)}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g) * std


def _blocks(g, dtype, rows, columns):
    """Packed rows [rows][columns / 64][block bytes]: uniform codes, fp16 scales |N(0, 0.02)|."""
    w = torch.randint(0, 256, (rows, columns // 64, BLOCK_BYTES[dtype]), dtype=torch.uint8, device=DEV, generator=g)
    w[:, :, :2] = _randn(g, rows, columns // 64, std=0.02).abs().half().view(torch.uint8).view(rows, columns // 64, 2)
    return w


def _scales(g, n):
    return (0.75 + 0.5 * torch.rand(n, device=DEV, generator=g)).half()


def _values(w):
    """Packed blocks [..., block bytes] to float64 values [..., 64]."""
    dtype = Q2 if w.shape[-1] == BLOCK_BYTES[Q2] else Q4
    scale = w[..., :2].contiguous().view(torch.float16).double()
    body, bits = w[..., 2:], 2 if dtype == Q2 else 4
    codes = torch.stack([(body >> s) & (2 ** bits - 1) for s in range(0, 8, bits)], -1).flatten(-2)
    return scale * ((2 * codes.double() - LEVELS[dtype]) / LEVELS[dtype])


def _product(w, s_in, s_out, x):
    """x [batch][columns] times the packed rows' transpose, float64 (a slice of rows at a time)."""
    xs = x.double() * s_in.double()
    out = [xs @ _values(w[r:r + 2048]).flatten(1).T for r in range(0, w.shape[0], 2048)]
    return torch.cat(out, 1) * s_out.double()


class _Registered:
    """Packed weights on the device with a registered tiled copy."""

    def __init__(self, g, dtype, rows, columns):
        self.dtype, self.rows, self.columns = dtype, rows, columns
        self.w, self.s_in, self.s_out = _blocks(g, dtype, rows, columns), _scales(g, columns), _scales(g, rows)
        self.registered = False

    def register(self):
        hip().register_tiled_weights(ctox_hip.TensorDType(self.dtype), self.w.data_ptr(), self.rows, self.columns)
        self.registered = True
        return self

    def __del__(self):
        if self.registered:
            hip().unregister_tiled_weights(self.w.data_ptr())


class _Transform(ctypes.Structure):
    """ctox_input_transform."""
    _fields_ = [("a", ctypes.c_void_p), ("b", ctypes.c_void_p), ("w", ctypes.c_void_p), ("mode", ctypes.c_uint32),
                ("a_stride", ctypes.c_uint32), ("b_stride", ctypes.c_uint32), ("off", ctypes.c_uint32),
                ("head_dim", ctypes.c_uint32), ("eps", ctypes.c_float), ("res_h", ctypes.c_void_p),
                ("res_sums", ctypes.c_void_p), ("a_parts", ctypes.c_uint32), ("a_part_stride", ctypes.c_uint32)]


def _check(status):
    if status:
        raise RuntimeError(ctox_hip.load_library().ctox_hip_last_error().decode())


def _inputs(c, seed):
    """The tensors a case starts from."""
    g, op = _gen(seed), c["op"]
    if op == "project":
        mats = []
        for _ in range(c["layers"]):
            bias = _randn(g, c["rows"], std=0.1) if c["bias"] else None
            mats.append((_blocks(g, c["dtype"], c["rows"], c["columns"]), _scales(g, c["columns"]), _scales(g, c["rows"]), bias))
        gate = _randn(g, c["layers"], c["batch"], c["columns"])
        # What a projection reads in a layer: normalised rows, or a down projection's SiLU(gate) * up.
        x = gate if c["dtype"] == Q4 else torch.nn.functional.silu(gate) * _randn(g, *gate.shape)
        return {"mats": mats, "x": x}
    if op == "mlp":
        H, inter, R = c["hidden"], c["inter"], c["batch"]
        return {"layers": [(_Registered(g, Q4, 2 * inter, H), _Registered(g, Q2, H, inter), _randn(g, H, std=0.1))
                           for _ in range(c["layers"])],
                "h": _randn(g, R, H), "delta": _randn(g, R, H)}
    if op in ("gdn_step", "gdn_scan"):
        T, heads = c.get("tokens", 1), c["heads"]
        kh, dk, dv = c.get("key_heads", heads), c.get("key_dim", 128), c.get("value_dim", 128)
        # Token rows [q | k | v] as the layer's convolution leaves them, after SiLU.
        rows = torch.nn.functional.silu(_randn(g, T, 2 * kh * dk + heads * dv))
        return {"rows": rows, "q": rows[:, :kh * dk], "k": rows[:, kh * dk:2 * kh * dk], "v": rows[:, 2 * kh * dk:],
                "ld": -torch.nn.functional.softplus(_randn(g, T, heads)), "beta": torch.sigmoid(_randn(g, T, heads)),
                "state": _randn(g, heads, dk, dv, std=0.1), "dims": (T, heads, kh, dk, dv)}
    if op == "gdn_core":
        R, heads, kh = c["rows"], c["heads"], c["key_heads"]
        channels = 2 * kh * 128 + heads * 128
        return {"proj": _randn(g, R, channels + heads * 128 + 2 * heads), "conv_w": _randn(g, channels, 4, std=0.5),
                "conv_in": _randn(g, channels, 4), "a_log": _randn(g, heads, std=0.3), "dt_bias": _randn(g, heads, std=0.3),
                "state": _randn(g, heads, 128, 128, std=0.1)}
    if op == "attention":
        T, kvh, pages = c["tokens"], c["kv_heads"], -(-c["tokens"] // c["page"])
        first = torch.arange(pages, device=DEV) * c["page"]
        count = torch.clamp(T - first, max=c["page"])
        # The retention policy: 128 sink and 256 recent tokens in Q4 pages, the rest demoted to Q2.
        sink = -(-128 // c["page"]) * c["page"]
        q4 = (first < sink) | (first + count > T - 256)
        vals = _randn(g, pages * c["page"], 2 * kvh * 4, 64)
        return {"values": vals, "q4": q4, "first": first, "count": count, "sink": sink,
                "query": _randn(g, c["rows"], c["heads"], 256)}
    if op in ("sample", "accept"):
        k = c.get("drafts", 0)
        # Logits of a trained head: a broad body with a handful of likely tokens.
        rows = _randn(g, k + 1, c["vocab"], std=2.0)
        top = torch.randint(0, c["vocab"], (k + 1, 12), device=DEV, generator=g)
        rows.scatter_add_(1, top, 10.0 + 4.0 * torch.rand(k + 1, 12, device=DEV, generator=g))
        draft = rows[:k] + _randn(g, k, c["vocab"], std=0.5)
        u = torch.rand(1, device=DEV, generator=g)
        return {"target": rows[:k].contiguous(), "bonus": rows[k].contiguous(), "draft": draft, "u": float(u),
                "rng": torch.randint(1, 2 ** 62, (1,), device=DEV, generator=g)}
    raise ValueError(op)


def _quantize(vals, dtype):
    """64-value blocks to packed bytes: scale = max |v|, codes the nearest level."""
    m = vals.abs().amax(-1, keepdim=True)
    levels = LEVELS[dtype]
    codes = torch.clamp(torch.round((vals / m + 1) * (levels / 2)), 0, levels).to(torch.uint8)
    per = 4 if dtype == Q2 else 2
    codes = codes.unflatten(-1, (64 // per, per))
    body = codes[..., 0]
    for i in range(1, per):
        body = body | (codes[..., i] << (8 // per * i))
    return torch.cat([m.half().view(torch.uint8), body], -1)


def _pages(c, i):
    """(Q4 pages, Q2 pages) as [page][token][bytes] tensors of the case's cache, in page order."""
    vals = i["values"].unflatten(0, (-1, c["page"]))
    out = {}
    for dtype, pick in ((Q4, i["q4"]), (Q2, ~i["q4"])):
        out[dtype] = _quantize(vals[pick], dtype).flatten(2)
    return out


def _paged_cache(c, i):
    """A cache in the state its pushes would have left it in, the pages written directly."""
    T, pages = c["tokens"], i["q4"].numel()
    n4 = int(i["q4"].sum())
    cache = DevicePagedKvCache(hip(), max(pages * c["page"], i["sink"], 256), c["kv_heads"], 256, page_tokens=c["page"],
                               sink_tokens=i["sink"], recent_tokens=256, q4_slots=max(1, n4))
    packed = _pages(c, i)
    cache.q4_pool[:packed[Q4].numel()] = packed[Q4].flatten()
    cache.q2_pool[:packed[Q2].numel()] = packed[Q2].flatten()
    q4 = i["q4"].long()
    slot = torch.where(i["q4"], torch.cumsum(q4, 0), torch.cumsum(1 - q4, 0)) - 1
    desc = torch.stack([q4, slot, i["count"], i["first"]], 1).to(torch.int32)
    cache.d_desc[:pages] = desc
    cache.desc[:pages] = desc.cpu().numpy().view(np.uint32)
    cache.n_pages, cache.n_tokens = pages, T
    return cache


class _DeviceFloats:
    """A float buffer of the engine as an array a tensor can wrap (the tensor keeps the engine)."""

    def __init__(self, engine, which, count):
        self.engine = engine
        ptr, _ = engine.buffer(which)
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (count,), "typestr": "<f4", "version": 2}


def _engine(c, seed):
    cfg = EngineConfig.qwen38_27b(max_tokens=c["context"] + 16384, drafts=0)
    cfg.num_hidden_layers = c["layers"]
    eng = Engine(hip(), cfg, seed=seed % 100003 + 1)
    eng.fill_context(c["context"], seed=seed % 1009 + 1)
    return eng, 1 + seed * 7919 % (cfg.vocab_size - 1)


# ---------------------------------------------------------------- a pass
def prepare(case, seed):
    c = dict(case)
    op = c["op"]
    if op == "decode":
        eng, token = _engine(c, seed)
        logits = torch.as_tensor(_DeviceFloats(eng, 0, eng.config.vocab_size), device=DEV)
        final = torch.as_tensor(_DeviceFloats(eng, 1, eng.config.hidden_size), device=DEV)
        return {"case": c, "engine": eng, "token": token, "out": {"logits": logits, "final": final}}
    i = _inputs(c, seed)
    s = {"case": c, "in": i}
    if op == "project":
        s["mats"] = []
        for w, s_in, s_out, bias in i.pop("mats"):
            s["mats"].append(hip().prepare(ctox_hip.FusedMatVec(
                ctox_hip.TensorDType(c["dtype"]), w.cpu().numpy(), c["rows"], c["columns"],
                s_in=ctox_hip.ScaleSlice.F16Le(s_in.cpu().numpy()), s_out=ctox_hip.ScaleSlice.F16Le(s_out.cpu().numpy()),
                bias=None if bias is None else bias.cpu().numpy(),
                activation=ctox_hip.Activation.Silu if c["silu"] else ctox_hip.Activation.Identity)))
        s["y"] = torch.empty(c["layers"], c["batch"], c["rows"], device=DEV)
    elif op == "mlp":
        R, H, inter = c["batch"], c["hidden"], c["inter"]
        for gate_up, down, _ in i["layers"]:
            gate_up.register()
            down.register()
        s["gu"] = torch.empty(6, R, 2 * inter, device=DEV)
        s["h"] = torch.empty(c["layers"], R, H, device=DEV)
        s["delta"] = torch.empty(c["layers"], R, H, device=DEV)
        s["sums"] = torch.empty(R, -(-H // 16), device=DEV)
    elif op in ("gdn_step", "gdn_scan"):
        T, heads, kh, dk, dv = i["dims"]
        if kh == heads:
            for n in "qkv":
                i[n] = i[n].contiguous()
        s["out"] = torch.empty(T, heads, dv, device=DEV)
    elif op == "gdn_core":
        R, heads = c["rows"], c["heads"]
        s["blocked"] = _block_state(i["state"])
        s["conv_out"] = torch.empty(R, *i["conv_in"].shape, device=DEV)
        s["state_out"] = torch.empty(R, i["state"].numel(), device=DEV)
        s["ld"], s["beta"] = torch.empty(R, heads, device=DEV), torch.empty(R, heads, device=DEV)
        s["out"] = torch.empty(R, heads, 128, device=DEV)
    elif op == "attention":
        s["cache"] = _paged_cache(c, i)
        del i["values"]
        s["out"] = torch.empty_like(i["query"])
    elif op == "sample":
        s["out"] = torch.zeros(4, dtype=torch.int32, device=DEV)
    elif op == "accept":
        s["tokens"] = torch.argmax(i["draft"], 1).to(torch.int32)
        s["out"] = torch.zeros(2, dtype=torch.int32, device=DEV)
    return s


def run(s):
    return globals()["_run_" + s["case"]["op"]](s, s["case"], s.get("in"))


def _run_project(s, c, i):
    for n, m in enumerate(s["mats"]):
        m.dispatch(i["x"][n].data_ptr(), c["batch"], s["y"][n].data_ptr())
    return s["y"]


def _run_mlp(s, c, i):
    """The engine's MLP blocks: each block's delta is added by the next one's norm."""
    lib, b = ctox_hip.load_library(), hip()
    R, H, inter = c["batch"], c["hidden"], c["inter"]
    sums_ok = R <= 5
    h, delta, sums = i["h"], i["delta"], None
    for n, (gate_up, down, norm) in enumerate(i["layers"]):
        h_out, out = s["h"][n], s["delta"][n]
        gu_parts = ctypes.c_uint32(1)
        _check(lib.ctox_hip_norm_matvec_parts_device(
            b.handle, h.data_ptr(), delta.data_ptr(), 1, R * H, h_out.data_ptr(), norm.data_ptr(), EPS, None, Q4,
            gate_up.w.data_ptr(), gate_up.s_in.data_ptr(), gate_up.s_out.data_ptr(), s["gu"].data_ptr(), 2 * inter, H, R,
            sums, -(-H // 16) if sums else 0, 6, ctypes.byref(gu_parts), None))
        x = _Transform(s["gu"].data_ptr(), None, None, 1, 2 * inter, 0, inter, 0, 0.0,
                       h_out.data_ptr() if sums_ok else None, s["sums"].data_ptr() if sums_ok else None,
                       gu_parts.value, R * 2 * inter)
        _check(lib.ctox_hip_transform_matvec_device(
            b.handle, ctypes.byref(x), Q2, down.w.data_ptr(), down.s_in.data_ptr(), down.s_out.data_ptr(), out.data_ptr(),
            H, inter, R, 0, ctypes.byref(ctypes.c_uint32(1)), None))
        h, delta = h_out, out
        sums = s["sums"].data_ptr() if sums_ok else None
    return {"h": s["h"], "delta": s["delta"]}


def _run_gdn_step(s, c, i):
    _, heads, _, dk, dv = i["dims"]
    hip().gated_delta_step_device(i["q"].data_ptr(), i["k"].data_ptr(), i["v"].data_ptr(), i["ld"].data_ptr(),
                                  i["beta"].data_ptr(), i["state"].data_ptr(), heads, dk, dv, s["out"].data_ptr())
    return {"out": s["out"], "state": i["state"]}


def _run_gdn_scan(s, c, i):
    T, heads, kh, dk, dv = i["dims"]
    ptrs = [i[n].data_ptr() for n in "qkv"]
    gates = (i["ld"].data_ptr(), i["beta"].data_ptr(), i["state"].data_ptr())
    if kh == heads:
        hip().gated_delta_sequence_device(*ptrs, *gates, T, heads, dk, dv, c["chunk"], s["out"].data_ptr())
    else:  # in place from the fused rows, key heads repeated
        stride = i["rows"].shape[1]
        hip().gated_delta_strided_device(*ptrs, stride, stride, *gates, T, heads, kh, dk, dv, c["chunk"],
                                         s["out"].data_ptr())
    return {"out": s["out"], "state": i["state"]}


def _run_gdn_core(s, c, i):
    R, heads, kh = c["rows"], c["heads"], c["key_heads"]
    channels, stride = i["conv_w"].shape[0], i["proj"].shape[1]
    _check(ctox_hip.load_library().ctox_hip_gdn_fused_snap_device(
        hip().handle, i["proj"].data_ptr(), stride, stride - 2 * heads, stride - heads, i["conv_w"].data_ptr(),
        i["conv_in"].data_ptr(), s["conv_out"].data_ptr(), channels * 4, 4, i["a_log"].data_ptr(), i["dt_bias"].data_ptr(),
        s["ld"].data_ptr(), s["beta"].data_ptr(), s["blocked"].data_ptr(), s["state_out"].data_ptr(), i["state"].numel(),
        1, R, heads, kh, 128, 128, s["out"].data_ptr(), None))
    return {"out": s["out"], "state": s["state_out"], "conv": s["conv_out"], "ld": s["ld"], "beta": s["beta"]}


def _run_attention(s, c, i):
    return s["cache"].attention(i["query"], c["rows"], c["heads"], s["out"])


def _run_sample(s, c, i):
    _check(ctox_hip.load_library().ctox_hip_sample_topk_topp_device(
        hip().handle, i["bonus"].data_ptr(), c["vocab"], c["temperature"], c["top_k"], c["top_p"], i["u"],
        s["out"].data_ptr(), None))
    return {"choice": s["out"][:3], "total": s["out"][3:].view(torch.float32)}


def _run_accept(s, c, i):
    hip().mtp_accept_device(i["draft"].data_ptr(), i["target"].data_ptr(), i["bonus"].data_ptr(), s["tokens"].data_ptr(),
                            c["drafts"], c["vocab"], c["temperature"], i["rng"].data_ptr(), s["out"].data_ptr())
    return {"choice": s["out"], "rng": i["rng"]}


def _run_decode(s, c, i):
    s["engine"].decode(s["token"])
    return s["out"]


# ---------------------------------------------------------------- work
def work(case):
    c, op = case, case["op"]
    if op == "project":
        n = c["rows"] * c["columns"]
        b = n // 64 * BLOCK_BYTES[c["dtype"]] + (c["rows"] + c["columns"]) * (2 + 4 * c["batch"]) + 4 * c["rows"] * c["bias"]
        return {"bytes": c["layers"] * b, "flops": 2 * c["layers"] * n * c["batch"]}
    if op == "mlp":
        n, R, H = c["hidden"] * c["inter"], c["batch"], c["hidden"]
        b = (2 * n * 34 + n * 18) // 64 + 2 * (2 * H + 3 * c["inter"]) + 4 * H + 4 * 4 * R * H
        return {"bytes": c["layers"] * b, "flops": 6 * c["layers"] * n * R}
    if op in ("gdn_step", "gdn_scan"):
        T, heads = c.get("tokens", 1), c["heads"]
        kh, dk, dv = c.get("key_heads", heads), c.get("key_dim", 128), c.get("value_dim", 128)
        return {"bytes": 4 * (T * (2 * kh * dk + 2 * heads * dv + 2 * heads) + 2 * heads * dk * dv),
                "flops": 8 * T * heads * dk * dv}
    if op == "gdn_core":
        R, heads, channels = c["rows"], c["heads"], 256 * c["key_heads"] + 128 * c["heads"]
        b = heads * 16384 * (1 + R) + R * (channels + heads * 128 + 4 * heads) + channels * 4 * (2 + R)
        return {"bytes": 4 * b, "flops": 8 * R * heads * 16384 + 8 * R * channels}
    if op == "attention":
        T, per = c["tokens"], 2 * c["kv_heads"] * 4
        sink = -(-128 // c["page"]) * c["page"]
        q4 = min(T, sink + 256)
        return {"bytes": per * (q4 * 34 + (T - q4) * 18) + 2 * 4 * c["rows"] * c["heads"] * 256,
                "flops": 4 * c["rows"] * c["heads"] * T * 256}
    if op == "sample":
        return {"bytes": 4 * c["vocab"], "flops": c["vocab"]}
    if op == "accept":
        return {"bytes": 4 * (2 * c["drafts"] + 1) * c["vocab"], "flops": 4 * (2 * c["drafts"] + 1) * c["vocab"]}
    gdn = c["layers"] - c["layers"] // 4
    attn = c["layers"] // 4
    q4 = gdn * (16480 + 6144) * 5120 + attn * (14336 + 6144) * 5120 + c["layers"] * 34816 * 5120 + 151936 * 5120
    q2 = c["layers"] * 5120 * 17408
    kv = work({"op": "attention", "tokens": c["context"] + 1, "page": 16, "rows": 1, "heads": 24, "kv_heads": 4})
    return {"bytes": (q4 * 34 + q2 * 18) // 64 + attn * kv["bytes"] + gdn * 2 * 48 * 16384 * 4 + 4 * 151936,
            "flops": 2 * (q4 + q2) + attn * kv["flops"] + gdn * 8 * 48 * 16384}


def tolerance(case):
    op = case["op"]
    if op in ("sample", "accept"):
        return {"rel": 1e-5, "differ": 0.0}
    if op == "attention":
        # Each output is a mean over tens of thousands of values of both signs, so 32-bit sums leave
        # 2.4e-5 of it against float64 at 32k tokens.
        return {"rel": 1e-4, "max": 1e-3}
    if op == "decode":
        # 3e-6 against float64; a key or value next to a rounding boundary may take the neighbouring
        # 4-bit code, which moves a short context's attention by about 1e-4.
        return {"rel": 2e-4, "max": 2e-3}
    return {"rel": 1e-5, "max": 1e-4}


# ---------------------------------------------------------------- float64
def exact(case, seed):
    return globals()["_exact_" + case["op"]](case, seed)


def _exact_project(c, seed):
    i, out = _inputs(c, seed), []
    for n, (w, s_in, s_out, bias) in enumerate(i["mats"]):
        y = _product(w, s_in, torch.ones_like(s_out), i["x"][n])
        y = (y if bias is None else y + bias.double()) * s_out.double()
        out.append(torch.nn.functional.silu(y) if c["silu"] else y)
    return torch.stack(out)


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1 + w.double())


def _exact_mlp(c, seed):
    i = _inputs(c, seed)
    h, delta, hs, ds = i["h"].double(), i["delta"].double(), [], []
    for gate_up, down, norm in i["layers"]:
        h = h + delta
        gu = _product(gate_up.w, gate_up.s_in, gate_up.s_out, _norm(h, norm))
        act = torch.nn.functional.silu(gu[:, :c["inter"]]) * gu[:, c["inter"]:]
        delta = _product(down.w, down.s_in, down.s_out, act)
        hs.append(h)
        ds.append(delta)
    return {"h": torch.stack(hs), "delta": torch.stack(ds)}


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _recur(q, k, v, ld, beta, state):
    """The recurrence in float64, token by token: q, k [T][key heads][dk], v [T][heads][dv]; yields (output, state)."""
    rep = v.shape[1] // q.shape[1]
    q = _unit(q.double()).repeat_interleave(rep, 1) / math.sqrt(q.shape[-1])
    k = _unit(k.double()).repeat_interleave(rep, 1)
    v, decay, beta, S = v.double(), ld.double().exp(), beta.double(), state.double().clone()
    for t in range(q.shape[0]):
        S *= decay[t][:, None, None]
        d = beta[t][:, None] * (v[t] - torch.matmul(k[t][:, None, :], S)[:, 0])
        S += k[t][:, :, None] * d[:, None, :]
        yield torch.matmul(q[t][:, None, :], S)[:, 0], S


def _exact_gdn_scan(c, seed):
    i = _inputs(c, seed)
    _, heads, kh, dk, dv = i["dims"]
    steps = _recur(i["q"].unflatten(1, (kh, dk)), i["k"].unflatten(1, (kh, dk)), i["v"].unflatten(1, (heads, dv)), i["ld"],
                   i["beta"], i["state"])
    out = []
    for o, state in steps:
        out.append(o)
    return {"out": torch.stack(out), "state": state}


_exact_gdn_step = _exact_gdn_scan


def _block_state(S):
    """[heads][128][128] to the engine's layout: per head and 16 value columns, [key % 16][value % 16][key / 16]."""
    heads = S.shape[0]
    return S.view(heads, 8, 16, 8, 16).permute(0, 3, 2, 4, 1).reshape(-1).contiguous()


def _conv(window, x, w):
    """One token of the causal convolution + SiLU: (window after it, outputs)."""
    window = torch.cat([window[:, 1:], x[:, None]], 1)
    return window, torch.nn.functional.silu((window * w.double()).sum(1))


def _exact_gdn_core(c, seed):
    i = _inputs(c, seed)
    R, heads, kh = c["rows"], c["heads"], c["key_heads"]
    channels = i["conv_w"].shape[0]
    window, rows, windows = i["conv_in"].double(), [], []
    for t in range(R):
        window, x = _conv(window, i["proj"][t, :channels].double(), i["conv_w"])
        rows.append(x)
        windows.append(window)
    rows = torch.stack(rows)
    a, b = i["proj"][:, -2 * heads:-heads].double(), i["proj"][:, -heads:].double()
    ld = -i["a_log"].double().exp() * torch.nn.functional.softplus(a + i["dt_bias"].double())
    beta = torch.sigmoid(b)
    q, k, v = rows.split([kh * 128, kh * 128, heads * 128], 1)
    out, states = [], []
    for o, S in _recur(q.unflatten(1, (kh, 128)), k.unflatten(1, (kh, 128)), v.unflatten(1, (heads, 128)), ld, beta, i["state"]):
        out.append(o)
        states.append(_block_state(S))
    return {"out": torch.stack(out), "state": torch.stack(states), "conv": torch.stack(windows), "ld": ld, "beta": beta}


def _attend(query, kv, kv_heads):
    """Rows' grouped-query attention over kv [tokens][K heads | V heads][256], causal from the last row back."""
    R, heads = query.shape[:2]
    T, group = kv.shape[0], heads // kv_heads
    K, V = kv[:, :kv_heads], kv[:, kv_heads:]
    out = torch.empty(R, heads, 256, dtype=torch.float64, device=DEV)
    for r in range(R):
        n = T - R + r + 1
        for h in range(kv_heads):
            s = query[r, h * group:(h + 1) * group].double() @ K[:n, h].T / 16.0
            out[r, h * group:(h + 1) * group] = torch.softmax(s, -1) @ V[:n, h]
    return out


def _exact_attention(c, seed):
    i = _inputs(c, seed)
    pages, kvh = _pages(c, i), c["kv_heads"]
    kv = torch.empty(i["q4"].numel(), c["page"], 2 * kvh, 256, dtype=torch.float64, device=DEV)
    kv[i["q4"]] = _values(pages[Q4].unflatten(-1, (-1, 34))).flatten(-2).unflatten(-1, (2 * kvh, 256))
    kv[~i["q4"]] = _values(pages[Q2].unflatten(-1, (-1, 18))).flatten(-2).unflatten(-1, (2 * kvh, 256))
    return _attend(i["query"], kv.flatten(0, 1)[:c["tokens"]], kvh)


def _exact_sample(c, seed):
    i = _inputs(c, seed)
    x = i["bonus"].double() / c["temperature"]
    val, tok = torch.sort(x.flip(0), descending=True, stable=True)  # ties: the later token first
    val, tok = val[:c["top_k"]], c["vocab"] - 1 - tok[:c["top_k"]]
    w = torch.exp(val - val[0])
    cum = torch.cumsum(w, 0)
    n = int((cum < c["top_p"] * cum[-1]).sum()) + 1
    n = min(n, w.numel())
    pick = min(int((cum[:n] < i["u"] * cum[n - 1]).sum()), n - 1)
    return {"choice": torch.tensor([int(tok[pick]), 0, n], dtype=torch.int32), "total": cum[n - 1:n]}


def _exact_accept(c, seed):
    return None  # whole numbers only


def _exact_decode(c, seed):
    """The first decode step after the filled context, in float64, from the engine's own weights and pages."""
    eng, token = _engine(c, seed)
    cfg, eps = eng.config, eng.config.rms_norm_epsilon
    H, inter = cfg.hidden_size, cfg.intermediate_size
    qh, kvh, hv, hk = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.linear_num_value_heads, cfg.linear_num_key_heads

    def on(raw, kind):
        return torch.from_numpy(np.frombuffer(raw, kind).copy()).to(DEV)

    def vec(name):
        return on(eng.tensor(name)["data"], np.float32).double()

    def mat(name):
        t = eng.tensor(name)
        w = on(t["data"], np.uint8).view(t["rows"], t["cols"] // 64, BLOCK_BYTES[t["dtype"]])
        return w, on(t["s_in"], np.float16), on(t["s_out"], np.float16)

    def times(name, x):
        return _product(*mat(name), x[None])[0]

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * (1 + vec(name))

    def mixer(p, x):
        rows = times(p + ".in", x)
        channels = 256 * hk + 128 * hv
        mixed, z, a, b = rows.split([channels, 128 * hv, hv, hv])
        _, conv = _conv(torch.zeros(channels, 4, dtype=torch.float64, device=DEV), mixed, vec(p + ".conv_w").view(channels, 4))
        q, k, v = conv.split([128 * hk, 128 * hk, 128 * hv])
        ld = -vec(p + ".a_log").exp() * torch.nn.functional.softplus(a + vec(p + ".dt_bias"))
        zero = torch.zeros(hv, 128, 128, dtype=torch.float64, device=DEV)
        core = next(_recur(q.view(1, hk, 128), k.view(1, hk, 128), v.view(1, hv, 128), ld[None], torch.sigmoid(b)[None], zero))[0]
        core = core * torch.rsqrt(core.square().mean(-1, keepdim=True) + eps) * vec(p + ".gnorm")
        return times(p + ".out", (core * torch.nn.functional.silu(z.view(hv, 128))).flatten())

    def rotate(x):
        half = cfg.rotary_dim // 2
        angle = c["context"] * cfg.rope_theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
        left, right = x[:, :half], x[:, half:2 * half]
        return torch.cat([left * angle.cos() - right * angle.sin(), right * angle.cos() + left * angle.sin(), x[:, 2 * half:]], 1)

    def attention(layer, x):
        p = "L%d" % layer
        qg, k, v = times(p + ".qkv", x).split([512 * qh, 256 * kvh, 256 * kvh])
        qg = qg.view(qh, 512)
        q = rotate(norm(qg[:, :256], p + ".q_norm"))
        k = rotate(norm(k.view(kvh, 256), p + ".k_norm"))
        new = _values(_quantize(torch.cat([k, v.view(kvh, 256)]).view(-1, 64), Q4)).view(1, 2 * kvh, 256)
        old = []
        for precision, tokens, _, raw in eng.cache_pages(layer):
            old.append((34 if precision else 18, tokens, raw))
        kv = []
        for size in (34, 18):  # page order does not matter: attention sums over all of them
            raw = b"".join(r for n, _, r in old if n == size)
            if raw:
                kv.append(_values(on(raw, np.uint8).view(-1, size)).view(-1, 2 * kvh, 256))
        out = _attend(q[None], torch.cat(kv + [new]), kvh)[0] * torch.sigmoid(qg[:, 256:])
        return times(p + ".o", out.flatten())

    w, s_in, s_out = mat("embed")
    h = _values(w[token:token + 1]).flatten() * s_in.double() * s_out[token].double()
    del w
    for n in range(c["layers"]):
        x = norm(h, "L%d.norm" % n)
        h = h + (attention(n, x) if (n + 1) % cfg.full_attention_interval == 0 else mixer("L%d" % n, x))
        gu = times("L%d.gate_up" % n, norm(h, "L%d.mlp_norm" % n))
        h = h + times("L%d.down" % n, torch.nn.functional.silu(gu[:inter]) * gu[inter:])
    final = norm(h, "final_norm")
    out = {"logits": times("lm_head", final), "final": final}
    eng.close()
    return out
