"""Measured workloads of the Qwen3-ASR text decoder, through the C ABI that its callers use.

Five kinds of work, each on the shapes of the two released model sizes (hidden 1024 and 2048, 16 query heads,
8 KV heads, head_dim 128, vocabulary 151936):

  decode_attn    one decode step's KV-cache path (append + attention) over a model's layers, for 1 to 32 streams
  prefill_attn   K/V append and causal attention of one layer's prompt, or of a chunk behind cached positions
  stream_proj    the projections of a multi-stream decode step: q|k|v, o, gate|up and down of four layers
  prefill        a whole cached call of a prompt through a decoder: layers, last-row logits, cache
  token          a whole cached call of one token through a decoder

Weights are f32, as the reference's loader requires, or f32 that hold bf16 values, as a checkpoint converted
from the released bf16 weights does.  Caches are f16 (the command line's usual choice) or f32 (the drop-in
API's default).  Inputs have the distributions of the repository's benchmark: weights N(0, 0.02), norm weights
near 1, embeddings and cached K/V N(0, 1).
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qwenasr.cpp_amd"))

import qwenasr_amd as qa  # noqa: E402

SIZES = {"0.6B": qa.QWEN3_ASR_0_6B, "1.7B": qa.QWEN3_ASR_1_7B}
HEADS, KV_HEADS, DIM = 16, 8, 128
Q_DIM, KV_DIM = HEADS * DIM, KV_HEADS * DIM
THETA, EPS = 1.0e6, 1.0e-6
SCALE = 1.0 / math.sqrt(DIM)
VOCAB = 151936


def listed():
    return [
        # A token of one short utterance: 11 s of audio are 143 audio rows and 13 prompt ids.  Two dependent
        # launches per layer over 0.6 MB each: launches and latency.
        {"name": "attn_token_short", "kind": "decode_attn", "streams": 1, "shortest": 156, "longest": 156,
         "cache": "f16", "layers": 28},
        # A step of 32 served streams with ragged contexts, short utterances to five minutes of audio.
        {"name": "attn_streams_ragged", "kind": "decode_attn", "streams": 32, "shortest": 156, "longest": 3913,
         "cache": "f16", "layers": 4},
        # The attention of a five-minute prompt.
        {"name": "attn_prompt_long", "kind": "prefill_attn", "tokens": 3913, "past": 0, "cache": "f16"},
        # The same with the drop-in API's default cache, for a prompt of odd length (80 s of audio).
        {"name": "attn_prompt_f32", "kind": "prefill_attn", "tokens": 1037, "past": 0, "cache": "f32"},
        # Projections of a step of 32 served streams, f32 weights and a converted bf16 checkpoint.
        {"name": "proj_streams_f32", "kind": "stream_proj", "size": "1.7B", "rows": 32, "weights": "f32"},
        {"name": "proj_streams_bf16", "kind": "stream_proj", "size": "1.7B", "rows": 32, "weights": "bf16"},
        # The prompt of a 3 s voice command (39 audio rows and 13 prompt ids).
        {"name": "prompt_command", "kind": "prefill", "size": "1.7B", "layers": 4, "tokens": 52, "weights": "bf16",
         "cache": "f16"},
        # The prompt of an 11 s utterance, the reference's own example: both weight types.
        {"name": "prompt_short_bf16", "kind": "prefill", "size": "1.7B", "layers": 4, "tokens": 156,
         "weights": "bf16", "cache": "f16"},
        {"name": "prompt_short_f32", "kind": "prefill", "size": "0.6B", "layers": 4, "tokens": 156, "weights": "f32",
         "cache": "f16"},
        # The prompt of five minutes of audio: both weight types.
        {"name": "prompt_long_bf16", "kind": "prefill", "size": "1.7B", "layers": 4, "tokens": 3913,
         "weights": "bf16", "cache": "f16"},
        {"name": "prompt_long_f32", "kind": "prefill", "size": "1.7B", "layers": 4, "tokens": 3913, "weights": "f32",
         "cache": "f16"},
        # One generated token behind that prompt (batch 1): the weights are streamed once.
        {"name": "token_long", "kind": "token", "size": "1.7B", "layers": 8, "past": 3930, "weights": "f32",
         "cache": "f16"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode_attn", "prefill_attn", "stream_proj", "stream_proj", "prefill", "prefill", "token"])
    size = rng.choice(sorted(SIZES))
    weights = rng.choice(["f32", "bf16"])
    cache = rng.choice(["f16", "f16", "f32"])
    if kind == "decode_attn":
        streams = _log_int(rng, 1, 32)
        a, b = sorted([_log_int(rng, 24, 3913), _log_int(rng, 24, 3913)])
        return {"kind": kind, "streams": streams, "shortest": a, "longest": b, "cache": cache,
                "layers": 28 if streams == 1 else 4}
    if kind == "prefill_attn":
        tokens = _log_int(rng, 2, 3913)
        past = rng.choice([0, 0, rng.randrange(1, 1500)])
        return {"kind": kind, "tokens": min(tokens, 3913 - past), "past": past, "cache": cache}
    if kind == "stream_proj":
        return {"kind": kind, "size": size, "rows": rng.randrange(2, 33), "weights": weights}
    if kind == "prefill":
        return {"kind": kind, "size": size, "layers": 4, "tokens": _log_int(rng, 14, 3913), "weights": weights,
                "cache": cache}
    return {"kind": kind, "size": size, "layers": 8, "past": _log_int(rng, 24, 4100), "weights": weights,
            "cache": cache}


# ------------------------------------------------------------------------------------------ inputs
class _Random:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        out = torch.empty(*shape, dtype=dtype, device="cuda")
        return out.normal_(0.0, std, generator=self.g)

    def norm_weight(self, n):
        return 1.0 + self.normal(n, std=0.1)

    def weight(self, rows, cols, kind):
        w = self.normal(rows, cols, std=0.02)
        return w.bfloat16().float() if kind == "bf16" else w


def _lengths(case):
    """Cached positions of each stream before the step: spread evenly from shortest to longest, in a mixed order."""
    n, a, b = case["streams"], case["shortest"], case["longest"]
    return [a + (b - a) * ((7 * i) % n) // max(1, n - 1) if n % 7 else a + (b - a) * i // max(1, n - 1) for i in range(n)]


def _layout(layers, streams, capacity, cache):
    return qa.KvLayout(layers, streams, KV_HEADS, DIM, capacity, qa.QA_CACHE_F16 if cache == "f16" else qa.QA_CACHE_F32)


def _cache_tensor(rnd, layers, streams, capacity, cache):
    return rnd.normal(layers, 2, streams, KV_HEADS, capacity, DIM, dtype=torch.float16 if cache == "f16" else torch.float32)


def _p(t, offset=0):
    return C.c_void_p(t.data_ptr() + offset * t.element_size())


def _workspace(nbytes):
    return torch.zeros(max(int(nbytes), 256), dtype=torch.uint8, device="cuda")


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


# ---- decode_attn
def _decode_attn_inputs(case, seed):
    rnd = _Random(seed)
    lens = _lengths(case)
    capacity = max(lens) + 256
    n = case["streams"]
    return {
        "lens": lens, "capacity": capacity,
        "qkv": rnd.normal(case["layers"], n, Q_DIM + 2 * KV_DIM),
        "q_norm": rnd.norm_weight(DIM), "k_norm": rnd.norm_weight(DIM),
        "cache": _cache_tensor(rnd, case["layers"], n, capacity, case["cache"]),
    }


def _prepare_decode_attn(case, seed):
    s = _decode_attn_inputs(case, seed)
    n, layers, lens = case["streams"], case["layers"], s["lens"]
    s["layout"] = _layout(layers, n, s["capacity"], case["cache"])
    s["past"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
    s["out"] = torch.zeros(layers, n, Q_DIM, device="cuda")
    s["ws"] = _workspace(qa.lib.qa_decode_attn_workspace_bytes(n, HEADS, s["capacity"]))
    lay = C.byref(s["layout"])
    s["calls"] = [(qa.lib.qa_decode_step_attn,
                   (_p(s["qkv"][l]), _p(s["q_norm"]), _p(s["k_norm"]), _p(s["cache"]), lay, l, _p(s["past"]), n,
                    max(lens) + 1, HEADS, THETA, EPS, SCALE, _p(s["out"][l]), _p(s["ws"]), s["ws"].numel(), _stream()))
                  for l in range(layers)]
    s["result"] = {"out": s["out"], "rows": [s["cache"][:, :, i, :, lens[i], :] for i in range(n)]}
    return s


# ---- prefill_attn
def _prefill_attn_inputs(case, seed):
    rnd = _Random(seed)
    t, past = case["tokens"], case["past"]
    capacity = t + past + 256
    return {
        "capacity": capacity, "qkv": rnd.normal(t, Q_DIM + 2 * KV_DIM),
        "q_norm": rnd.norm_weight(DIM), "k_norm": rnd.norm_weight(DIM),
        "cache": _cache_tensor(rnd, 1, 1, capacity, case["cache"]),
    }


def _prepare_prefill_attn(case, seed):
    s = _prefill_attn_inputs(case, seed)
    t, past = case["tokens"], case["past"]
    s["layout"] = _layout(1, 1, s["capacity"], case["cache"])
    s["past"] = torch.tensor([past], dtype=torch.int32, device="cuda")
    s["q"] = torch.zeros(t, Q_DIM, device="cuda")
    s["out"] = torch.zeros(t, Q_DIM, device="cuda")
    s["ws"] = _workspace(qa.lib.qa_prefill_attn_workspace_bytes(t, HEADS))
    lay = C.byref(s["layout"])
    s["calls"] = [
        (qa.lib.qa_kv_append, (_p(s["qkv"]), _p(s["q_norm"]), _p(s["k_norm"]), _p(s["q"]), _p(s["cache"]), lay, 0,
                               _p(s["past"]), 1, t, HEADS, THETA, EPS, _stream())),
        (qa.lib.qa_prefill_attn, (_p(s["q"]), _p(s["cache"]), lay, 0, 0, past, t, HEADS, SCALE, _p(s["out"]),
                                  _p(s["ws"]), s["ws"].numel(), _stream())),
    ]
    s["result"] = {"out": s["out"], "q": s["q"], "rows": s["cache"][:, :, :, :, past:past + t, :]}
    return s


# ---- stream_proj
PROJ_LAYERS = 4


def _stream_proj_inputs(case, seed):
    rnd = _Random(seed)
    z = SIZES[case["size"]]
    h, i, rows = z.hidden, z.intermediate, case["rows"]
    layers = [{
        "attn_norm": rnd.norm_weight(h), "ffn_norm": rnd.norm_weight(h),
        "qkv": rnd.weight(Q_DIM + 2 * KV_DIM, h, case["weights"]), "o": rnd.weight(h, Q_DIM, case["weights"]),
        "gu": rnd.weight(2 * i, h, case["weights"]), "down": rnd.weight(h, i, case["weights"]),
        "attn": rnd.normal(rows, Q_DIM, std=0.3),
    } for _ in range(PROJ_LAYERS)]
    return {"x0": rnd.normal(rows, h), "layers": layers}


def _prepare_stream_proj(case, seed):
    s = _stream_proj_inputs(case, seed)
    z = SIZES[case["size"]]
    h, i, rows = z.hidden, z.intermediate, case["rows"]
    w3 = Q_DIM + 2 * KV_DIM
    b16 = case["weights"] == "bf16"
    fn = qa.lib.qa_gemm_rows_fused_bf16 if b16 else qa.lib.qa_gemm_rows_fused
    if b16:
        for layer in s["layers"]:
            for k in ("qkv", "o", "gu", "down"):
                layer[k] = layer[k].bfloat16()
    parts = (h + 31) // 32
    s["stats0"] = torch.zeros(parts, 32, dtype=torch.float64, device="cuda")
    s["stats0"][:, :rows] = s["x0"].double().reshape(rows, parts, 32).square().sum(2).t()
    s["x"] = s["x0"].clone()
    s["stats"] = torch.zeros(parts, 32, dtype=torch.float64, device="cuda")
    s["qkv"] = torch.zeros(PROJ_LAYERS, rows, w3, device="cuda")
    s["act"] = torch.zeros(PROJ_LAYERS, rows, i, device="cuda")
    need = max(qa.lib.qa_gemm_rows_workspace_bytes(n, k, rows) for n, k in ((w3, h), (h, Q_DIM), (2 * i, h), (h, i)))
    s["ws"] = _workspace(need)
    ws, wb, st = _p(s["ws"]), s["ws"].numel(), _stream()
    none = C.c_void_p(None)
    calls = []
    for l, w in enumerate(s["layers"]):
        stats = s["stats0"] if l == 0 else s["stats"]
        calls += [
            (fn, (_p(w["qkv"]), w3, h, _p(s["x"]), rows, _p(s["qkv"][l]), 0, _p(w["attn_norm"]), _p(stats), parts, EPS,
                  none, 0, ws, wb, st)),
            (fn, (_p(w["o"]), h, Q_DIM, _p(w["attn"]), rows, _p(s["x"]), 1, none, none, 0, EPS, _p(s["stats"]), 0, ws,
                  wb, st)),
            (fn, (_p(w["gu"]), 2 * i, h, _p(s["x"]), rows, _p(s["act"][l]), 0, _p(w["ffn_norm"]), _p(s["stats"]), parts,
                  EPS, none, 1, ws, wb, st)),
            (fn, (_p(w["down"]), h, i, _p(s["act"][l]), rows, _p(s["x"]), 1, none, none, 0, EPS, _p(s["stats"]), 0, ws,
                  wb, st)),
        ]
    s["calls"] = calls
    s["result"] = {"qkv": s["qkv"], "act": s["act"], "x": s["x"]}
    return s


# ---- prefill and token: a decoder
class _Weights:
    """Host weights of a text model in the form qa.Decoder takes (as a loaded checkpoint holds them)."""

    ORDER = ("attn_norm", "ffn_norm", "q", "k", "v", "o", "q_norm", "k_norm", "gate", "up", "down")

    def __init__(self, case, device_layers, embd, out_norm):
        z = SIZES[case["size"]]
        self.cfg = z.config(n_layers=case["layers"])
        self.layers = [{k: w[k].cpu().numpy() for k in self.ORDER} for w in device_layers]
        self.embd = embd.cpu().numpy()
        self.out_norm = out_norm.cpu().numpy()

    def weights(self):
        table = (qa.LayerWeights * len(self.layers))()
        for row, w in zip(table, self.layers):
            for k in self.ORDER:
                setattr(row, k, w[k].ctypes.data_as(qa.fp))
        top = qa.ModelWeights(table, self.embd.ctypes.data_as(qa.fp), self.out_norm.ctypes.data_as(qa.fp),
                              self.embd.ctypes.data_as(qa.fp))
        return table, top


def _model_inputs(case, seed):
    rnd = _Random(seed)
    z = SIZES[case["size"]]
    h, i, kind = z.hidden, z.intermediate, case["weights"]

    def norm(n):
        w = rnd.norm_weight(n)
        return w.bfloat16().float() if kind == "bf16" else w

    layers = [{
        "attn_norm": norm(h), "ffn_norm": norm(h), "q": rnd.weight(Q_DIM, h, kind), "k": rnd.weight(KV_DIM, h, kind),
        "v": rnd.weight(KV_DIM, h, kind), "o": rnd.weight(h, Q_DIM, kind), "q_norm": norm(DIM), "k_norm": norm(DIM),
        "gate": rnd.weight(i, h, kind), "up": rnd.weight(i, h, kind), "down": rnd.weight(h, i, kind),
    } for _ in range(case["layers"])]
    tokens = case.get("tokens", 1)
    past = case.get("past", 0)
    capacity = tokens + past + 256
    return {
        "layers": layers, "embd": rnd.weight(VOCAB, h, kind), "out_norm": norm(h), "x": rnd.normal(tokens, h),
        "past": past, "tokens": tokens, "capacity": capacity,
        "cached": _cache_tensor(rnd, case["layers"], 1, capacity, case["cache"]) if past else None,
    }


class _DeviceView:
    """A decoder's cache for torch.as_tensor, whose tensor keeps this object and so the decoder that owns the memory."""

    def __init__(self, decoder, address, shape, cache):
        self.decoder = decoder
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f2" if cache == "f16" else "<f4",
                                         "data": (address, False), "version": 2, "strides": None}


def _prepare_model(case, seed):
    s = _model_inputs(case, seed)
    weights = _Weights(case, s.pop("layers"), s.pop("embd"), s.pop("out_norm"))
    dec = qa.Decoder(weights, 1, s["capacity"], qa.QA_CACHE_F16 if case["cache"] == "f16" else qa.QA_CACHE_F32)
    dec.model = None   # the decoder holds its own copies
    assert dec.weights_bf16 == (case["weights"] == "bf16")
    s["decoder"] = dec
    s["x"] = s["x"].cpu().numpy()
    address, lay = dec.cache()
    shape = (lay.n_layers, 2, lay.n_streams, lay.n_kv_heads, lay.max_seq, lay.head_dim)
    view = torch.as_tensor(_DeviceView(dec, address, shape, case["cache"]), device="cuda")
    cached = s.pop("cached")
    if cached is not None:
        view.copy_(cached)
    s["rows"] = view[:, :, :, :, s["past"]:s["past"] + s["tokens"], :]
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "token"):
        return _prepare_model(case, seed)
    return {"decode_attn": _prepare_decode_attn, "prefill_attn": _prepare_prefill_attn,
            "stream_proj": _prepare_stream_proj}[kind](case, seed)


def run(state):
    if "decoder" in state:
        logits = state["decoder"].forward(state["x"], state["past"])
        return {"logits": logits, "rows": state["rows"]}
    if "x0" in state:
        state["x"].copy_(state["x0"])   # the step's input rows
    for fn, args in state["calls"]:
        rc = fn(*args)
        if rc:
            qa.check(rc)
    return state["result"]


# ------------------------------------------------------------------------------------------ work
def _layer_params(z):
    return (Q_DIM + 2 * KV_DIM) * z.hidden + z.hidden * Q_DIM + 3 * z.hidden * z.intermediate


def work(case):
    kind = case["kind"]
    if kind == "decode_attn":
        esz = 2 if case["cache"] == "f16" else 4
        positions = sum(n + 1 for n in _lengths(case))
        n, layers = case["streams"], case["layers"]
        per_row = 2 * KV_DIM * esz
        return {"bytes": layers * (positions * per_row + n * 4 * (Q_DIM + 2 * KV_DIM + Q_DIM)),
                "flops": layers * positions * 4 * Q_DIM}
    if kind == "prefill_attn":
        esz = 2 if case["cache"] == "f16" else 4
        t, past = case["tokens"], case["past"]
        pairs = t * past + t * (t + 1) // 2
        return {"bytes": t * 4 * (Q_DIM + 2 * KV_DIM + 2 * Q_DIM) + (2 * t + past) * 2 * KV_DIM * esz,
                "flops": 4 * Q_DIM * pairs}
    z = SIZES[case["size"]]
    wsz = 2 if case["weights"] == "bf16" else 4
    params = _layer_params(z)
    if kind == "stream_proj":
        rows = case["rows"]
        acts = rows * 4 * (3 * z.hidden + Q_DIM + 2 * KV_DIM + Q_DIM + 2 * z.intermediate)
        return {"bytes": PROJ_LAYERS * (params * wsz + acts), "flops": PROJ_LAYERS * 2 * rows * params}
    t, past, layers = case.get("tokens", 1), case.get("past", 0), case["layers"]
    esz = 2 if case["cache"] == "f16" else 4
    pairs = t * past + t * (t + 1) // 2
    head = VOCAB * z.hidden
    return {"bytes": (layers * params + head) * wsz + layers * (2 * t + past) * 2 * KV_DIM * esz + 4 * t * z.hidden + 4 * VOCAB,
            "flops": layers * (2 * t * params + 4 * Q_DIM * pairs) + 2 * head}


# ------------------------------------------------------------------------------------------ tolerance
def tolerance(case):
    """About four times the error against 64 bits, which another order of the f32 sums, or another place of the
    f16 roundings, can show at most: f32 paths 2e-7 to 7e-7; attention over f16 caches 2.9e-4 to 3.7e-4 (q and
    the probabilities round to f16); whole calls over f16 caches 1e-4 to 2.5e-4 (the stored rows' rounding
    included).  "max": single elements beside the root mean square of outputs whose scale varies by position."""
    kind = case["kind"]
    if kind == "stream_proj":
        return {"rel": 4.0e-6, "max": 4.0e-4}
    if kind in ("decode_attn", "prefill_attn"):
        return {"rel": 1.4e-3, "max": 2.0e-2} if case["cache"] == "f16" else {"rel": 4.0e-6, "max": 4.0e-4}
    return {"rel": 1.0e-3, "max": 2.0e-2} if case["cache"] == "f16" else {"rel": 4.0e-6, "max": 4.0e-4}


# ------------------------------------------------------------------------------------------ 64-bit results
def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    """x [..., n, DIM] at positions pos [n]: NEOX pairs (i, i + DIM / 2)."""
    half = DIM // 2
    inv = torch.exp(-math.log(THETA) * torch.arange(half, dtype=torch.float64, device=x.device) * 2 / DIM)
    ang = pos.double()[:, None] * inv
    c, s = ang.cos(), ang.sin()
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _prep(qkv, q_norm, k_norm, pos):
    """Rows [n, q|k|v] to q [HEADS, n, DIM], k and v [KV_HEADS, n, DIM], normalised and rotated."""
    n = qkv.shape[0]
    q = qkv[:, :Q_DIM].reshape(n, HEADS, DIM).transpose(0, 1)
    k = qkv[:, Q_DIM:Q_DIM + KV_DIM].reshape(n, KV_HEADS, DIM).transpose(0, 1)
    v = qkv[:, Q_DIM + KV_DIM:].reshape(n, KV_HEADS, DIM).transpose(0, 1)
    return _rope(_rms(q, q_norm), pos), _rope(_rms(k, k_norm), pos), v


def _attend(q, k, v, past):
    """Causal attention of q [HEADS, n, DIM] at positions past .. over k, v [KV_HEADS, past + n, DIM]: [n, Q_DIM]."""
    n, total = q.shape[1], k.shape[1]
    out = torch.empty(n, Q_DIM, dtype=torch.float64, device=q.device)
    keep = torch.arange(total, device=q.device)[None] <= past + torch.arange(n, device=q.device)[:, None]
    for h in range(HEADS):
        kt = k[h // 2].t().contiguous()
        s = (q[h] @ kt) * SCALE
        s = s.masked_fill(~keep, -math.inf)
        out[:, h * DIM:(h + 1) * DIM] = torch.softmax(s, -1) @ v[h // 2]
    return out


def _exact_decode_attn(case, seed):
    s = _decode_attn_inputs(case, seed)
    n, layers, lens = case["streams"], case["layers"], s["lens"]
    out = torch.zeros(layers, n, Q_DIM, dtype=torch.float64, device="cuda")
    rows = [torch.zeros(layers, 2, KV_HEADS, DIM, dtype=torch.float64, device="cuda") for _ in range(n)]
    for l in range(layers):
        for i, past in enumerate(lens):
            pos = torch.tensor([past], device="cuda")
            q, k, v = _prep(s["qkv"][l, i:i + 1].double(), s["q_norm"], s["k_norm"], pos)
            rows[i][l, 0], rows[i][l, 1] = k[:, 0], v[:, 0]
            kk = torch.cat([s["cache"][l, 0, i, :, :past].double(), k], 1)
            vv = torch.cat([s["cache"][l, 1, i, :, :past].double(), v], 1)
            out[l, i] = _attend(q, kk, vv, past)[0]
    return {"out": out, "rows": rows}


def _exact_prefill_attn(case, seed):
    s = _prefill_attn_inputs(case, seed)
    t, past = case["tokens"], case["past"]
    q, k, v = _prep(s["qkv"].double(), s["q_norm"], s["k_norm"], past + torch.arange(t, device="cuda"))
    kk = torch.cat([s["cache"][0, 0, 0, :, :past].double(), k], 1)
    vv = torch.cat([s["cache"][0, 1, 0, :, :past].double(), v], 1)
    return {"out": _attend(q, kk, vv, past), "q": q.transpose(0, 1).reshape(t, Q_DIM),
            "rows": torch.stack([k, v])[None, :, None]}


def _swiglu(gu, i):
    return torch.nn.functional.silu(gu[:, :i]) * gu[:, i:]


def _exact_stream_proj(case, seed):
    s = _stream_proj_inputs(case, seed)
    i = SIZES[case["size"]].intermediate
    x = s["x0"].double()
    qkv, act = [], []
    for w in s["layers"]:
        qkv.append(_rms(x, w["attn_norm"]) @ w["qkv"].double().t())
        x = x + w["attn"].double() @ w["o"].double().t()
        act.append(_swiglu(_rms(x, w["ffn_norm"]) @ w["gu"].double().t(), i))
        x = x + act[-1] @ w["down"].double().t()
    return {"qkv": torch.stack(qkv), "act": torch.stack(act), "x": x}


def _exact_model(case, seed):
    s = _model_inputs(case, seed)
    i = SIZES[case["size"]].intermediate
    t, past = s["tokens"], s["past"]
    pos = past + torch.arange(t, device="cuda")
    x = s["x"].double()
    rows = []
    for l, w in enumerate(s["layers"]):
        h = _rms(x, w["attn_norm"])
        qkv = torch.cat([h @ w[k].double().t() for k in ("q", "k", "v")], 1)
        q, k, v = _prep(qkv, w["q_norm"], w["k_norm"], pos)
        rows.append(torch.stack([k, v])[:, None])
        kk, vv = k, v
        if past:
            kk = torch.cat([s["cached"][l, 0, 0, :, :past].double(), k], 1)
            vv = torch.cat([s["cached"][l, 1, 0, :, :past].double(), v], 1)
        x = x + _attend(q, kk, vv, past) @ w["o"].double().t()
        h = _rms(x, w["ffn_norm"])
        gu = torch.cat([h @ w[k].double().t() for k in ("gate", "up")], 1)
        x = x + _swiglu(gu, i) @ w["down"].double().t()
    last = _rms(x[-1:], s["out_norm"])[0]
    logits = torch.cat([part.double() @ last for part in s["embd"].split(16384)])
    return {"logits": logits.cpu().numpy(), "rows": torch.stack(rows)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "token"):
        return _exact_model(case, seed)
    return {"decode_attn": _exact_decode_attn, "prefill_attn": _exact_prefill_attn,
            "stream_proj": _exact_stream_proj}[kind](case, seed)
