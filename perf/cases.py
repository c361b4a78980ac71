"""The work this library is measured on, through its public entry points.

Three groups:

* projections on device buffers (``zq.*_dev``): what a runtime that keeps its
  activations in HBM enqueues -- decode GEMVs from the smallest (k/v of a
  4096-wide layer) to the vocabulary projection, the fused FFN half of a
  layer, prefill GEMMs with int8 and with fp32 activations;
* the host-pointer slot (``zq.gemm`` / ``zq.gemv`` on numpy arrays with resident
  weights): what a CPU runtime that hands single projections to the GPU calls;
* the device-resident decoder (``Model``): a prefill, and a prefill followed
  by decode steps.

Sizes are those of the benchmark's decoder (hidden 4096, 8 KV heads of 128,
FFN 14336, vocabulary 128256; the decoder itself with fewer layers and a
smaller vocabulary) and generic ones around them.  Weights are quantised
normals, activations normals with a few large channels, as the inputs of a
transformer's projections have.
"""
import math

import numpy as np
import torch

from zeninfer_amd import gguf, zq
from zeninfer_amd.model import PREFILL_F32, PREFILL_INT8, Model

FMT = zq.FORMATS
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}
TAIL = zq.WEIGHT_TAIL_PAD
DEV = "cuda:0"
EPS = 1e-5


# ---------------------------------------------------------------- cases ----
def listed():
    return [
        # The smallest decode projection: k or v of one layer, one launch.
        {"name": "gemv_kv_q8_0", "kind": "gemv", "fmt": "Q8_0", "rows": "1024", "cols": 4096},
        # Decode q|k|v of one layer in one batched launch.
        {"name": "gemv_qkv_q4_k", "kind": "gemv", "fmt": "Q4_K", "rows": "4096+1024+1024", "cols": 4096},
        # The vocabulary projection of a decode step.
        {"name": "gemv_head_q6_k", "kind": "gemv", "fmt": "Q6_K", "rows": "128256", "cols": 4096},
        # o, residual, norm, gate|up, SiLU*up and down of one decode step.
        {"name": "ffn_step_q8_0", "kind": "ffn", "fmt": "Q8_0", "hidden": 4096, "attn": 4096, "ffn": 14336},
        # Prefill of a 512-token prompt with int8 activations (the route the
        # decoder takes for Q8_0), one FFN projection.
        {"name": "gemm_i8_q8_0_m512", "kind": "gemm", "fmt": "Q8_0", "act": "int8", "tokens": 512, "rows": "14336",
         "cols": 4096},
        # A short, odd prompt with int8 activations.
        {"name": "gemm_i8_q4_0_m33", "kind": "gemm", "fmt": "Q4_0", "act": "int8", "tokens": 33, "rows": "4096",
         "cols": 14336},
        # The same 512-token prefill with the default (fp32) activations.
        {"name": "gemm_f32_q8_0_m512", "kind": "gemm", "fmt": "Q8_0", "act": "f32", "tokens": 512, "rows": "14336",
         "cols": 4096},
        # q|k|v of a short chat turn: few tokens, fp32 activations.
        {"name": "gemm_f32_qkv_q4_k_m19", "kind": "gemm", "fmt": "Q4_K", "act": "f32", "tokens": 19,
         "rows": "4096+1024+1024", "cols": 4096},
        # A long prompt's down projection on a super-block format.
        {"name": "gemm_f32_q6_k_m1000", "kind": "gemm", "fmt": "Q6_K", "act": "f32", "tokens": 1000, "rows": "4096",
         "cols": 14336},
        # A projection handed over by a CPU runtime: host activations in, host
        # outputs out, weights resident.
        {"name": "host_gemm_q4_0_m64", "kind": "host_gemm", "fmt": "Q4_0", "act": "f32", "tokens": 64, "rows": "4096",
         "cols": 4096},
        # A whole prefill: the benchmark's decoder at two layers, int8 activations.
        {"name": "model_prefill_q8_0", "kind": "model", "fmt": "Q8_0", "mode": "int8", "layers": 2, "hidden": 4096,
         "heads": 32, "kv_heads": 8, "ffn": 14336, "vocab": 32000, "prompt": 512, "steps": 0},
        # A short prompt and the decode steps after it, super-block projections.
        {"name": "model_decode_q5_k", "kind": "model", "fmt": "Q5_K", "mode": "f32", "layers": 2, "hidden": 4096,
         "heads": 32, "kv_heads": 8, "ffn": 14336, "vocab": 32000, "prompt": 70, "steps": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(case):
    """Rows of a case's weight matrices, written "4096" or "4096+1024+1024"."""
    return [int(r) for r in case["rows"].split("+")] if "rows" in case else None


def _cols(rng, fmt, act, lo=256, hi=16384):
    step = 256 if BLOCK[fmt][0] == 256 or rng.random() < 0.6 else (64 if act == "int8" else 32)
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "ffn", "gemm", "gemm", "gemm", "gemm", "host_gemv", "host_gemm", "model"])
    fmt = rng.choice(sorted(FMT))
    if kind == "ffn":
        step = 256 if BLOCK[fmt][0] == 256 else 64
        dims = {k: max(step, _log(rng, lo, hi) // step * step)
                for k, lo, hi in (("hidden", 512, 6144), ("attn", 512, 6144), ("ffn", 1024, 16384))}
        return {"kind": kind, "fmt": fmt, **dims}
    if kind == "model":
        heads, kv = rng.choice([(32, 8), (24, 8), (16, 16), (16, 2)])
        return {"kind": kind, "fmt": fmt, "mode": "int8" if fmt in ("Q8_0", "Q4_0") and rng.random() < 0.5 else "f32",
                "layers": rng.randint(1, 2), "hidden": 256 * rng.randint(4, 16), "heads": heads, "kv_heads": kv,
                "ffn": 256 * rng.randint(8, 56), "vocab": _log(rng, 4000, 32000), "prompt": _log(rng, 2, 500),
                "steps": rng.randint(0, 8)}
    if kind in ("gemv", "host_gemv"):
        rows = [_log(rng, 64, 32000)] if rng.random() < 0.6 else [_log(rng, 64, 8192) for _ in range(rng.randint(2, 3))]
        if kind == "host_gemv":
            rows = [max(r, 1500) for r in rows]
            return {"kind": kind, "fmt": fmt, "rows": "+".join(map(str, rows)), "cols": _cols(rng, fmt, "f32", 1024)}
        return {"kind": kind, "fmt": fmt, "rows": "+".join(map(str, rows)), "cols": _cols(rng, fmt, "f32")}
    act = "int8" if fmt in ("Q8_0", "Q4_0") and rng.random() < 0.5 else "f32"
    tokens = _log(rng, 1, 1000 if kind == "gemm" else 200)
    rows = [_log(rng, 128, 14336)] if rng.random() < 0.7 else [_log(rng, 128, 4096) for _ in range(rng.randint(2, 3))]
    cols = _cols(rng, fmt, act, 512, 14336)
    if kind == "host_gemm":  # the slot keeps projections under 256 Ki weights on the CPU
        rows, cols = [max(r, 1100) for r in rows[:1]], max(cols, 1024)
    return {"kind": kind, "fmt": fmt, "act": act, "tokens": tokens, "rows": "+".join(map(str, rows)), "cols": cols}


# --------------------------------------------------------------- inputs ----
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _half_bytes(d):
    return d.to(torch.float16).contiguous().view(torch.uint8).reshape(*d.shape, 2)


def _blocks(fmt, n, g):
    """n blocks of a quantised weight matrix as uint8 [n, block bytes]; weights of about 0.02 standard deviation."""
    if fmt in ("Q8_0", "Q4_0"):
        w = torch.randn(n, 32, generator=g, device=DEV) * 0.02
        if fmt == "Q8_0":
            d = w.abs().amax(1, keepdim=True) / 127.0
            q = torch.clamp(torch.round(w / d), -127, 127).to(torch.int8).view(torch.uint8)
            return torch.cat([_half_bytes(d).reshape(n, 2), q], 1)
        top = w.gather(1, w.abs().argmax(1, keepdim=True))
        d = top / -8.0
        q = torch.clamp(torch.floor(w / d + 8.5), 0, 15).to(torch.uint8)
        return torch.cat([_half_bytes(d).reshape(n, 2), q[:, :16] | (q[:, 16:] << 4)], 1)
    if fmt == "Q6_K":
        q = torch.clamp(torch.round(torch.randn(n, 256, generator=g, device=DEV) * 10 + 32), 0, 63).to(torch.uint8)
        sc = torch.randint(40, 128, (n, 16), generator=g, device=DEV)
        sc = (sc * (torch.randint(0, 2, (n, 16), generator=g, device=DEV) * 2 - 1)).to(torch.int8).view(torch.uint8)
        d = (0.7 + 0.6 * torch.rand(n, generator=g, device=DEV)) * 2.4e-5
        q = q.reshape(n, 2, 4, 32)
        lo = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        hi = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        return torch.cat([lo.reshape(n, 128), hi.reshape(n, 64), sc, _half_bytes(d)], 1)
    top = 15 if fmt == "Q4_K" else 31
    mid = (top + 1) / 2 - 0.5
    q = torch.clamp(torch.round(torch.randn(n, 256, generator=g, device=DEV) * (top / 5.0) + mid), 0, top).to(torch.uint8)
    sc = torch.randint(20, 64, (n, 8), generator=g, device=DEV).to(torch.uint8)
    mn = torch.clamp(sc.float() + torch.randint(-6, 7, (n, 8), generator=g, device=DEV), 0, 63).to(torch.uint8)
    d = (0.7 + 0.6 * torch.rand(n, generator=g, device=DEV)) * (0.02 * 5.0 / (top * 42.0))
    head = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                      (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    q = q.reshape(n, 8, 32)
    nib = ((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).reshape(n, 128)
    parts = [_half_bytes(d), _half_bytes(d * mid), head]
    if fmt == "Q5_K":
        parts.append(sum((q[:, j] >> 4) << j for j in range(8)))
    return torch.cat(parts + [nib], 1)


def _weights(fmt, rows, cols, g):
    """A device weight buffer: the rows' blocks, then the tail pad."""
    be, bb = BLOCK[fmt]
    total = rows * (cols // be)
    buf = torch.zeros(total * bb + TAIL, dtype=torch.uint8, device=DEV)
    step = (1 << 26) // be
    for b in range(0, total, step):
        n = min(step, total - b)
        buf[b * bb:(b + n) * bb] = _blocks(fmt, n, g).reshape(-1)
    return buf


def _acts(tokens, cols, g):
    x = torch.randn(tokens, cols, generator=g, device=DEV)
    x[:, torch.randint(0, cols, (max(1, cols // 512),), generator=g, device=DEV)] *= 12.0
    return x


def _act_mode(case):
    return zq.ACT_INT8 if case["act"] == "int8" else zq.ACT_DEFAULT


def _tokens(case, seed):
    n = case["prompt"] + case["steps"]
    return np.random.default_rng(seed).integers(0, case["vocab"], n).astype(np.uint32)


def _model_tensors(case, seed):
    """(GGUF name, format or None, rows, cols, device tensor) of every tensor of the case's decoder, one at a time."""
    H, F, Q, KV, V = case["hidden"], case["ffn"], case["heads"] * 128, case["kv_heads"] * 128, case["vocab"]
    fmt, g = case["fmt"], _gen(seed)
    names = [("token_embd", "Q8_0", V, H)]
    for layer in range(case["layers"]):
        p = "blk.%d." % layer
        names += [(p + "attn_norm", None, 1, H), (p + "attn_q", fmt, Q, H), (p + "attn_k", fmt, KV, H),
                  (p + "attn_v", fmt, KV, H), (p + "attn_output", fmt, H, Q), (p + "ffn_norm", None, 1, H),
                  (p + "ffn_gate", fmt, F, H), (p + "ffn_up", fmt, F, H), (p + "ffn_down", fmt, H, F)]
    for name, f, rows, cols in names + [("output_norm", None, 1, H), ("output", "Q8_0", V, H)]:
        yield name, f, rows, cols, (1.0 + 0.1 * torch.randn(cols, generator=g, device=DEV) if f is None else
                                    _weights(f, rows, cols, g))


def _model(case, seed):
    w = gguf.GGUFWriter()
    for key, t, v in [("general.architecture", gguf.STRING, "llama"), ("llama.embedding_length", gguf.U32, case["hidden"]),
                      ("llama.block_count", gguf.U32, case["layers"]),
                      ("llama.attention.head_count", gguf.U32, case["heads"]),
                      ("llama.attention.head_count_kv", gguf.U32, case["kv_heads"]),
                      ("llama.attention.key_length", gguf.U32, 128), ("llama.feed_forward_length", gguf.U32, case["ffn"]),
                      ("llama.context_length", gguf.U32, 8192), ("llama.rope.dimension_count", gguf.U32, 128),
                      ("llama.rope.freq_base", gguf.F32, 500000.0),
                      ("llama.attention.layer_norm_rms_epsilon", gguf.F32, EPS)]:
        w.add_meta(key, t, v)
    for name, f, rows, cols, t in _model_tensors(case, seed):
        if f is None:
            w.add_tensor(name + ".weight", [cols], gguf.GGML_F32, t.cpu().numpy().tobytes())
        else:
            w.add_tensor(name + ".weight", [cols, rows], FMT[f], memoryview(t[:t.numel() - TAIL].cpu().numpy()))
    with gguf.GGUFFile(data=w.to_bytes()) as file:
        m = Model.from_gguf(file, 1024)
    m.set_prefill_mode(PREFILL_INT8 if case["mode"] == "int8" else PREFILL_F32)
    return m


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "model":
        s.update(model=_model(case, seed), tokens=_tokens(case, seed))
        return s
    g = _gen(seed)
    fmt = case["fmt"]
    if kind == "ffn":
        H, A, F = case["hidden"], case["attn"], case["ffn"]
        s.update(wo=_weights(fmt, H, A, g), wg=_weights(fmt, F, H, g), wu=_weights(fmt, F, H, g),
                 wd=_weights(fmt, H, F, g), norm=1.0 + 0.1 * torch.randn(H, generator=g, device=DEV),
                 x=_acts(1, H, g)[0].contiguous(), att=_acts(1, A, g)[0].contiguous(), out=torch.empty(H, device=DEV))
        s["ws_bytes"] = zq.ffn_residual_workspace_bytes(H, F)
        s["ws"] = torch.empty(max(s["ws_bytes"], 16), dtype=torch.uint8, device=DEV)
        return s
    cols, tokens, rows = case["cols"], case.get("tokens", 1), _rows(case)
    ws = [_weights(fmt, r, cols, g) for r in rows]
    x = _acts(tokens, cols, g)
    if kind.startswith("host"):
        s["w"] = [w.cpu().numpy() for w in ws]
        s["x"] = x.cpu().numpy()
        for w in s["w"]:  # a new tensor, possibly at the address of one that is gone
            zq.release(w)
        return s
    s.update(w=ws, x=x.reshape(-1), y=[torch.empty(tokens * r, device=DEV) for r in rows])
    if kind == "gemm":
        act = _act_mode(case)
        n = (zq.gemm_workspace_bytes(FMT[fmt], tokens, rows[0], cols, act) if len(ws) == 1 else
             zq.gemm_batch_workspace_bytes(FMT[fmt], rows, tokens, cols, act))
        s["ws_bytes"], s["ws"] = n, torch.empty(max(n, 16), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "model":
        m, t, n = state["model"], state["tokens"], case["prompt"]
        out = [m.prefill(t[:n])[1]]
        for k in range(case["steps"]):
            out.append(m.decode(t[n + k])[1])
        return out
    fmt, rows, cols = FMT[case["fmt"]], _rows(case), case.get("cols")
    if kind == "host_gemv":
        if len(rows) > 1:
            return zq.gemv_batch(fmt, state["w"], state["x"], rows, cols)
        return zq.gemv(fmt, state["w"][0], state["x"], rows[0], cols)
    if kind == "host_gemm":
        return zq.gemm(fmt, state["w"][0], state["x"], case["tokens"], rows[0], cols, _act_mode(case))
    stream = torch.cuda.current_stream()
    if kind == "ffn":
        zq.ffn_residual_fused_dev(fmt, state["wo"], state["wg"], state["wu"], state["wd"], state["norm"], state["x"],
                                  state["att"], state["out"], case["hidden"], case["attn"], case["ffn"], EPS,
                                  state["ws"], state["ws_bytes"], stream)
        return state["out"]
    if kind == "gemv":
        if len(rows) > 1:
            zq.gemv_batch_dev(fmt, state["x"], list(zip(state["w"], state["y"], rows)), cols, stream)
        else:
            zq.gemv_dev(fmt, state["w"][0], state["x"], state["y"][0], rows[0], cols, stream)
        return state["y"]
    if len(rows) > 1:
        zq.gemm_batch_dev(fmt, state["x"], list(zip(state["w"], state["y"], rows)), case["tokens"], cols,
                          _act_mode(case), state["ws"], state["ws_bytes"], stream)
    else:
        zq.gemm_dev(fmt, state["w"][0], state["x"], state["y"][0], case["tokens"], rows[0], cols, _act_mode(case),
                    state["ws"], state["ws_bytes"], stream)
    return state["y"]


# ----------------------------------------------------- work, tolerances ----
def _wbytes(fmt, rows, cols):
    be, bb = BLOCK[fmt]
    return rows * (cols // be) * bb


def work(case):
    kind, fmt = case["kind"], case["fmt"]
    if kind == "ffn":
        H, A, F = case["hidden"], case["attn"], case["ffn"]
        return {"bytes": _wbytes(fmt, H, A) + 2 * _wbytes(fmt, F, H) + _wbytes(fmt, H, F) + 4 * (3 * H + A),
                "flops": 2 * (H * A + 3 * H * F)}
    if kind == "model":
        H, F, Q, KV, V = case["hidden"], case["ffn"], case["heads"] * 128, case["kv_heads"] * 128, case["vocab"]
        shapes = [(Q, H), (KV, H), (KV, H), (H, Q), (F, H), (F, H), (H, F)]
        wb = case["layers"] * sum(_wbytes(fmt, r, c) for r, c in shapes)
        per_tok = 2 * case["layers"] * sum(r * c for r, c in shapes)
        head, headb = 2 * V * H, _wbytes("Q8_0", V, H) + 4 * V
        T, n = case["prompt"], case["steps"]
        att = case["layers"] * 4 * Q * (T * (T + 1) // 2 + sum(T + i + 1 for i in range(n)))
        kv = case["layers"] * 8 * KV * (T + sum(T + i + 1 for i in range(n)))
        return {"bytes": (1 + n) * (wb + headb) + kv, "flops": (T + n) * per_tok + (1 + n) * head + att}
    T, cols = case.get("tokens", 1), case["cols"]
    return {"bytes": sum(_wbytes(fmt, r, cols) + 4 * T * r for r in _rows(case)) + 4 * T * cols,
            "flops": sum(2 * T * r * cols for r in _rows(case))}


def tolerance(case):
    # Projections are 32-bit sums of exact products (the int8 route's block
    # dots are whole numbers and its quantiser has one right result): 1e-7 to
    # 2e-6 off the float64 product, the long rows furthest.
    if case["kind"] != "model":
        return {"rel": 1e-5}
    # The decoder on fp32 activations is 3e-6 off float64.  With int8
    # activations another order of one layer's sums flips the rounding of
    # activations in those after it: 1.5e-2 off the same arithmetic in float64.
    return {"rel": 6e-2} if case["mode"] == "int8" else {"rel": 1.5e-5}


# ---------------------------------------------------------------- exact ----
def _decode(fmt, raw):
    """Blocks [n, block bytes] -> float64 [n, elements]."""
    def half(a):
        return raw[:, a:a + 2].contiguous().view(torch.float16).double()

    n = raw.shape[0]
    if fmt == "Q8_0":
        return raw[:, 2:].contiguous().view(torch.int8).double() * half(0)
    if fmt == "Q4_0":
        return (torch.cat([raw[:, 2:] & 15, raw[:, 2:] >> 4], 1).double() - 8) * half(0)
    if fmt == "Q6_K":
        lo, hi = raw[:, :128].reshape(n, 2, 2, 32), raw[:, 128:192].reshape(n, 2, 32)
        q = torch.stack([((lo[:, :, k & 1] >> (4 * (k >> 1))) & 15) | (((hi >> (2 * k)) & 3) << 4) for k in range(4)], 2)
        sc = raw[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
        return ((q.reshape(n, 2, 4, 2, 16).double() - 32) * sc).reshape(n, 256) * half(208)
    s = raw[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    nib = raw[:, -128:].reshape(n, 4, 32)
    q = torch.stack([nib & 15, nib >> 4], 2).reshape(n, 8, 32)
    if fmt == "Q5_K":
        q = q | torch.stack([((raw[:, 16:48] >> j) & 1) << 4 for j in range(8)], 1)
    return ((q.double() * sc[:, :, None]) * half(0)[:, :, None] - (mn * half(2))[:, :, None]).reshape(n, 256)


def _product(fmt, w, X, rows, cols):
    """X [tokens, cols] float64 times the matrix's transpose, in float64, some rows at a time."""
    be, bb = BLOCK[fmt]
    per, out = cols // be, []
    step = max(1, (1 << 25) // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        W = _decode(fmt, w[r * per * bb:(r + n) * per * bb].reshape(n * per, bb)).reshape(n, cols)
        out.append(X @ W.t().contiguous())
    return torch.cat(out, 1)


def _quantised(X):
    """The values int8 activations stand for: per 32, d = amax / 127 and whole multiples of it (each step rounded to
    32 bits as the quantiser's definition has it), halves away from zero."""
    b = X.double().reshape(X.shape[0], -1, 32)
    d = (b.abs().amax(2, keepdim=True) / 127.0).float().double()
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d)).float().double()
    v = torch.clamp((b * inv).float().double(), -127, 127)
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    return (q * d).reshape(X.shape)


def _model_exact(case, seed):
    H, nh, kh, V = case["hidden"], case["heads"], case["kv_heads"], case["vocab"]
    toks = torch.from_numpy(_tokens(case, seed).astype(np.int64)).to(DEV)
    T, P = toks.numel(), case["prompt"]

    parts = {name: (f, rows, cols, t) for name, f, rows, cols, t in _model_tensors(case, seed)}

    def norm(name, v):
        v = v / torch.sqrt((v * v).mean(-1, keepdim=True) + EPS)
        return v * parts[name][3].double()

    be, bb = BLOCK["Q8_0"]
    emb = parts["token_embd"][3][:V * (H // be) * bb].reshape(V, -1)[toks]
    h = _decode("Q8_0", emb.reshape(-1, bb)).reshape(T, H)
    freq = np.float32(500000.0) ** (np.float32(-2.0) * np.arange(64, dtype=np.float32) / np.float32(128))
    ang = torch.from_numpy(np.arange(T, dtype=np.float32)[:, None] * freq[None]).to(DEV).double()
    cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def rope(v, heads):
        v = v.reshape(T, heads, 64, 2)
        a, b = v[..., 0], v[..., 1]
        return torch.stack([a * cs - b * sn, a * sn + b * cs], -1).reshape(T, heads, 128)

    mask = torch.full((T, T), -math.inf, device=DEV, dtype=torch.float64).triu(1)
    for layer in range(case["layers"]):
        def proj(name, v):
            f, rows, cols, w = parts["blk.%d.%s" % (layer, name)]
            return _product(f, w, v, rows, cols)

        a = norm("blk.%d.attn_norm" % layer, h)
        q, k, v = proj("attn_q", a), proj("attn_k", a), proj("attn_v", a)
        q, k, v = rope(q, nh), rope(k, kh), v.reshape(T, kh, 128)
        att = torch.empty(T, nh, 128, device=DEV, dtype=torch.float64)
        for hd in range(nh):
            g = hd // (nh // kh)
            p = torch.softmax(q[:, hd].contiguous() @ k[:, g].t().contiguous() / math.sqrt(128.0) + mask, -1)
            att[:, hd] = p @ v[:, g].contiguous()
        h = h + proj("attn_output", att.reshape(T, nh * 128))
        a = norm("blk.%d.ffn_norm" % layer, h)
        h = h + proj("ffn_down", torch.nn.functional.silu(proj("ffn_gate", a)) * proj("ffn_up", a))
    out = _product("Q8_0", parts["output"][3], norm("output_norm", h[P - 1:]), V, H)
    return [r.cpu().numpy() for r in out]


def exact(case, seed):
    kind, fmt = case["kind"], case["fmt"]
    if kind == "model":
        # int8 activations of a deep chain have no one value to compare with
        return None if case["mode"] == "int8" else _model_exact(case, seed)
    s = prepare(case, seed)
    if kind == "ffn":
        H, A, F = case["hidden"], case["attn"], case["ffn"]
        h1 = _product(fmt, s["wo"], s["att"].double()[None], H, A) + s["x"].double()
        a = h1 / torch.sqrt((h1 * h1).mean() + EPS) * s["norm"].double()
        f = torch.nn.functional.silu(_product(fmt, s["wg"], a, F, H)) * _product(fmt, s["wu"], a, F, H)
        return (h1 + _product(fmt, s["wd"], f, H, F))[0]
    T, cols = case.get("tokens", 1), case["cols"]
    X = torch.as_tensor(s["x"]).to(DEV).reshape(T, cols)
    X = _quantised(X) if case.get("act") == "int8" else X.double()
    out = [_product(fmt, torch.as_tensor(w).to(DEV), X, r, cols).reshape(-1) for w, r in zip(s["w"], _rows(case))]
    if kind == "host_gemv":
        out = [o.cpu().numpy() for o in out]
        return out if len(out) > 1 else out[0]
    return out[0].cpu().numpy() if kind == "host_gemm" else out
