"""The calls that a user of this framework makes, as cases that can be timed.

Shapes are those of the synthetic BitNet b1.58 2B configuration
(0xbitnet_amd/synth.py: 30 layers, hidden 2560, 20 query / 5 KV heads of 128,
FFN 6912, vocabulary 128256, 4096 positions) and of the GEMV/GEMM sweep in
bench.py.  Kinds of case:

  ffn      the gated FFN of one block on n rows: one row as in batch-1 decode
           (fused norm + GEMV), more as in prefill and batched decode (row
           quantization + GEMM); n = 1 .. 2048
  linear   one ternary matrix on int8 activations, m = 1 (GEMV) .. 4096 rows
  decode   attention of one decode step for a batch of sequences of different
           lengths, over the f16 cache and its octet copy of V
  layer    the attention half of a block over n prompt tokens behind pos0
           cached ones: norm + quantize, q|k|v GEMM with RoPE and KV append,
           causal attention, sub-norm + quantize, o_proj into the residual
  head     final norm + tied f16 LM head for one row, then the token draw
  request  a whole call on the 2B model: prompt prefill, then greedy decode

Operator cases go through the C ABI (include/oxbitnet_ops.h) on torch tensors:
prepare() resolves each call's arguments as a C program would hold them, run()
makes the calls.  Whole calls go through Model.
"""
import importlib
import math

import torch

pkg = importlib.import_module("0xbitnet_amd")
synth = importlib.import_module("0xbitnet_amd.synth")
native = importlib.import_module("0xbitnet_amd._native")

D, F, H, HKV, HD, V = 2560, 6912, 20, 5, 128, 128256
DQ, DKV = H * HD, HKV * HD
MAX_SEQ = 4096
EPS, SUB_EPS = 1e-5, 1e-5
ROPE_BASE = 500000.0
LAYERS = 30
SCALE = 0.016            # a BitNet per-tensor scale of the size synth.py draws
DEV = "cuda"


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the FFN half of every batch-1 decode step: the smallest call, two launches
        {"name": "ffn_decode", "kind": "ffn", "n": 1},
        # the widest decode matrix of the sweep: one token, weights from HBM
        {"name": "gemv_8192x28672", "kind": "linear", "N": 8192, "K": 28672, "m": 1},
        # one chat at long context
        {"name": "attn_decode_1", "kind": "decode", "batch": 1, "longest": 2304},
        # a serving batch of 32 chats of different lengths
        {"name": "attn_decode_32", "kind": "decode", "batch": 32, "longest": 2304},
        # the FFN of a small serving batch's decode step
        {"name": "ffn_rows_8", "kind": "ffn", "n": 8},
        # a chat turn of ordinary, odd length
        {"name": "attn_layer_101", "kind": "layer", "n": 101, "pos0": 0},
        # the 512-token prefill block
        {"name": "ffn_rows_512", "kind": "ffn", "n": 512},
        # a long document's attention
        {"name": "attn_layer_2048", "kind": "layer", "n": 2048, "pos0": 0},
        # the widest matrix over a large ragged batch of prompt tokens
        {"name": "gemm_8192x28672_4001", "kind": "linear", "N": 8192, "K": 28672, "m": 4001},
        # each generated token's logits and draw, with the reference's default options
        {"name": "head_sample", "kind": "head", "top_k": 50, "temperature": 1.0, "penalty": 1.1},
        # a chat request: short prompt, a reply of 64 tokens
        {"name": "request_chat", "kind": "request", "prompt": 70, "tokens": 64, "kv": "f16"},
        # reading a long document: prompt to first token
        {"name": "request_prompt_2048", "kind": "request", "prompt": 2048, "tokens": 0, "kv": "f16"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "linear", "linear", "decode", "decode", "layer", "layer",
                       "head", "request"])
    if kind == "ffn":
        return {"kind": kind, "n": _log_int(rng, 2, 2048)}   # one row: the listed case
    if kind == "linear":
        N, K = rng.choice([(8192, 28672), (28672, 8192), (13824, 2560), (2560, 6912),
                           (6912, 2560), (3840, 2560), (2560, 2560), (5120, 8192)])
        # the block's small matrices alone only for a batch of rows (one row: ffn)
        return {"kind": kind, "N": N, "K": K, "m": _log_int(rng, 1 if N * K > 4e7 else 64, 2400)}
    if kind == "decode":
        return {"kind": kind, "batch": _log_int(rng, 1, 32), "longest": _log_int(rng, 200, 4000)}
    if kind == "layer":
        n = _log_int(rng, 2, 2048)
        # a later turn of a chat has cached positions before it
        pos0 = rng.choice([0, 0, 0, _log_int(rng, 16, 1500)])
        return {"kind": kind, "n": n, "pos0": pos0}
    if kind == "head":
        return {"kind": kind, "top_k": rng.choice([0, 1, 40, 50, 50, _log_int(rng, 2, 2000)]),
                "temperature": round(rng.uniform(0.5, 1.5), 3),
                "penalty": rng.choice([1.0, 1.1])}
    # the f32 cache is the reference's own type (a parity mode: shorter prompts)
    if rng.random() < 0.2:
        return {"kind": kind, "prompt": _log_int(rng, 4, 256), "tokens": _log_int(rng, 2, 32),
                "kv": "f32"}
    return {"kind": kind, "prompt": _log_int(rng, 4, 1500), "tokens": _log_int(rng, 2, 48),
            "kv": "f16"}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _ternary(g, N, K):
    """Codes w + 1 of a uniform ternary matrix, uint8 [N][K]."""
    return torch.randint(0, 3, (N, K), generator=g, device=DEV, dtype=torch.uint8)


def _pack(codes):
    """I2_S rows [N][K/4] of the codes, then the tiled layout the kernels read."""
    N, K = codes.shape
    c = codes.view(N, K // 128, 4, 32)
    nat = ((c[:, :, 0] << 6) | (c[:, :, 1] << 4) | (c[:, :, 2] << 2) | c[:, :, 3]).contiguous()
    out = torch.empty(N * K // 4, dtype=torch.uint8, device=DEV)
    _call("oxb_repack_i2s_tiled", nat, out, N, K)
    torch.cuda.synchronize()
    return out


def _scales(g, N):
    """One matrix's scale, replicated per row."""
    s = SCALE * (0.8 + 0.4 * torch.rand((), generator=g, device=DEV))
    return s.float().expand(N).contiguous()


def _gamma(g, n):
    return 0.5 + torch.rand(n, generator=g, device=DEV)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _lengths(case, seed):
    """Cached positions of each sequence: the longest, others down to a half of it."""
    g = torch.Generator()
    g.manual_seed(int(seed))
    b, top = case["batch"], case["longest"]
    r = torch.randint((top + 1) // 2, top + 1, (b,), generator=g)
    r[0] = top
    return r.tolist()


def _inputs(case, seed):
    """What the path reads, from the seed alone: natural (unpacked) values."""
    g, kind = _gen(seed), case["kind"]
    if kind == "ffn":
        n = case["n"]
        return {"x": _normal(g, n, D), "wgu": _ternary(g, 2 * F, D), "sgu": _scales(g, 2 * F),
                "wd": _ternary(g, D, F), "sd": _scales(g, D), "norm": _gamma(g, D),
                "sub": _gamma(g, F), "y": _normal(g, n, D)}
    if kind == "linear":
        N, K, m = case["N"], case["K"], case["m"]
        # absmax-quantized normal rows: most values within +-40, one of 127
        x = _normal(g, m, K)
        q = torch.round(x * (127.0 / x.abs().amax(1, keepdim=True))).clamp(-127, 127).to(torch.int8)
        return {"xq": q, "xs": (0.02 + 0.02 * torch.rand(m, generator=g, device=DEV)),
                "w": _ternary(g, N, K), "sw": _scales(g, N)}
    if kind == "decode":
        b, top = case["batch"], case["longest"]
        return {"q": _normal(g, b, DQ), "k": _normal(g, b, HKV, top, HD).half(),
                "v": _normal(g, b, HKV, top, HD).half(), "len": _lengths(case, seed)}
    if kind == "layer":
        n, p = case["n"], case["pos0"]
        return {"x": _normal(g, n, D), "wqkv": _ternary(g, DQ + 2 * DKV, D),
                "sqkv": _scales(g, DQ + 2 * DKV), "wo": _ternary(g, D, DQ), "so": _scales(g, D),
                "norm": _gamma(g, D), "sub": _gamma(g, DQ), "y": _normal(g, n, D),
                "k": 0.6 * _normal(g, HKV, p, HD).half(), "v": 0.6 * _normal(g, HKV, p, HD).half()}
    if kind == "head":
        e = torch.empty(V, D, dtype=torch.float16, device=DEV)
        for r in range(0, V, 16384):
            m = min(16384, V - r)
            e[r:r + m] = (0.02 * _normal(g, m, D)).half()
        return {"x": _normal(g, D), "norm": _gamma(g, D), "e": e,
                "recent": torch.randint(0, V, (64,), generator=g, device=DEV, dtype=torch.int32),
                "u": torch.rand(1, generator=g, device=DEV)}
    return {"ids": torch.randint(0, V, (case["prompt"],), generator=g, device=DEV).cpu().numpy()}


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _bind(name, *args):
    """A C ABI call with its arguments (tensors as pointers, then the current stream)."""
    fn = getattr(native.lib(), name)
    args = (*args, torch.cuda.current_stream().cuda_stream)
    vals = [a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args]
    return name, fn, [t(v) for t, v in zip(fn.argtypes, vals)], args


def _run(call):
    name, fn, vals, _ = call
    if fn(*vals):
        raise native.NativeError(f"{name}: {native.last_error()}")


def _call(name, *args):
    _run(_bind(name, *args))


def _rows_state(n, *Ks):
    """Buffers of quantized rows: token-tiled int8, scales, sums."""
    pad = (n + 63) // 64 * 64
    return (torch.zeros(pad * max(Ks), dtype=torch.int8, device=DEV),
            torch.zeros(pad, device=DEV), torch.zeros(pad, dtype=torch.int32, device=DEV))


def _gemm_ws(*shapes):
    """A split-K workspace for the largest of the (N, K, n) shapes (counters zero)."""
    b = max(native.lib().oxb_gemm_ws_bytes(*s) for s in shapes)
    return torch.zeros(max(b, 16), dtype=torch.uint8, device=DEV), b


def _tiled_rows(q):
    """int8 rows [m][K] in the token-tiled layout of oxb_gemm_i8."""
    m, K = q.shape
    t = torch.zeros((m + 63) // 64 * 64, K, dtype=torch.int8, device=DEV)
    t[:m] = q
    t = t.view(-1, 16, K // 256, 2, 4, 2, 16)       # tile, token, stage, half, plane, c, byte
    return t.permute(0, 2, 4, 3, 5, 1, 6).contiguous()


def _octets(v):
    """V rows [..][S][128] in position octets (round8(S) positions)."""
    *lead, S, hd = v.shape
    S8 = (S + 7) // 8 * 8
    pad = torch.zeros(*lead, S8, hd, dtype=v.dtype, device=DEV)
    pad[..., :S, :] = v
    return pad.view(*lead, S8 // 8, 8, hd).transpose(-1, -2).contiguous()


def prepare(case, seed):
    """{"calls": the C ABI calls of one pass, "out": the buffers they leave}, or a Model."""
    kind, i = case["kind"], _inputs(case, seed)
    if kind == "ffn":
        n = case["n"]
        wgu, wd, h, y = _pack(i["wgu"]), _pack(i["wd"]), torch.empty(n, F, device=DEV), i["y"]
        if n == 1:   # fused norm + quantize + GEMV
            calls = [_bind("oxb_bitlinear_gateup", wgu, i["x"], i["norm"], EPS, i["sgu"], 2 * F, D,
                           h),
                     _bind("oxb_bitlinear_gemv", wd, h, i["sub"], SUB_EPS, i["sd"], D, F, y, 1,
                           None, None, None)]
        else:
            xt, sc, sm = _rows_state(n, D, F)
            ws, wsb = _gemm_ws((2 * F, D, n), (D, F, n))
            calls = [_bind("oxb_quantize_rows_tiled", i["x"], i["norm"], EPS, n, D, xt, sc, sm),
                     _bind("oxb_gemm_i8_ws", wgu, xt, sc, sm, i["sgu"], 2 * F, D, n, h, None, 2,
                           ws, wsb),
                     _bind("oxb_quantize_rows_tiled", h, i["sub"], SUB_EPS, n, F, xt, sc, sm),
                     _bind("oxb_gemm_i8_ws", wd, xt, sc, sm, i["sd"], D, F, n, y, None, 1, ws,
                           wsb)]
        out = {"h": h, "y": y}
    elif kind == "linear":
        N, K, m = case["N"], case["K"], case["m"]
        w, out = _pack(i["w"]), torch.empty(m, N, device=DEV)
        xs, sums = i["xs"], i["xq"].sum(1, dtype=torch.int32)
        if m == 1:
            calls = [_bind("oxb_gemv_i8", w, i["xq"], xs, sums, i["sw"], N, K, out, None)]
        else:
            pad = (m + 63) // 64 * 64 - m
            xs, sums = torch.cat([xs, xs.new_zeros(pad)]), torch.cat([sums, sums.new_zeros(pad)])
            calls = [_bind("oxb_gemm_i8_ws", w, _tiled_rows(i["xq"]), xs, sums, i["sw"], N, K, m,
                           out, None, 0, *_gemm_ws((N, K, m)))]
    elif kind == "decode":
        b, top = case["batch"], case["longest"]
        pos = torch.tensor([n - 1 for n in i["len"]], dtype=torch.int32, device=DEV)
        out = torch.empty(b, DQ, device=DEV)
        calls = [_bind("oxb_attn_decode_batch_v8", i["q"], i["k"], i["v"], _octets(i["v"]), pos, 1,
                       HKV * top * HD, HKV * ((top + 7) // 8 * 8) * HD, b, H, HKV, HD, top,
                       torch.empty(b, H, top, device=DEV), out)]
    elif kind == "layer":
        n, p = case["n"], case["pos0"]
        kc = torch.zeros(HKV * MAX_SEQ * HD + 64 * HD, dtype=torch.float16, device=DEV)
        vc = kc.clone()
        for c, rows in ((kc, i["k"]), (vc, i["v"])):
            c[:HKV * MAX_SEQ * HD].view(HKV, MAX_SEQ, HD)[:, :p] = rows
        rope = torch.empty(MAX_SEQ, HD // 2, 2)
        native.check(native.lib().oxb_rope_table(rope.data_ptr(), MAX_SEQ, HD, ROPE_BASE), "rope")
        q, attn = torch.empty(n, DQ, device=DEV), torch.empty(n, DQ, device=DEV)
        xt, sc, sm = _rows_state(n, D, DQ)
        calls = [_bind("oxb_quantize_rows_tiled", i["x"], i["norm"], EPS, n, D, xt, sc, sm),
                 _bind("oxb_gemm_qkv", _pack(i["wqkv"]), xt, sc, sm, i["sqkv"], DQ, DKV, HD, D, n,
                       p, q, kc, vc, MAX_SEQ, rope.to(DEV)),
                 _bind("oxb_attn_prefill", q, kc, vc, n, p, H, HKV, HD, MAX_SEQ, attn),
                 _bind("oxb_quantize_rows_tiled", attn, i["sub"], SUB_EPS, n, DQ, xt, sc, sm),
                 _bind("oxb_gemm_i8_ws", _pack(i["wo"]), xt, sc, sm, i["so"], D, DQ, n, i["y"],
                       None, 1, *_gemm_ws((D, DQ, n)))]
        out = {"y": i["y"], "k": kc, "v": vc}
    elif kind == "head":
        e = torch.empty(native.lib().oxb_lm_bytes(V, D), dtype=torch.uint8, device=DEV)
        _call("oxb_repack_lm", i["e"], e, V, D)
        b = native.lib().oxb_sample_ws_bytes(V)
        logits, token = torch.empty(V, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
        calls = [_bind("oxb_lm_head_argmax", i["x"], i["norm"], EPS, e, V, D, logits,
                       torch.zeros(8, dtype=torch.int32, device=DEV),
                       torch.zeros(16, dtype=torch.int32, device=DEV), 0),
                 _bind("oxb_sample_device", logits, V, case["temperature"], case["top_k"],
                       case["penalty"], i["recent"], 64, i["u"], token,
                       torch.zeros(b, dtype=torch.uint8, device=DEV), b)]
        out = {"logits": logits, "token": token}
    else:
        path = synth.cached_gguf(synth.BITNET_2B, seed=1234)
        return {"ids": i["ids"], "tokens": case["tokens"],
                "model": pkg.Model(path, max_seq=MAX_SEQ, kv=case["kv"])}
    torch.cuda.synchronize()
    return {"calls": calls, "out": out}


def run(s):
    if "calls" in s:
        for call in s["calls"]:
            _run(call)
        return s["out"]
    m, n = s["model"], s["tokens"]
    m.reset()
    first, logits = m.forward(s["ids"], want_logits=n == 0)
    if n == 0:
        return {"logits": logits, "first": first}
    tokens = m.decode_greedy(n - 1) if n > 1 else []
    last, logits = m.step()
    return {"logits": logits, "tokens": torch.tensor([first, *tokens, last])}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far another implementation may be off
# ---------------------------------------------------------------------------
def _linear_work(N, K, m):
    return N * K / 4 + m * K + 4 * m * N, 2.0 * m * N * K


def _attn_pairs(n, p):
    return n * p + n * (n + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "ffn":
        n = case["n"]
        weights = (2 * F * D + D * F) / 4
        # the rows in, the residual in and out, h out (it is returned)
        return {"bytes": weights + 4 * (2 * F + D + D + F) + 4 * n * (3 * D + F),
                "flops": 2.0 * n * 3 * F * D}
    if kind == "linear":
        b, f = _linear_work(case["N"], case["K"], case["m"])
        return {"bytes": b + 4 * case["N"], "flops": f}
    if kind == "decode":
        # the mean length of a batch is three quarters of the longest
        b, top = case["batch"], case["longest"]
        positions = top + (b - 1) * 0.75 * top
        return {"bytes": positions * HKV * HD * 2 * 2 + 8 * b * DQ,
                "flops": 4.0 * positions * DQ}
    if kind == "layer":
        n, p = case["n"], case["pos0"]
        return {"bytes": ((DQ + 2 * DKV) * D + D * DQ) / 4 + 4 * n * 3 * D +
                2 * 2 * HKV * HD * (p + 2 * n),
                "flops": 2.0 * n * ((DQ + 2 * DKV) * D + D * DQ) + 4.0 * DQ * _attn_pairs(n, p)}
    if kind == "head":
        return {"bytes": 2.0 * V * D + 4 * V, "flops": 2.0 * V * D}
    n, t = case["prompt"], case["tokens"]
    per_layer = (DQ + 2 * DKV) * D + D * DQ + 3 * F * D
    kv = 2 * (4 if case["kv"] == "f32" else 2) * HKV * HD * LAYERS
    pairs = _attn_pairs(n, 0) + _attn_pairs(t, n)
    return {"bytes": (1 + t) * (LAYERS * per_layer / 4 + 2.0 * V * D) + kv * (n + t * (n + t / 2)),
            "flops": 2.0 * (n + t) * LAYERS * per_layer + 4.0 * DQ * LAYERS * pairs +
            2.0 * (1 + t) * V * D}


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 2e-7}        # exact integers, two f32 products: 4e-8 seen
    if kind == "decode":
        return {"rel": 4e-6}        # f32 chains of up to 4000 terms: 1e-6 seen
    if kind == "head":
        return {"rel": 4e-7}        # f32 sums of 2560 products: 1e-7 seen
    if kind in ("ffn", "layer"):
        # f32 sums, then int8 rounding: a last-bit difference moves a value at
        # a rounding boundary by one step of 1/127 of its row's largest (5e-4
        # seen in the FFN, 8e-4 in the attention half)
        return {"rel": 2e-3 if kind == "ffn" else 3e-3, "max": 0.3}
    # the same over 30 layers, where such steps add up
    return {"rel": 0.03, "differ": 0.01}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _quant64(x, gamma, eps):
    """RMSNorm and absmax int8 rows: whole values, scales."""
    x = x.double()
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma.double()
    am = x.abs().amax(-1, keepdim=True)
    return torch.round(x * (127.0 / am)).clamp(-127, 127), am / 127.0


def _bitlinear64(x, gamma, eps, codes, scale):
    q, s = _quant64(x, gamma, eps)
    return (q @ (codes.double() - 1.0).t()) * (scale.double() * s)


def _rope64(x, pos0):
    """Neighbouring pairs (2i, 2i + 1) of each head rotated by pos * base^(-2i/hd)."""
    n = x.shape[0]
    i = torch.arange(HD // 2, dtype=torch.float64, device=DEV)
    pos = torch.arange(pos0, pos0 + n, dtype=torch.float64, device=DEV)
    th = pos[:, None] * ROPE_BASE ** (-2.0 * i / HD)
    co, si = torch.cos(th)[:, None], torch.sin(th)[:, None]
    x = x.reshape(n, -1, HD // 2, 2)
    a, b = x[..., 0], x[..., 1]
    return torch.stack([a * co - b * si, a * si + b * co], -1).view(n, -1, HD)


def exact(case, seed):
    kind = case["kind"]
    if kind == "request":
        return None   # 30 layers of rounding to int8: no one value to compare with
    i = _inputs(case, seed)
    if kind == "ffn":
        g = _bitlinear64(i["x"], i["norm"], EPS, i["wgu"], i["sgu"])
        h = torch.relu(g[:, 0::2]) ** 2 * g[:, 1::2]     # rows: gate0, up0, gate1, ...
        return {"h": h, "y": i["y"].double() + _bitlinear64(h, i["sub"], SUB_EPS, i["wd"], i["sd"])}
    if kind == "linear":
        acc = i["xq"].double() @ (i["w"].double() - 1.0).t()
        return acc * (i["sw"].double() * i["xs"].double()[:, None])
    if kind == "decode":
        out = torch.empty(case["batch"], H, HD, dtype=torch.float64, device=DEV)
        for z, n in enumerate(i["len"]):
            q = i["q"][z].double().view(HKV, H // HKV, HD)
            for h in range(HKV):
                k, v = i["k"][z, h, :n].double(), i["v"][z, h, :n].double()
                p = torch.softmax((q[h] @ k.t()) / math.sqrt(HD), -1)
                out[z, h * (H // HKV):(h + 1) * (H // HKV)] = p @ v
        return out.view(case["batch"], DQ)
    if kind == "layer":
        n, p = case["n"], case["pos0"]
        r = _bitlinear64(i["x"], i["norm"], EPS, i["wqkv"], i["sqkv"])
        q = _rope64(r[:, :DQ], p)
        new_k = _rope64(r[:, DQ:DQ + DKV], p).half()
        new_v = r[:, DQ + DKV:].reshape(n, HKV, HD).half()
        k = torch.cat([i["k"], new_k.transpose(0, 1)], 1)
        v = torch.cat([i["v"], new_v.transpose(0, 1)], 1)
        att = torch.empty(n, H, HD, dtype=torch.float64, device=DEV)
        hide = torch.arange(p + n, device=DEV)[None] > torch.arange(p, p + n, device=DEV)[:, None]
        for h in range(H):
            kh, vh = k[h // (H // HKV)].double(), v[h // (H // HKV)].double()
            sc = (q[:, h] @ kh.t()) / math.sqrt(HD)
            att[:, h] = torch.softmax(sc.masked_fill_(hide, -math.inf), -1) @ vh
        y = i["y"].double() + _bitlinear64(att.view(n, DQ), i["sub"], SUB_EPS, i["wo"], i["so"])
        out = {"y": y}
        for name, rows in (("k", k), ("v", v)):
            c = torch.zeros(HKV * MAX_SEQ * HD + 64 * HD, dtype=torch.float64, device=DEV)
            c[:HKV * MAX_SEQ * HD].view(HKV, MAX_SEQ, HD)[:, :p + n] = rows.double()
            out[name] = c
        return out
    x = i["x"].double()
    x = x / torch.sqrt((x * x).mean() + EPS) * i["norm"].double()
    logits = torch.cat([e.double() @ x for e in i["e"].split(16384)])
    return {"logits": logits, "token": None}
