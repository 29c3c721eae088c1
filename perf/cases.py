"""The measured work of this framework: calls that a program makes through the
public entry points (sera.c_amd/q3q4.py over include/q3_q4_linear.h and
include/sera_q4k.h), at the sizes of one Qwen3-32B layer (hidden 5120, heads
8192 + 2 x 1024, MLP 25600, vocabulary 151936) and at generic odd sizes.

listed() names the cases and draw() gives more of the same ranges:

  linear  one q3_cuda_q4k_linear call: Q4_K (GGUF bytes or 16-row tiles) or
          Q6_K (GGUF bytes or the split layout), 1 to 2048 tokens
  group   one sera_linear_group call: several matrices on one input, with the
          RMSNorm or the SiLU*up producer and the residual add
  layer   the linear steps of the first decoder layer: embedding gather, then
          RMSNorm + q/k/v, o + residual, RMSNorm + gate/up, SiLU*up + down +
          residual (attention itself is outside this framework, its output is
          an input here), called directly or replayed as a HIP graph
  select  the selected-row LM head of speculative decoding: the logits of a few
          candidate tokens of each branch

Weights are N(0, 0.02) quantized to the GGUF block formats, activations N(0, 1)
with 1% of the channels 20 times larger (outlier channels). exact() computes
the same values in 64 bits from the quantized operands: the Q8_1 activations
and the rounded block scales are part of the path's definition, every product
and sum after them is exact here.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "sera.c_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "sera.c_amd"))

Q4K, Q4K_TILED, Q6K, Q6K_SPLIT = 12, 268, 14, 270
DEV = "cuda:0"
EPS = 1e-6
MAX_TOKENS, MAX_FEATURES, MAX_K = 2048, 151936, 25600
ROWS_CHUNK = 8192      # weight rows made, or multiplied in 64 bits, at a time

_context = None        # the process-wide library context and its workspace


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest call of a decode step: one k or v projection, one token
        {"name": "decode_kv_m1", "kind": "linear", "qtype": Q4K, "M": 1, "N": 1024, "K": 5120},
        # one decoder layer of a one-token decode step, replayed as a graph
        {"name": "decode_layer_m1", "kind": "layer", "qtype": Q4K, "M": 1, "hidden": 5120, "q": 8192, "kv": 1024,
         "mlp": 25600, "graph": True},
        # the same layer for a few speculative branches, weights uploaded as tiles
        {"name": "branch_layer_m6_tiled", "kind": "layer", "qtype": Q4K_TILED, "M": 6, "hidden": 5120, "q": 8192,
         "kv": 1024, "mlp": 25600, "graph": False},
        # the LM head of a decode step on Q6_K weights in the split layout
        {"name": "lm_head_q6k_m1", "kind": "linear", "qtype": Q6K_SPLIT, "M": 1, "N": 151936, "K": 5120},
        # down projections stay Q6_K in mixed files: speculative branches on GGUF bytes
        {"name": "down_q6k_m5", "kind": "linear", "qtype": Q6K, "M": 5, "N": 5120, "K": 25600},
        # one candidate row per branch through the LM head
        {"name": "lm_head_m16", "kind": "linear", "qtype": Q4K, "M": 16, "N": 151936, "K": 5120},
        # a small batch of ragged prompts through the MLP's first half
        {"name": "batch_gate_up_m37", "kind": "group", "qtype": Q4K, "M": 37, "Ns": "25600 25600", "K": 5120,
         "op": "rmsnorm", "accumulate": False},
        # a small model's projection at sizes that fill no tile
        {"name": "small_odd_m203", "kind": "linear", "qtype": Q4K, "M": 203, "N": 1333, "K": 1792},
        # prefill of one prompt through one layer
        {"name": "prefill_layer_m512", "kind": "layer", "qtype": Q4K, "M": 512, "hidden": 5120, "q": 8192,
         "kv": 1024, "mlp": 25600, "graph": False},
        # prefill through a Q6_K down projection
        {"name": "prefill_down_q6k_m512", "kind": "linear", "qtype": Q6K, "M": 512, "N": 5120, "K": 25600},
        # a packed batch of branches behind a shared prefix
        {"name": "packed_gate_up_m2048", "kind": "group", "qtype": Q4K, "M": 2048, "Ns": "25600 25600", "K": 5120,
         "op": "rmsnorm", "accumulate": False},
        # speculative decoding scores 128 candidate tokens of 16 branches
        {"name": "candidates_q6k", "kind": "select", "qtype": Q6K, "branches": 16, "per_branch": 128, "N": 151936,
         "K": 5120},
    ]


def _rows(case):
    """The row counts of a group case's matrices."""
    return [int(n) for n in case["Ns"].split()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "group", "layer", "select"])
    qtype = rng.choice([Q4K, Q4K, Q4K_TILED, Q6K, Q6K_SPLIT])
    if kind == "select":
        return {"kind": kind, "qtype": qtype, "branches": _log_int(rng, 1, 32), "per_branch": _log_int(rng, 1, 512),
                "N": 16 * _log_int(rng, 64, 9496), "K": 256 * _log_int(rng, 4, 32)}
    if kind == "layer":
        hidden = 256 * rng.randint(2, 20)
        return {"kind": kind, "qtype": qtype, "M": _log_int(rng, 1, 640), "hidden": hidden,
                "q": 256 * rng.randint(2, 32), "kv": 16 * rng.randint(8, 64), "mlp": 256 * rng.randint(8, 100),
                "graph": rng.random() < 0.5}
    while True:
        M = _log_int(rng, 1, 2048)
        N = _log_int(rng, 256, 28672)
        if qtype == Q4K_TILED:
            N = (N + 15) // 16 * 16
        K = 256 * _log_int(rng, 1, 100)
        if kind == "group":
            Ns = [N] + [max(16, N // rng.choice([1, 1, 4, 8]) // 16 * 16) for _ in range(rng.randint(1, 2))]
            case = {"kind": kind, "qtype": qtype, "M": M, "Ns": " ".join(str(n) for n in Ns), "K": K,
                    "op": rng.choice(["plain", "rmsnorm", "silu"]), "accumulate": rng.random() < 0.3}
        else:
            Ns = [N]
            case = {"kind": kind, "qtype": qtype, "M": M, "N": N, "K": K}
        # no dearer than the largest listed case (Q6_K costs about 1.5 times Q4_K)
        if M * sum(Ns) * K * (1 if qtype in (Q4K, Q4K_TILED) else 2) <= 2048 * 51200 * 5120:
            return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _generator(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * (seed + 1) + salt)
    return g


def _fp16_bytes(x):
    return x.to(torch.float16).contiguous().view(torch.uint8)


def _q4k_rows(w):
    """Q4_K blocks of w [rows, K]: the fields (d, dmin, sc, m, q) and the
    144-byte blocks (fp16 d, dmin; 6-bit scales and mins in 12 bytes; nibbles)."""
    rows, K = w.shape
    b = w.view(rows, K // 256, 8, 32)
    lo = b.amin(-1).clamp(max=0.0)
    step = ((b.amax(-1) - lo) / 15.0).clamp(min=1e-8)
    d = (step.amax(-1) / 63.0).to(torch.float16)
    dmin = ((-lo).amax(-1) / 63.0).clamp(min=6e-8).to(torch.float16)
    sc = (step / d.float()[..., None]).round().clamp(1, 63)
    m = (-lo / dmin.float()[..., None]).round().clamp(0, 63)
    scale = (d.float()[..., None] * sc)[..., None]
    q = ((b + (dmin.float()[..., None] * m)[..., None]) / scale).round().clamp(0, 15).to(torch.uint8)
    out = torch.empty((rows, K // 256, 144), dtype=torch.uint8, device=w.device)
    out[..., 0:2] = _fp16_bytes(d[..., None])
    out[..., 2:4] = _fp16_bytes(dmin[..., None])
    s8, m8 = sc.to(torch.uint8), m.to(torch.uint8)
    out[..., 4:8] = s8[..., :4] | (s8[..., 4:] >> 4 << 6)
    out[..., 8:12] = m8[..., :4] | (m8[..., 4:] >> 4 << 6)
    out[..., 12:16] = (s8[..., 4:] & 15) | (m8[..., 4:] & 15) << 4
    pairs = q.view(rows, K // 256, 4, 2, 32)
    out[..., 16:] = (pairs[..., 0, :] | pairs[..., 1, :] << 4).reshape(rows, K // 256, 128)
    return (d, dmin, sc, m, q), out.view(rows, -1)


def _q6k_rows(w):
    """Q6_K blocks of w [rows, K]: the fields (d, sc, q - 32) and the 210-byte
    blocks (low nibbles, high bits, int8 scales of 16 weights, fp16 d)."""
    rows, K = w.shape
    b = w.view(rows, K // 256, 16, 16)
    step = (b.abs().amax(-1) / 31.0).clamp(min=1e-8)
    d = (step.amax(-1) / 127.0).clamp(min=6e-8).to(torch.float16)
    sc = (step / d.float()[..., None]).round().clamp(1, 127)
    q = (b / (d.float()[..., None] * sc)[..., None]).round().clamp(-32, 31)
    u = (q + 32).to(torch.uint8).view(rows, K // 256, 2, 4, 32)      # half, quarter, position
    out = torch.empty((rows, K // 256, 210), dtype=torch.uint8, device=w.device)
    low, high = u & 15, u >> 4
    out[..., 0:128] = (low[..., 0:2, :] | low[..., 2:4, :] << 4).reshape(rows, K // 256, 128)
    out[..., 128:192] = (high[..., 0, :] | high[..., 1, :] << 2 | high[..., 2, :] << 4 |
                         high[..., 3, :] << 6).reshape(rows, K // 256, 64)
    out[..., 192:208] = sc.to(torch.int8).view(torch.uint8)
    out[..., 208:210] = _fp16_bytes(d[..., None])
    return (d, sc, q), out.view(rows, -1)


def _weight_chunks(qtype, N, K, seed, salt):
    """(first row, fields, GGUF bytes) of N x K weights, ROWS_CHUNK rows at a time."""
    g = _generator(seed, salt)
    for r in range(0, N, ROWS_CHUNK):
        w = torch.randn((min(ROWS_CHUNK, N - r), K), generator=g, device=DEV) * 0.02
        yield (r,) + (_q4k_rows(w) if qtype in (Q4K, Q4K_TILED) else _q6k_rows(w))


def _weights(qtype, N, K, seed, salt):
    """The matrix on the device in the layout of qtype, as the loader leaves it."""
    import q3q4
    gguf = torch.empty(q3q4.weight_bytes(qtype, N, K), dtype=torch.uint8, device=DEV)
    row = gguf.numel() // N
    for r, _, b in _weight_chunks(qtype, N, K, seed, salt):
        gguf[r * row:(r + b.shape[0]) * row] = b.reshape(-1)
    if qtype in (Q4K, Q6K):
        return gguf
    dst = torch.empty_like(gguf)
    q3q4.weight_to_device_layout(qtype, N, K, gguf, dst)
    torch.cuda.current_stream().synchronize()
    return dst


def _activations(M, K, seed, salt):
    g = _generator(seed, salt)
    x = torch.randn((M, K), generator=g, device=DEV)
    loud = torch.randperm(K, generator=g, device=DEV)[:max(1, K // 100)]
    x[:, loud] *= 20.0
    return x


def _gamma(K, seed, salt):
    return 1.0 + 0.1 * torch.randn(K, generator=_generator(seed, salt), device=DEV)


def _ids(count, N, seed, salt):
    return torch.randint(0, N, (count,), generator=_generator(seed, salt), device=DEV, dtype=torch.int32)


VOCAB = 4096           # rows of the layer case's embedding table


def _layer_matrices(case):
    h, q, kv, mlp = case["hidden"], case["q"], case["kv"], case["mlp"]
    return {"q": (q, h), "k": (kv, h), "v": (kv, h), "o": (h, q), "gate": (mlp, h), "up": (mlp, h), "down": (h, mlp)}


def _linear_context():
    """The library's process-wide context, made once as a program does."""
    global _context
    if _context is None:
        import q3q4
        _context = q3q4.Linear(device=0, max_tokens=MAX_TOKENS, max_features=MAX_FEATURES, max_k=MAX_K)
    return _context


def prepare(case, seed):
    import q3q4
    _linear_context()
    kind, qt = case["kind"], case["qtype"]
    st = {"kind": kind, "case": case}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        st["geometry"] = q3q4.bind_geometry(qt, K, N)
        st["weight"] = _weights(qt, N, K, seed, 1)
        st["x"] = _activations(M, K, seed, 2)
        st["y"] = torch.empty((M, N), device=DEV)
    elif kind == "group":
        M, K = case["M"], case["K"]
        st["geometries"] = [q3q4.bind_geometry(qt, K, n) for n in _rows(case)]
        st["weights"] = [_weights(qt, n, K, seed, 10 + i) for i, n in enumerate(_rows(case))]
        st["x"] = _activations(M, K, seed, 2)
        st["x2"] = _activations(M, K, seed, 3) if case["op"] == "silu" else None
        st["gamma"] = _gamma(K, seed, 4) if case["op"] == "rmsnorm" else None
        st["flags"] = {"plain": 0, "rmsnorm": q3q4.LIN_RMSNORM, "silu": q3q4.LIN_SILU_MUL}[case["op"]]
        st["y"] = [torch.empty((M, n), device=DEV) for n in _rows(case)]
        st["residual"] = None
        if case["accumulate"]:
            st["flags"] |= q3q4.LIN_ACCUMULATE
            st["residual"] = [_activations(M, n, seed, 20 + i) for i, n in enumerate(_rows(case))]
    elif kind == "layer":
        M, h = case["M"], case["hidden"]
        mats = _layer_matrices(case)
        st["g"] = {n: q3q4.bind_geometry(qt, K, N) for n, (N, K) in mats.items()}
        st["w"] = {n: _weights(qt, N, K, seed, 30 + i) for i, (n, (N, K)) in enumerate(mats.items())}
        st["y"] = {n: torch.empty((M, mats[n][0]), device=DEV) for n in ("q", "k", "v", "gate", "up")}
        st["table"] = _weights(qt, VOCAB, h, seed, 5)
        st["ids"] = _ids(M, VOCAB, seed, 6)
        st["hidden"] = torch.empty((M, h), device=DEV)
        st["attn"] = _activations(M, case["q"], seed, 7)
        st["gamma1"], st["gamma2"] = _gamma(h, seed, 8), _gamma(h, seed, 9)
        if case["graph"]:
            _layer_step(st)                      # a program warms a step up before it captures it
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                _layer_step(st)
            st["graph"] = graph
    else:
        n = case["branches"] * case["per_branch"]
        st["weight"] = _weights(qt, case["N"], case["K"], seed, 1)
        st["hidden"] = _activations(case["branches"], case["K"], seed, 2)
        st["ids"] = _ids(n, case["N"], seed, 3)
        st["y"] = torch.empty((case["branches"], case["per_branch"]), device=DEV)
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _layer_step(st):
    import q3q4
    g, w, y, h = st["g"], st["w"], st["y"], st["hidden"]
    qt = st["case"]["qtype"]
    q3q4.embedding(qt, st["table"], VOCAB, st["case"]["hidden"], st["ids"], h)
    q3q4.linear_group([g["q"], g["k"], g["v"]], [w["q"], w["k"], w["v"]], [y["q"], y["k"], y["v"]], h,
                      gamma=st["gamma1"], eps=EPS, flags=q3q4.LIN_RMSNORM)
    q3q4.linear_group([g["o"]], [w["o"]], [h], st["attn"], flags=q3q4.LIN_ACCUMULATE)
    q3q4.linear_group([g["gate"], g["up"]], [w["gate"], w["up"]], [y["gate"], y["up"]], h, gamma=st["gamma2"],
                      eps=EPS, flags=q3q4.LIN_RMSNORM)
    q3q4.linear_group([g["down"]], [w["down"]], [h], y["gate"], x2=y["up"],
                      flags=q3q4.LIN_SILU_MUL | q3q4.LIN_ACCUMULATE)
    return [y["q"], y["k"], y["v"], y["gate"], y["up"], h]


def run(st):
    import ctypes

    import q3q4
    kind = st["kind"]
    if kind == "linear":
        # the C boundary as a forward pass calls it, without the optional timing statistics
        err = ctypes.create_string_buffer(256)
        x = st["x"]
        if not q3q4.load().q3_cuda_q4k_linear(ctypes.byref(st["geometry"]), st["weight"].data_ptr(), x.data_ptr(),
                                              x.shape[0], st["y"].data_ptr(),
                                              torch.cuda.current_stream().cuda_stream, None, err, 256):
            raise RuntimeError(err.value.decode())
        return st["y"]
    if kind == "group":
        if st["residual"] is not None:
            for y, r in zip(st["y"], st["residual"]):
                y.copy_(r)
        q3q4.linear_group(st["geometries"], st["weights"], st["y"], st["x"], x2=st["x2"], gamma=st["gamma"], eps=EPS,
                          flags=st["flags"])
        return st["y"]
    if kind == "layer":
        if "graph" in st:
            st["graph"].replay()
            y = st["y"]
            return [y["q"], y["k"], y["v"], y["gate"], y["up"], st["hidden"]]
        return _layer_step(st)
    c = st["case"]
    q3q4.candidate_logits(c["qtype"], st["weight"], c["N"], c["K"], st["hidden"], st["ids"], c["per_branch"], st["y"])
    return st["y"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _weight_bytes(qtype, N, K):
    return N * (K // 256) * (144 if qtype in (Q4K, Q4K_TILED) else 210)


def work(case):
    kind, qt = case["kind"], case["qtype"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _weight_bytes(qt, N, K) + 4 * M * (K + N), "flops": 2 * M * N * K}
    if kind == "group":
        M, K, N = case["M"], case["K"], sum(_rows(case))
        b = sum(_weight_bytes(qt, n, K) for n in _rows(case)) + 4 * M * (K * (2 if case["op"] == "silu" else 1) + N)
        return {"bytes": b + (4 * M * N if case["accumulate"] else 0), "flops": 2 * M * N * K}
    if kind == "layer":
        M, h = case["M"], case["hidden"]
        mats = _layer_matrices(case)
        b = sum(_weight_bytes(qt, N, K) for N, K in mats.values()) + _weight_bytes(qt, min(M, VOCAB), h)
        acts = case["q"] + 2 * case["kv"] + 2 * case["mlp"] + h + case["q"]     # the outputs, attention's input
        return {"bytes": b + 4 * M * acts, "flops": 2 * M * sum(N * K for N, K in mats.values())}
    n = case["branches"] * case["per_branch"]
    return {"bytes": _weight_bytes(qt, n, case["K"]) + 4 * (case["branches"] * case["K"] + 2 * n),
            "flops": 2 * n * case["K"]}


def tolerance(case):
    # Plain products: fp32 sums in another order, up to 5e-7 measured. With a
    # producer the last place of the normalized row can move single
    # activations to the next of 127 quantization steps (4e-5 measured), and a
    # layer quantizes again what its first half computed (2e-3 measured).
    if case["kind"] == "layer":
        return {"rel": 8e-3, "max": 8e-2}
    if case["kind"] == "group" and case["op"] != "plain":
        return {"rel": 2e-4, "max": 2e-2}
    return {"rel": 2e-6, "max": 4e-5}


# ---------------------------------------------------------------------------
# the same values in 64 bits
# ---------------------------------------------------------------------------

def _round_half_away(x):
    x = x.double()      # |x| + 0.5 is exact there
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _q8(x, rule):
    """Q8_1 quants and scales of x [M, K] fp32 as 64-bit numbers: rule "row"
    (up to 8 tokens), "ds4" (Q4_K above) or "d4" (Q6_K above); the third
    result is the block sum the Q4_K min term takes."""
    x = x.cpu()
    b = x.view(x.shape[0], -1, 32)
    amax = b.abs().amax(-1)
    if rule == "row":
        d = amax / torch.full_like(amax, 127.0)
        q = torch.where(amax[..., None] == 0, 0.0, _round_half_away(b / d[..., None]))
        d = d.to(torch.float16)
        s = d.double() * q.sum(-1)
    else:
        inv = torch.full_like(amax, 127.0) / amax      # a scalar numerator would become a reciprocal
        q = torch.where(amax[..., None] == 0, 0.0, _round_half_away(b * inv[..., None]))
        d = torch.where(amax == 0, torch.zeros_like(amax), 1.0 / inv)
        v = b.view(b.shape[0], b.shape[1], 8, 4)
        p = ((v[..., 0] + v[..., 1]) + v[..., 2]) + v[..., 3]
        for o in (4, 2):
            p = p[..., :o] + p[..., o:2 * o]
        s = (p[..., 0] + p[..., 1]).to(torch.float16).double()
        if rule == "ds4":
            d = d.to(torch.float16)
    return q.to(DEV), d.double().to(DEV), s.to(DEV)


def _matmul(qtype, x, N, K, seed, salt):
    """x [M, K] fp32 times the matrix of (seed, salt), from quantized operands, in 64 bits."""
    M = x.shape[0]
    q4 = qtype in (Q4K, Q4K_TILED)
    rule = "row" if M <= 8 else ("ds4" if q4 else "d4")
    q, d, s = _q8(x, rule)
    xq = (q * d[..., None]).view(M, K)
    out = torch.empty((M, N), dtype=torch.float64, device=DEV)
    for r, f, _ in _weight_chunks(qtype, N, K, seed, salt):
        rows = f[0].shape[0]
        if q4:
            dd, dmin, sc, m, qw = f
            scale = dd.double()[..., None] * sc.double()
            mins = dmin.double()[..., None] * m.double()
            if rule == "ds4":        # the tile path stores both products as fp16
                scale = scale.float().to(torch.float16).double()
                mins = mins.float().to(torch.float16).double()
            y = xq @ (qw.double() * scale[..., None]).view(rows, K).T
            y -= s @ mins.view(rows, K // 32).T
        else:
            dd, sc, qw = f
            y = xq @ (qw.double() * (dd.double()[..., None] * sc.double())[..., None]).view(rows, K).T
        out[:, r:r + rows] = y
    return out


def _rmsnorm(x, gamma):
    x = x.double()
    inv = (1.0 / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)).float()
    return x.float() * inv * gamma


def _silu_mul(g, u):
    return (g.double() / (1.0 + torch.exp(-g.double())) * u.double()).float()


def _gathered_rows(qtype, N, K, ids, seed, salt):
    out = torch.empty((ids.numel(), K), dtype=torch.float64, device=DEV)
    for r, f, _ in _weight_chunks(qtype, N, K, seed, salt):
        hit = (ids >= r) & (ids < r + f[0].shape[0])
        i = (ids[hit] - r).long()
        if qtype in (Q4K, Q4K_TILED):
            dd, dmin, sc, m, qw = (t[i].double() for t in f)
            w = qw * (dd[..., None] * sc)[..., None] - (dmin[..., None] * m)[..., None]
        else:
            dd, sc, qw = (t[i].double() for t in f)
            w = qw * (dd[..., None] * sc)[..., None]
        out[hit] = w.reshape(-1, K)
    return out


def exact(case, seed):
    kind, qt = case["kind"], case["qtype"]
    if kind == "linear":
        return _matmul(qt, _activations(case["M"], case["K"], seed, 2), case["N"], case["K"], seed, 1)
    if kind == "group":
        M, K = case["M"], case["K"]
        x = _activations(M, K, seed, 2)
        if case["op"] == "rmsnorm":
            x = _rmsnorm(x, _gamma(K, seed, 4))
        elif case["op"] == "silu":
            x = _silu_mul(x, _activations(M, K, seed, 3))
        y = [_matmul(qt, x, n, K, seed, 10 + i) for i, n in enumerate(_rows(case))]
        if case["accumulate"]:
            y = [v + _activations(M, n, seed, 20 + i).double() for i, (v, n) in enumerate(zip(y, _rows(case)))]
        return y
    if kind == "layer":
        M, h = case["M"], case["hidden"]
        salts = {n: 30 + i for i, n in enumerate(_layer_matrices(case))}

        def mm(x, n):
            N, K = _layer_matrices(case)[n]
            return _matmul(qt, x, N, K, seed, salts[n])

        res = _gathered_rows(qt, VOCAB, h, _ids(M, VOCAB, seed, 6), seed, 5)
        x = _rmsnorm(res.float(), _gamma(h, seed, 8))
        q, k, v = mm(x, "q"), mm(x, "k"), mm(x, "v")
        res = res + mm(_activations(M, case["q"], seed, 7), "o")
        x = _rmsnorm(res.float(), _gamma(h, seed, 9))
        gate, up = mm(x, "gate"), mm(x, "up")
        res = res + mm(_silu_mul(gate.float(), up.float()), "down")
        return [q, k, v, gate, up, res]
    w = _gathered_rows(qt, case["N"], case["K"], _ids(case["branches"] * case["per_branch"], case["N"], seed, 3),
                       seed, 1)
    x = _activations(case["branches"], case["K"], seed, 2).double()
    return (w.view(case["branches"], case["per_branch"], -1) * x[:, None, :]).sum(-1)
