"""The work a user of the engine has it do, as measurable cases.

Every case is one pass through the public entry points of air_amd.capi over
inputs made from a seed.  Four kinds of pass:

  linears    the projections of a stack of Qwen2 layers (fused q|k|v with its
             bias, o, fused gate|up, down), one down projection per layer, or
             one single matrix: what a host that runs its own step calls;
  step       a whole greedy decode step, one row per sequence: embedding rows,
             the layers over the paged KV pool, the final norm, lm_head, argmax
             (logits and tokens come back), launched as one HIP graph per batch
             width as HipStepEngine launches it;
  prefill    the layers of a prompt step on the prefill tactic;
  attention  the online-softmax attention of one layer over the paged pool.

Shapes are those of the repository's configurations (Qwen2-0.5B and Qwen2-7B
widths) and generic ones; weights are w ~ N(0, 0.02) quantized to the GGUF
encodings, activations and cached keys and values ~ N(0, 1), as there.
"""
import ctypes
import math

import numpy as np
import torch

from air_amd import capi, quant

TYPES = {"q8_0": capi.TYPE_Q8_0, "q4_0": capi.TYPE_Q4_0, "q4_k": capi.TYPE_Q4_K, "q6_k": capi.TYPE_Q6_K,
         "f16": capi.TYPE_F16, "bf16": capi.TYPE_BF16}
BLOCKS = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210), "f16": (1, 2), "bf16": (1, 2)}
EPS = 1e-6
ROPE_BASE = 1e6
PAGE_TOKENS = 16
SIGMA = 0.02


def listed():
    return [
        # The smallest call: one FFN up-projection of a 0.5B model for one row.
        # Latency of a single launch.
        dict(name="single_q8_0_m1", kind="linears", which="single", format="q8_0", hidden=896, kv=128, ffn=4864,
             layers=1, m=1),
        # A token of a small model served alone: hundreds of short launches.
        dict(name="step_05b_q8_0_m1", kind="step", format="q8_0", hidden=896, heads=14, kv_heads=2, ffn=4864,
             vocab=151936, layers=24, m=1, context_min=200, context_max=200),
        # A token of a 7B model served alone (interactive use): weight streaming.
        dict(name="step_7b_q8_0_m1", kind="step", format="q8_0", hidden=3584, heads=28, kv_heads=4, ffn=18944,
             vocab=152064, layers=4, m=1, context_min=600, context_max=600),
        # A batched decode step of a server: 32 sequences of ragged lengths.
        dict(name="step_7b_q8_0_m32", kind="step", format="q8_0", hidden=3584, heads=28, kv_heads=4, ffn=18944,
             vocab=152064, layers=4, m=32, context_min=512, context_max=640),
        # Small decode batches of the 7B projections.
        dict(name="block_7b_q8_0_m8", kind="linears", which="block", format="q8_0", hidden=3584, kv=512, ffn=18944,
             layers=3, m=8),
        # 4-bit files at the batch widths they are served at.
        dict(name="block_7b_q4_k_m16", kind="linears", which="block", format="q4_k", hidden=3584, kv=512, ffn=18944,
             layers=4, m=16),
        dict(name="block_7b_q4_0_m64", kind="linears", which="block", format="q4_0", hidden=3584, kv=512, ffn=18944,
             layers=4, m=64),
        # The Q6_K share of a mixed 4-bit file (ffn_down), an odd batch.
        dict(name="down_7b_q6_k_m13", kind="linears", which="down", format="q6_k", hidden=3584, kv=512, ffn=18944,
             layers=6, m=13),
        # A small model kept in half precision, a few rows.
        dict(name="block_05b_f16_m5", kind="linears", which="block", format="f16", hidden=896, kv=128, ffn=4864,
             layers=12, m=5),
        # A full prompt quantum of a 7B model.
        dict(name="prefill_7b_q8_0_m512", kind="prefill", format="q8_0", hidden=3584, heads=28, kv_heads=4, ffn=18944,
             layers=2, m=512, sequences=1, start=0),
        # The projections of a ragged prompt remainder, 4-bit file.
        dict(name="block_7b_q4_k_m301", kind="linears", which="block", format="q4_k", hidden=3584, kv=512, ffn=18944,
             layers=2, m=301),
        # Decode attention over long, ragged contexts.
        dict(name="attention_7b_long", kind="attention", heads=28, kv_heads=4, head_dim=128, m=24, run=1,
             context_min=700, context_max=4000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges the listed ones stand for."""
    kind = rng.choice(["linears", "linears", "linears", "step", "prefill", "attention"])
    if kind == "linears":
        fmt = rng.choice(["q8_0", "q8_0", "q4_0", "q4_k", "q6_k", "f16", "bf16"])
        step = 256 if BLOCKS[fmt][0] == 256 else 32
        hidden = step * max(1, _log_int(rng, 768, 4608) // step)
        ffn = step * max(1, _log_int(rng, 2048, 19456) // step)
        kv = 32 * rng.randint(2, 32)
        m = _log_int(rng, 1, 64) if rng.random() < 0.75 else _log_int(rng, 65, 512)
        case = dict(kind=kind, which=rng.choice(["block", "block", "down", "single"]), format=fmt, hidden=hidden,
                    kv=kv, ffn=ffn, m=m, layers=1)
        per_layer = work(case)
        limit = min(0.6e9 / per_layer["bytes"], 0.2e12 / per_layer["flops"])
        case["layers"] = max(1, min(16, int(limit)))
        return case
    if kind == "step":
        head_dim = rng.choice([64, 128])
        kv_heads = rng.choice([2, 4, 8] if head_dim == 64 else [2, 4])
        heads = kv_heads * rng.randint(2, 7)
        fmt = rng.choice(["q8_0", "q8_0", "q4_0", "q4_k"])
        if fmt == "q4_k" and heads * head_dim % 256:
            fmt = "q4_0"
        hidden = heads * head_dim
        ffn = 256 * max(4, int(hidden * rng.uniform(2.5, 5.5)) // 256)
        lo = _log_int(rng, 20, 2000)
        return dict(kind=kind, format=fmt, hidden=hidden, heads=heads, kv_heads=kv_heads, ffn=ffn,
                    vocab=16 * _log_int(rng, 2000, 9500) + rng.randint(0, 15), layers=rng.randint(1, 3),
                    m=_log_int(rng, 1, 48), context_min=lo, context_max=lo + rng.randint(0, lo))
    if kind == "prefill":
        kv_heads = rng.choice([2, 4])
        head_dim = rng.choice([64, 128])
        heads = kv_heads * rng.randint(2, 7)
        hidden = heads * head_dim
        fmt = rng.choice(["q8_0", "q4_0", "q4_k"]) if hidden % 256 == 0 else rng.choice(["q8_0", "q4_0"])
        return dict(kind=kind, format=fmt, hidden=hidden, heads=heads, kv_heads=kv_heads,
                    ffn=256 * max(4, int(hidden * rng.uniform(2.5, 5.2)) // 256), layers=rng.randint(1, 2),
                    m=_log_int(rng, 66, 512), sequences=rng.randint(1, 4), start=rng.choice([0, 0, 256, 1000]))
    head_dim = rng.choice([64, 128])
    kv_heads = rng.choice([2, 4, 8])
    lo = _log_int(rng, 30, 2000)
    prompt = rng.random() < 0.4
    return dict(kind=kind, heads=kv_heads * rng.randint(1, 8), kv_heads=kv_heads, head_dim=head_dim,
                m=_log_int(rng, 1, 4) if prompt else _log_int(rng, 1, 32),
                run=_log_int(rng, 16, 128) if prompt else 1,
                context_min=lo, context_max=lo + rng.randint(0, lo))


# ---- shapes ----------------------------------------------------------------

def _shapes(case):
    """(name, k, n, bias) of one layer's matrices."""
    h, f = case["hidden"], case["ffn"]
    if case.get("which") == "single":
        return [("single", h, f, False)]
    if case.get("which") == "down":
        return [("down", f, h, False)]
    kv = case["kv"] if "kv" in case else case["kv_heads"] * (h // case["heads"])
    return [("qkv", h, h + 2 * kv, True), ("o", h, h, False), ("gate_up", h, 2 * f, False), ("down", f, h, False)]


def _weight_bytes(fmt, k, n):
    elements, size = BLOCKS[fmt]
    return n * (k // elements) * size


def _contexts(case):
    """Tokens of each sequence once the step has run, spread over the case's range."""
    m, lo, hi = case["m"], case["context_min"], case["context_max"]
    return [lo + (hi - lo) * ((i * 7) % m) // max(m - 1, 1) for i in range(m)]


def _prompt_runs(case):
    """Rows of each sequence of a prompt step: uneven shares of m rows."""
    m, s = case["m"], case["sequences"]
    weights = [2 + (i % 3) for i in range(s)]
    runs = [m * w // sum(weights) for w in weights]
    runs[0] += m - sum(runs)
    return runs


def work(case):
    m = case["m"]
    if case["kind"] == "linears":
        nbytes = flops = 0
        for _, k, n, bias in _shapes(case):
            nbytes += _weight_bytes(case["format"], k, n) + 4 * m * (k + n) + (4 * n if bias else 0)
            flops += 2 * m * k * n
        return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}
    if case["kind"] == "attention":
        heads, kv_heads, hd, run = case["heads"], case["kv_heads"], case["head_dim"], case["run"]
        nbytes = flops = 0
        for tokens in _contexts(case):
            nbytes += 8 * kv_heads * hd * (tokens + run - 1) + 8 * heads * hd * run
            flops += 4 * heads * hd * sum(tokens + r for r in range(run))
        return {"bytes": nbytes, "flops": flops}
    h = case["hidden"]
    hd = h // case["heads"]
    kv = case["kv_heads"] * hd
    nbytes = flops = 0
    for _, k, n, bias in _shapes(case):
        nbytes += _weight_bytes(case["format"], k, n) + (4 * n if bias else 0)
        flops += 2 * m * k * n
    nbytes += 8 * h                                              # the two norms' weights
    if case["kind"] == "step":
        tokens = _contexts(case)
        nbytes += 8 * kv * sum(tokens)                           # keys and values, the row's own written
        flops += 4 * h * sum(tokens)
        nbytes, flops = nbytes * case["layers"], flops * case["layers"]
        nbytes += _weight_bytes(case["format"], h, case["vocab"]) + m * _weight_bytes(case["format"], h, 1)
        nbytes += 4 * m * case["vocab"] + 4 * h + 4 * m
        flops += 2 * m * h * case["vocab"]
        return {"bytes": nbytes, "flops": flops}
    for run in _prompt_runs(case):
        nbytes += 8 * kv * (case["start"] + run)
        flops += 4 * h * sum(case["start"] + r + 1 for r in range(run))
    return {"bytes": nbytes * case["layers"] + 8 * m * h, "flops": flops * case["layers"]}


# ---- inputs ----------------------------------------------------------------

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=gen.device, dtype=torch.float32)


def _canonical(fmt, k, n, seed):
    """Canonical GGUF rows (uint8 [n, row bytes]) of w ~ N(0, 0.02)."""
    dev = _device()
    if TYPES[fmt] in quant.BLOCK:
        return quant.synthetic_weights_device(TYPES[fmt], k, n, seed, dev, SIGMA)
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    if fmt in ("f16", "bf16"):
        dtype = torch.float16 if fmt == "f16" else torch.bfloat16
        return (_normal(gen, n, k) * SIGMA).to(dtype).view(torch.uint8)
    # Q6_K: uniform 6-bit codes under int8 sub-block scales, d so that the
    # weights' deviation is SIGMA (codes 18.5, scales ~80 in the mean square).
    blocks = torch.randint(0, 256, (n, k // 256, 210), generator=gen, device=dev, dtype=torch.uint8)
    scales = torch.randint(40, 112, (n, k // 256, 16), generator=gen, device=dev, dtype=torch.int16)
    signs = torch.randint(0, 2, (n, k // 256, 16), generator=gen, device=dev, dtype=torch.int16) * 2 - 1
    blocks[..., 192:208] = (scales * signs).to(torch.int8).view(torch.uint8)
    d = (SIGMA / (18.5 * 80.0)) * (0.75 + 0.5 * torch.rand((n, k // 256, 1), generator=gen, device=dev))
    blocks[..., 208:210] = d.to(torch.float16).view(torch.uint8)
    return blocks.reshape(n, -1)


def _decoded(fmt, k, n, canon):
    """float64 weights [n, k] of canonical rows, in plain torch."""
    if fmt == "f16":
        return canon.view(torch.float16).double()
    if fmt == "bf16":
        return canon.view(torch.bfloat16).double()
    elements, size = BLOCKS[fmt]
    b = canon.reshape(n, k // elements, size)

    def half(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()

    if fmt == "q8_0":
        return (half(0) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(n, k)
    if fmt == "q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], dim=2).double() - 8.0
        return (half(0) * q).reshape(n, k)
    if fmt == "q4_k":
        s = b[..., 4:16]
        sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], dim=2).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], dim=2).double()
        g = b[..., 16:].reshape(n, k // 256, 4, 1, 32)
        q = torch.cat([g & 15, g >> 4], dim=3).reshape(n, k // 256, 8, 32).double()
        return ((half(0) * sc)[..., None] * q - (half(2) * mn)[..., None]).reshape(n, k)
    ql = b[..., 0:128].reshape(n, k // 256, 2, 2, 32)
    qh = b[..., 128:192].reshape(n, k // 256, 2, 1, 32)
    low = torch.cat([ql & 15, ql >> 4], dim=3)                                  # four runs of 32 per half
    high = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], dim=3)
    q = (low | (high << 4)).double().reshape(n, k // 256, 16, 16) - 32.0
    sc = half(208) * b[..., 192:208].contiguous().view(torch.int8).double()
    return (sc[..., None] * q).reshape(n, k)


def _matrix_seed(seed, layer, index):
    return seed * 1000003 + layer * 101 + index * 13 + 7


def _rope_table(positions, dims):
    i = np.arange(dims // 2)
    angle = np.arange(positions)[:, None] * (1.0 / ROPE_BASE ** (2.0 * i / dims))[None, :]
    return torch.from_numpy(np.stack([np.cos(angle), np.sin(angle)], axis=-1))   # float64 [positions, half, 2]


def _inputs(case, seed):
    """Every input tensor of a case but the weights, from the seed alone."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 7919 + 17)
    m = case["m"]
    if case["kind"] == "linears":
        ins = {}
        for name, k, n, bias in _shapes(case):
            ins[name] = [(_normal(gen, m, k), _normal(gen, n) * 0.1 if bias else None)
                         for _ in range(case["layers"])]
        return ins
    if case["kind"] == "attention":
        heads, kv_heads, hd, layers = case["heads"], case["kv_heads"], case["head_dim"], 1
        runs = [case["run"]] * m
        tokens = [t + case["run"] - 1 for t in _contexts(case)]
    else:
        heads, kv_heads, layers = case["heads"], case["kv_heads"], case["layers"]
        hd = case["hidden"] // heads
        runs = [1] * m if case["kind"] == "step" else _prompt_runs(case)
        tokens = _contexts(case) if case["kind"] == "step" else [case["start"] + r for r in runs]
    rng = np.random.default_rng(seed)
    pages = [(t + PAGE_TOKENS - 1) // PAGE_TOKENS for t in tokens]
    order = rng.permutation(sum(pages))
    tables, positions, used = [], [], 0
    for run, t, p in zip(runs, tokens, pages):
        row = list(order[used:used + p]) + [-1] * (max(pages) - p)
        used += p
        tables += [row] * run
        positions += range(t - run, t)
    kv = kv_heads * hd
    ins = {"runs": runs, "tokens": tokens, "heads": heads, "kv_heads": kv_heads, "head_dim": hd, "rows": sum(runs),
           "tables": torch.tensor(np.array(tables), dtype=torch.int32, device=dev),
           "positions": torch.tensor(positions, dtype=torch.int32, device=dev),
           "pool": _normal(gen, sum(pages), layers, 2, PAGE_TOKENS, kv)}
    if case["kind"] == "attention":
        ins["qkv"] = _normal(gen, sum(runs), heads * hd + 2 * kv)
        return ins
    h = case["hidden"]
    ins["attn_norm"] = 1.0 + 0.1 * _normal(gen, layers, h)
    ins["ffn_norm"] = 1.0 + 0.1 * _normal(gen, layers, h)
    ins["out_norm"] = 1.0 + 0.1 * _normal(gen, h)
    ins["bias"] = 0.1 * _normal(gen, layers, h + 2 * kv)
    ins["rope"] = _rope_table(max(tokens), hd)
    if case["kind"] == "step":
        ins["ids"] = torch.randint(0, case["vocab"], (m,), generator=gen, device=dev, dtype=torch.int32)
    else:
        ins["hidden"] = _normal(gen, m, h)
    return ins


# ---- state and passes --------------------------------------------------------

class State:
    """What a program keeps between calls: a context, resident matrices, the
    device buffers and, for decode steps, the captured graph."""

    def __init__(self, case):
        self.case = case
        self.ctx = capi.Context(torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream)
        self.lib = capi.lib()
        self.mats = []
        self.head = None
        self.graph = None

    def matrix(self, k, n, seed):
        fmt = self.case["format"]
        canon = _canonical(fmt, k, n, seed)
        return capi.Matrix(self.ctx, TYPES[fmt], k, n, canon, canon.numel(), on_device=True)

    def layers(self, seed):
        self.mats = [{name: self.matrix(k, n, _matrix_seed(seed, layer, i))
                      for i, (name, k, n, _) in enumerate(_shapes(self.case))} for layer in range(self.case["layers"])]

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.graph = None
            for mat in [x for layer in self.mats for x in layer.values()] + ([self.head] if self.head else []):
                mat.release()
            self.ctx.close()
        except Exception:
            pass


def _buffer(*shape):
    return torch.empty(shape, device=_device(), dtype=torch.float32)


def prepare(case, seed):
    s = State(case)
    s.ins = ins = _inputs(case, seed)
    m = case["m"]
    if case["kind"] == "linears":
        s.layers(seed)
        s.out = [{name: _buffer(m, n) for name, _, n, _ in _shapes(case)} for _ in range(case["layers"])]
        s.ctx.reserve(max(k for _, k, _, _ in _shapes(case)), m)
        return s
    heads, kv_heads, hd, rows = ins["heads"], ins["kv_heads"], ins["head_dim"], ins["rows"]
    kv = kv_heads * hd
    pool = ins["pool"]
    s.kv = capi.KvLayout(pool.data_ptr(), PAGE_TOKENS, kv, pool.shape[1], ins["tables"].shape[1], pool.shape[0])
    tiles = capi.attention_tiles(ins["runs"], heads, kv_heads)
    s.tile_count = len(tiles)
    s.tiles = torch.tensor(np.array(tiles, dtype=np.uint32).view(np.int32), device=_device())
    s.max_tokens = max(ins["tokens"])
    s.att = _buffer(rows, heads * hd)
    if case["kind"] == "attention":
        return s
    h, f = case["hidden"], case["ffn"]
    s.layers(seed)
    s.rope = ins["rope"].to(device=_device(), dtype=torch.float32)
    s.hidden, s.normed, s.qkv = _buffer(m, h), _buffer(m, h), _buffer(m, h + 2 * kv)
    s.act, s.proj = _buffer(m, f), _buffer(m, h)
    if case["kind"] == "prefill":
        s.gate_up = _buffer(m, 2 * f)
        s.ctx.reserve(f, m)
        return s
    s.head = s.matrix(h, case["vocab"], _matrix_seed(seed, case["layers"], 0))
    s.logits = _buffer(m, case["vocab"])
    s.tokens = torch.empty(m, dtype=torch.int32, device=_device())
    s.ctx.reserve(f, m)
    # One eager step (every buffer grown), then the step recorded as a graph.
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        s.ctx.set_stream(side.cuda_stream)
        _decode_step(s)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        _decode_step(s)
    s.graph = graph
    s.ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    return s


def _attention(s, layer):
    ins = s.ins
    heads, kv_heads, hd = ins["heads"], ins["kv_heads"], ins["head_dim"]
    qkv = ins["qkv"] if "qkv" in ins else s.qkv
    capi.check(s.lib.air_hip_attention_online(
        s.ctx.handle, ctypes.byref(s.kv), qkv.data_ptr(), qkv.shape[1], ins["rows"], ins["positions"].data_ptr(),
        ins["tables"].data_ptr(), layer, heads, kv_heads, hd, s.tiles.data_ptr(), s.tile_count, s.max_tokens,
        s.att.data_ptr()))


def _decode_step(s):
    """Embedding to argmax for m rows, one per sequence, with the element-wise
    work fused into the linears (one row: the M = 1 entry point)."""
    case, ins, lib, ctx = s.case, s.ins, s.lib, s.ctx.handle
    m, h, layers = case["m"], case["hidden"], case["layers"]
    heads, kv_heads, hd = ins["heads"], ins["kv_heads"], ins["head_dim"]
    x, normed, qkv, act = s.hidden.data_ptr(), s.normed.data_ptr(), s.qkv.data_ptr(), s.act.data_ptr()
    att, kv = s.att.data_ptr(), ctypes.byref(s.kv)
    positions, tables = ins["positions"].data_ptr(), ins["tables"].data_ptr()
    rope = (heads, kv_heads, hd, hd, s.rope.data_ptr(), s.rope.shape[0])
    check = capi.check
    check(lib.air_hip_matrix_rows(ctx, s.head.handle, ins["ids"].data_ptr(), m, x))
    attn = [ins["attn_norm"][i].data_ptr() for i in range(layers)] + [ins["out_norm"].data_ptr()]
    ffn = [ins["ffn_norm"][i].data_ptr() for i in range(layers)]
    if m == 1:
        for i in range(layers):
            mats = s.mats[i]
            check(lib.air_hip_decode_linear_fused(ctx, mats["qkv"].handle, x, qkv, ins["bias"][i].data_ptr(), attn[i],
                                                  EPS, capi.EPILOGUE_STORE))
            check(lib.air_hip_rope_kv_append(ctx, kv, qkv, s.qkv.shape[1], m, positions, tables, i, *rope))
            _attention(s, i)
            check(lib.air_hip_decode_linear_fused(ctx, mats["o"].handle, att, x, None, None, 0.0,
                                                  capi.EPILOGUE_RESIDUAL))
            check(lib.air_hip_rms_norm(ctx, x, ffn[i], normed, m, h, EPS))
            check(lib.air_hip_decode_linear_fused(ctx, mats["gate_up"].handle, normed, act, None, None, 0.0,
                                                  capi.EPILOGUE_SWIGLU))
            check(lib.air_hip_decode_linear_fused(ctx, mats["down"].handle, act, x, None, None, 0.0,
                                                  capi.EPILOGUE_RESIDUAL))
        check(lib.air_hip_rms_norm(ctx, x, attn[layers], normed, m, h, EPS))
    else:
        check(lib.air_hip_rms_norm(ctx, x, attn[0], normed, m, h, EPS))
        for i in range(layers):
            mats = s.mats[i]
            check(lib.air_hip_linear_rope_kv(ctx, mats["qkv"].handle, normed, m, qkv, ins["bias"][i].data_ptr(), kv,
                                             positions, tables, i, *rope, capi.LINEAR_DECODE))
            _attention(s, i)
            check(lib.air_hip_linear_epilogue(ctx, mats["o"].handle, att, m, x, None, capi.EPILOGUE_RESIDUAL_LOAD,
                                              ffn[i], normed, EPS, capi.LINEAR_DECODE))
            check(lib.air_hip_linear_epilogue(ctx, mats["gate_up"].handle, normed, m, act, None, capi.EPILOGUE_SWIGLU,
                                              None, None, 0.0, capi.LINEAR_DECODE))
            check(lib.air_hip_linear_epilogue(ctx, mats["down"].handle, act, m, x, None, capi.EPILOGUE_RESIDUAL_LOAD,
                                              attn[i + 1], normed, EPS, capi.LINEAR_DECODE))
    s.head.linear(s.normed, s.logits, m, tactic=capi.LINEAR_DECODE)
    check(lib.air_hip_argmax(ctx, s.logits.data_ptr(), m, case["vocab"], s.tokens.data_ptr()))


def _prefill(s):
    """The layers of a prompt step over m rows, from the hidden rows given."""
    case, ins, lib, ctx = s.case, s.ins, s.lib, s.ctx.handle
    m, h, layers, f = case["m"], case["hidden"], case["layers"], case["ffn"]
    heads, kv_heads, hd = ins["heads"], ins["kv_heads"], ins["head_dim"]
    s.hidden.copy_(ins["hidden"])
    x, normed, qkv, act = s.hidden.data_ptr(), s.normed.data_ptr(), s.qkv.data_ptr(), s.act.data_ptr()
    kv, proj, att = ctypes.byref(s.kv), s.proj.data_ptr(), s.att.data_ptr()
    tactic = capi.LINEAR_PREFILL
    check = capi.check
    attn = [ins["attn_norm"][i].data_ptr() for i in range(layers)] + [ins["out_norm"].data_ptr()]
    check(lib.air_hip_rms_norm_prefill(ctx, x, None, attn[0], normed, m, h, EPS))
    for i in range(layers):
        mats = s.mats[i]
        check(lib.air_hip_linear(ctx, mats["qkv"].handle, normed, qkv, ins["bias"][i].data_ptr(), m, tactic))
        check(lib.air_hip_rope_kv_append(ctx, kv, qkv, s.qkv.shape[1], m, ins["positions"].data_ptr(),
                                         ins["tables"].data_ptr(), i, heads, kv_heads, hd, hd, s.rope.data_ptr(),
                                         s.rope.shape[0]))
        _attention(s, i)
        check(lib.air_hip_linear_epilogue(ctx, mats["o"].handle, att, m, x, None, capi.EPILOGUE_RESIDUAL_PREFILL,
                                          ins["ffn_norm"][i].data_ptr(), normed, EPS, tactic))
        check(lib.air_hip_linear(ctx, mats["gate_up"].handle, normed, s.gate_up.data_ptr(), None, m, tactic))
        check(lib.air_hip_silu_mul_prefill(ctx, s.gate_up.data_ptr(), act, m, f))
        check(lib.air_hip_linear(ctx, mats["down"].handle, act, proj, None, m, tactic))
        norm = lib.air_hip_rms_norm_prefill if i + 1 < layers else lib.air_hip_add_rms_norm
        check(norm(ctx, x, proj, attn[i + 1], normed, m, h, EPS))


def run(state):
    s = state
    case = s.case
    if case["kind"] == "linears":
        for layer, mats in enumerate(s.mats):
            for name, mat in mats.items():
                x, bias = s.ins[name][layer]
                mat.linear(x, s.out[layer][name], case["m"], bias=bias)
        return [y for layer in s.out for y in layer.values()]
    if case["kind"] == "attention":
        _attention(s, 0)
        return s.att
    if case["kind"] == "prefill":
        _prefill(s)
        return [s.hidden, s.normed, s.ins["pool"]]
    s.graph.replay()
    return [s.logits, s.tokens, s.hidden, s.ins["pool"]]


# ---- what the results should be ----------------------------------------------

def tolerance(case):
    if case["kind"] == "attention":
        return {"rel": 2e-6}                     # f32 products, sums and exponentials
    if case["kind"] == "prefill":
        return {"rel": 3e-3}                     # f16 operands, one rounding each, over the layers
    if case["kind"] == "step":
        # f32 sums of exact codes and activations held to ~21 bits, through
        # every layer; a token may differ only where two logits nearly tie.
        return {"rel": 8e-6, "differ": 0.05}
    if case["m"] > capi.MAX_DECODE_ROWS:
        return {"rel": 3e-3}                     # f16 operands
    return {"rel": 2e-6}                         # f32 sums


def _exact_attention(ins, q, pool, layer):
    """float64 attention of every row over its sequence's cached tokens."""
    heads, kv_heads, hd = ins["heads"], ins["kv_heads"], ins["head_dim"]
    group = heads // kv_heads
    out = torch.empty((ins["rows"], heads * hd), dtype=torch.float64, device=q.device)
    row = 0
    for run, tokens in zip(ins["runs"], ins["tokens"]):
        pages = ins["tables"][row, :(tokens + PAGE_TOKENS - 1) // PAGE_TOKENS].long()
        kv = pool[pages, layer].double().transpose(0, 1).reshape(2, -1, kv_heads, hd)[:, :tokens]
        last = ins["positions"][row:row + run].long()
        for g in range(kv_heads):
            k, v = kv[0, :, g], kv[1, :, g]
            qg = q[row:row + run].double().reshape(run, heads, hd)[:, g * group:(g + 1) * group].reshape(-1, hd)
            s = (qg @ k.T.contiguous() / math.sqrt(hd)).reshape(run, group, tokens)
            s = s.masked_fill(torch.arange(tokens, device=q.device) > last[:, None, None], -math.inf)
            o = torch.softmax(s, dim=2).reshape(-1, tokens) @ v
            out[row:row + run, g * group * hd:(g + 1) * group * hd] = o.reshape(run, group * hd)
        row += run
    return out


def _exact_layers(case, seed, ins, x):
    """float64 layers of a step or prompt; the pool gets the rows' k and v."""
    h, f = case["hidden"], case["ffn"]
    heads, kv_heads, hd = ins["heads"], ins["kv_heads"], ins["head_dim"]
    pool = ins["pool"].double()
    table = ins["rope"].to(x.device)[ins["positions"].long()]
    cos, sin = table[:, None, :, 0], table[:, None, :, 1]
    pages = torch.gather(ins["tables"].long(), 1, (ins["positions"].long() // PAGE_TOKENS)[:, None])[:, 0]
    slots = ins["positions"].long() % PAGE_TOKENS

    def norm(v, w):
        return v / torch.sqrt((v * v).mean(dim=1, keepdim=True) + EPS) * w.double()

    def rotate(v):
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=2)

    for layer in range(case["layers"]):
        w = {}
        for i, (name, k, n, _) in enumerate(_shapes(case)):
            w[name] = (k, n, _matrix_seed(seed, layer, i))

        def product(v, name):
            k, n, matrix_seed = w[name]
            return v @ _decoded(case["format"], k, n, _canonical(case["format"], k, n, matrix_seed)).T

        qkv = product(norm(x, ins["attn_norm"][layer]), "qkv") + ins["bias"][layer].double()
        q = rotate(qkv[:, :h].reshape(-1, heads, hd)).reshape(-1, h)
        kv = kv_heads * hd
        pool[pages, layer, 0, slots] = rotate(qkv[:, h:h + kv].reshape(-1, kv_heads, hd)).reshape(-1, kv)
        pool[pages, layer, 1, slots] = qkv[:, h + kv:]
        x = x + product(_exact_attention(ins, q, pool, layer), "o")
        gu = product(norm(x, ins["ffn_norm"][layer]), "gate_up")
        x = x + product(gu[:, :f] / (1.0 + torch.exp(-gu[:, :f])) * gu[:, f:], "down")
    return x, norm(x, ins["out_norm"]), pool


def exact(case, seed):
    ins = _inputs(case, seed)
    if case["kind"] == "linears":
        out = []
        for layer in range(case["layers"]):
            for i, (name, k, n, _) in enumerate(_shapes(case)):
                x, bias = ins[name][layer]
                w = _decoded(case["format"], k, n, _canonical(case["format"], k, n, _matrix_seed(seed, layer, i)))
                y = x.double() @ w.T
                out.append(y if bias is None else y + bias.double())
        return out
    if case["kind"] == "attention":
        width = ins["heads"] * ins["head_dim"]
        return _exact_attention(ins, ins["qkv"][:, :width], ins["pool"], 0)
    if case["kind"] == "prefill":
        x, normed, pool = _exact_layers(case, seed, ins, ins["hidden"].double())
        return [x, normed, pool]
    head = _decoded(case["format"], case["hidden"], case["vocab"],
                    _canonical(case["format"], case["hidden"], case["vocab"], _matrix_seed(seed, case["layers"], 0)))
    x, normed, pool = _exact_layers(case, seed, ins, head[ins["ids"].long()].clone())
    logits = normed @ head.T
    return [logits, logits.argmax(dim=1).to(torch.int32), x, pool]
