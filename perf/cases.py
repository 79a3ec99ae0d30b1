"""The calls whose speed matters to a user of this library, and how to make, run and check one.

The work of an inference program on the paged-attention path: decode steps of a batch
(`engine.decode_step`, one launch a layer, captured in a HIP graph as a serving loop does),
prompts (`LucAttn.paged_prefill`, called layer by layer), the one-row products of a decode
step (`rmsnorm_gemv`, `gemv`, `gate_up_silu`, captured too), top-k / top-p sampling of a
logits row, and the Qwen2 model loop as a whole (a prompt, and a captured decode step).

`listed()` are the sizes that stand for each kind of use; `draw` spreads others over the
same ranges.  A state holds what a program has in hand before the call.  The attention
entry points rope q and k in place in the qkv rows; a program's projection writes those
rows anew for every call, and one copy of the projected rows for all layers stands for it.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if "lucciola_rs_amd" not in sys.modules:
    _spec = importlib.util.spec_from_file_location(
        "lucciola_rs_amd", os.path.join(_ROOT, "lucciola-rs_amd", "__init__.py"),
        submodule_search_locations=[os.path.join(_ROOT, "lucciola-rs_amd")])
    _pkg = importlib.util.module_from_spec(_spec)
    sys.modules["lucciola_rs_amd"] = _pkg
    _spec.loader.exec_module(_pkg)
from lucciola_rs_amd import engine, library, model  # noqa: E402

PAGE = 16
ROPE_BASE = 1e6
EPS = 1e-6


def listed():
    return [
        # one sequence, short context: the latency of a chat's next token, every layer of it
        {"name": "decode_single", "kind": "decode", "batch": 1, "hq": 14, "hkv": 2, "d": 64,
         "dtype": "f16", "lo": 512, "hi": 512, "layers": 24},
        # a serving batch of mixed short contexts (the benchmark's workload)
        {"name": "decode_b32_mixed", "kind": "decode", "batch": 32, "hq": 14, "hkv": 2, "d": 64,
         "dtype": "f16", "lo": 128, "hi": 4096, "layers": 24},
        # few sequences of long documents
        {"name": "decode_b8_32k", "kind": "decode", "batch": 8, "hq": 12, "hkv": 2, "d": 128,
         "dtype": "bf16", "lo": 30000, "hi": 32768, "layers": 4},
        # the largest: a full batch of long mixed contexts
        {"name": "decode_b64_long", "kind": "decode", "batch": 64, "hq": 28, "hkv": 4, "d": 128,
         "dtype": "bf16", "lo": 1024, "hi": 16384, "layers": 2},
        # a batch of short ragged prompts (chat turns), from an empty cache
        {"name": "prefill_short", "kind": "prefill", "batch": 6, "rows_lo": 17, "rows_hi": 300,
         "start_lo": 0, "start_hi": 0, "hq": 14, "hkv": 2, "d": 64, "dtype": "f16", "layers": 4},
        # one prompt of an odd length (a single user's document)
        {"name": "prefill_1x1531", "kind": "prefill", "batch": 1, "rows_lo": 1531, "rows_hi": 1531,
         "start_lo": 0, "start_hi": 0, "hq": 28, "hkv": 4, "d": 128, "dtype": "bf16", "layers": 2},
        # a chunk of a long prompt (or a new turn of a long chat) after its cached prefix
        {"name": "prefill_chunk", "kind": "prefill", "batch": 1, "rows_lo": 512, "rows_hi": 512,
         "start_lo": 8000, "start_hi": 8000, "hq": 12, "hkv": 2, "d": 128, "dtype": "f16",
         "layers": 2},
        # four long prompts at once (the benchmark's prefill workload)
        {"name": "prefill_4x2048", "kind": "prefill", "batch": 4, "rows_lo": 2048, "rows_hi": 2048,
         "start_lo": 0, "start_hi": 0, "hq": 14, "hkv": 2, "d": 64, "dtype": "bf16", "layers": 2},
        # the one-row products of a decode step, four layers of a mid-sized model
        {"name": "one_row_products", "kind": "rows", "hidden": 2048, "qkv": 3072, "inter": 8192,
         "layers": 4},
        # a token drawn from a logits row
        {"name": "sample_top_p", "kind": "sample", "vocab": 151936, "top_k": 1024, "top_p": 0.9},
        # the whole model on a prompt, to the logits that the first token is drawn from
        {"name": "model_prompt", "kind": "model_prompt", "rows": 700},
        # the whole model's next token, one captured graph, and its logits
        {"name": "model_decode", "kind": "model_decode", "pos": 700},
    ]


# head layouts in use: (query heads, kv heads, head_dim)
_HEADS = [(14, 2, 64), (14, 2, 64), (12, 2, 128), (28, 4, 128), (28, 4, 128), (16, 8, 64),
          (32, 8, 128), (4, 2, 64), (8, 8, 128), (16, 2, 128)]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 6 + ["rows"] * 2 + ["sample", "model_prompt",
                                                                     "model_decode"])
    if kind == "decode":
        hq, hkv, d = rng.choice(_HEADS)
        per_token = hkv * d * 4
        hi = _log_int(rng, 40, 32768)
        # at most 0.6 GB of K and V a layer
        batch = _log_int(rng, 1, max(1, min(64, int(0.6e9 / (per_token * hi)))))
        lo = rng.choice([hi, max(1, hi // 2), max(1, hi // 16)])
        return {"kind": kind, "batch": batch, "hq": hq, "hkv": hkv, "d": d,
                "dtype": rng.choice(["f16", "bf16", "bf16"]), "lo": lo, "hi": hi,
                "layers": rng.choice([2, 3])}
    if kind == "prefill":
        hq, hkv, d = rng.choice(_HEADS)
        batch = rng.choice([1, 1, 1, 2, 3, 5, 8])
        start_hi = rng.choice([0, 0, _log_int(rng, 16, 12000)])
        rows_hi = _log_int(rng, 2, 3000)
        # at most 12 GFLOP a layer
        while 4.0 * d * hq * batch * rows_hi * (start_hi + rows_hi / 2 + 1) > 12e9:
            rows_hi = max(2, rows_hi * 3 // 4)
        rows_lo = rng.choice([rows_hi, max(1, rows_hi // 8)])
        return {"kind": kind, "batch": batch, "rows_lo": rows_lo, "rows_hi": rows_hi,
                "start_lo": start_hi // 3, "start_hi": start_hi, "hq": hq, "hkv": hkv, "d": d,
                "dtype": rng.choice(["f16", "bf16", "bf16"]), "layers": 2}
    if kind == "rows":
        hidden = 128 * _log_int(rng, 2, 24)
        return {"kind": kind, "hidden": hidden, "qkv": hidden + 128 * _log_int(rng, 2, 16),
                "inter": 8 * _log_int(rng, 64, 1024), "layers": rng.choice([2, 3, 4])}
    if kind == "sample":
        return {"kind": kind, "vocab": _log_int(rng, 32000, 262144),
                "top_k": rng.choice([32, 64, 256, 1024]), "top_p": rng.choice([0.8, 0.9, 0.95])}
    if kind == "model_prompt":
        return {"kind": kind, "rows": _log_int(rng, 5, 700)}
    return {"kind": kind, "pos": _log_int(rng, 3, 2000)}


# ---- inputs, from the seed alone ----------------------------------------------------------

_DT = {"f16": torch.float16, "bf16": torch.bfloat16}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(gen, shape, std, dtype, mean=0.0):
    return torch.randn(shape, generator=gen, device="cuda").mul_(std).add_(mean).to(dtype)


def _pool(gen, shape, std, dtype):
    """A K or V pool as earlier steps would have filled it, drawn in pieces."""
    pool = torch.empty(shape, dtype=dtype, device="cuda")
    flat = pool.view(-1)
    step = 1 << 26
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=gen, device="cuda").mul_(std)
    return pool


def _tables(seed, ctx, spare=1.1):
    """Pages dealt from a shuffled pool with some to spare: (tables [B, pages], pool pages)."""
    rng = np.random.default_rng(int(seed))
    pages = [-(-int(c) // PAGE) for c in ctx]
    total = int(sum(pages) * spare) + 2
    perm = rng.permutation(total).astype(np.int32)
    tables = np.zeros((len(ctx), max(pages)), np.int32)
    off = 0
    for b, n in enumerate(pages):
        tables[b, :n] = perm[off:off + n]
        off += n
    return tables, total


# q and k of this size give scores of standard deviation about 2, as trained heads do
_QK_STD, _V_STD, _BIAS_STD = 1.4, 1.0, 0.1


def _attention_inputs(case, seed, ctx, rows):
    """Projected qkv rows of every layer, biases, pools and tables."""
    gen = _gen(seed)
    dt = _DT[case["dtype"]]
    hq, hkv, d, layers = case["hq"], case["hkv"], case["d"], case["layers"]
    tables, pages = _tables(seed, ctx)
    shape = (pages, layers, hkv, PAGE, d)
    row = (hq + 2 * hkv) * d
    proj = _normal(gen, (layers, rows, row), _QK_STD, dt)
    bias = _normal(gen, (layers, row), _BIAS_STD, dt)
    return {"proj": proj, "bias": bias, "tables": torch.from_numpy(tables).cuda(),
            "k": _pool(gen, shape, _QK_STD, dt), "v": _pool(gen, shape, _V_STD, dt)}


# The lengths belong to the case (so that outputs of any seed have one shape): mixed, not
# sorted, the longest among them.
def _decode_lengths(case):
    ctx = np.random.default_rng(case["batch"]).integers(case["lo"], case["hi"] + 1, case["batch"])
    ctx[case["batch"] // 2] = case["hi"]
    return ctx


def _prefill_lengths(case):
    rng = np.random.default_rng(case["batch"])
    rows = rng.integers(case["rows_lo"], case["rows_hi"] + 1, case["batch"])
    rows[case["batch"] // 2] = case["rows_hi"]
    starts = rng.integers(case["start_lo"], case["start_hi"] + 1, case["batch"])
    return rows, starts


_MODEL = model.QWEN25_05B
_MODEL_CTX = 2048  # positions that the model's cache and captured step are sized for


def _model_weights(seed):
    """Random weights in the model's fused layout, as GPU tensors; the projections back into
    the hidden state are smaller by sqrt(2 layers), so that no layer drowns the others."""
    c, gen, dt = _MODEL, _gen(seed), torch.bfloat16
    H, I, V = c.hidden_size, c.intermediate_size, c.vocab_size
    back = 0.02 / math.sqrt(2 * c.num_hidden_layers)
    w = {"embed_tokens": _normal(gen, (V, H), 0.1, dt),
         "final_norm": _normal(gen, (H,), 0.02, dt, 1.0), "layers": []}
    for _ in range(c.num_hidden_layers):
        w["layers"].append({
            "input_layernorm": _normal(gen, (H,), 0.02, dt, 1.0),
            "qkv_proj": _normal(gen, (c.qkv_dim, H), 0.02, dt),
            "qkv_bias": _normal(gen, (c.qkv_dim,), 0.02, dt),
            "o_proj": _normal(gen, (H, H), back, dt),
            "post_attention_layernorm": _normal(gen, (H,), 0.02, dt, 1.0),
            "gate_up_proj": _normal(gen, (2 * I, H), 0.02, dt),
            "down_proj": _normal(gen, (H, I), back, dt)})
    return w


def _bits(w):
    if isinstance(w, dict):
        return {k: _bits(v) for k, v in w.items()}
    if isinstance(w, list):
        return [_bits(v) for v in w]
    return w.view(torch.int16).cpu().numpy().view(np.uint16)


def _model_ids(seed, n):
    return [int(i) for i in np.random.default_rng(int(seed) + 1).integers(0, _MODEL.vocab_size, n)]


def _model_cache(seed):
    """K and V of earlier positions, as page-ordered pools of the model's cache."""
    c, gen = _MODEL, _gen(int(seed) + 2)
    shape = (_MODEL_CTX // PAGE, c.num_hidden_layers, c.num_key_value_heads, PAGE, c.head_dim)
    return _normal(gen, shape, 1.0, torch.bfloat16), _normal(gen, shape, 0.5, torch.bfloat16)


def _rows_inputs(case, seed):
    gen, dt = _gen(seed), torch.bfloat16
    H, Q, I = case["hidden"], case["qkv"], case["inter"]
    return _normal(gen, (H,), 1.0, dt), [
        {"n1": _normal(gen, (H,), 0.02, dt, 1.0), "qkv": _normal(gen, (Q, H), 0.03, dt),
         "o": _normal(gen, (H, H), 0.03, dt), "n2": _normal(gen, (H,), 0.02, dt, 1.0),
         "gu": _normal(gen, (2 * I, H), 0.03, dt), "down": _normal(gen, (H, I), 0.03, dt)}
        for _ in range(case["layers"])]


# ---- the calls ----------------------------------------------------------------------------

def prepare(case, seed):
    lib = library.default(torch.cuda.current_device())
    kind = case["kind"]
    if kind == "decode":
        return _prepare_decode(lib, case, seed)
    if kind == "prefill":
        rows, starts = _prefill_lengths(case)
        cu = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
        s = _attention_inputs(case, seed, rows + starts, int(cu[-1]))
        max_ctx = int((rows + starts).max())
        out = torch.empty((case["layers"], int(cu[-1]), case["hq"] * case["d"]),
                          dtype=s["proj"].dtype, device="cuda")
        s.update(case=case, lib=lib, rows=int(cu[-1]), max_ctx=max_ctx, out=out,
                 qkv=torch.empty_like(s["proj"]), cu=torch.from_numpy(cu).cuda(),
                 start=torch.from_numpy(starts.astype(np.int32)).cuda(),
                 rope=engine.RopeCache(max_ctx, case["d"], ROPE_BASE, lib=lib))
        return s
    if kind == "rows":
        return _prepare_rows(lib, case, seed)
    if kind == "sample":
        gen = _gen(seed)
        return {"case": case, "lib": lib,
                "logits": _normal(gen, (case["vocab"],), 2.0, torch.bfloat16),
                "buffer": torch.zeros(2 * 1024, dtype=torch.int32, device="cuda"),
                "rand": float(np.random.default_rng(int(seed)).uniform(0.05, 0.95)),
                "idx": torch.zeros(1, dtype=torch.int32, device="cuda")}
    m = model.Qwen2Model(_MODEL, _bits(_model_weights(seed)), max_positions=_MODEL_CTX, lib=lib)
    if kind == "model_prompt":
        return {"case": case, "model": m, "ids": _model_ids(seed, case["rows"])}
    k, v = _model_cache(seed)
    m.kv.k_pool.copy_(k)
    m.kv.v_pool.copy_(v)
    return {"case": case, "model": m, "token": _model_ids(seed, 1)[0],
            "graph": m.capture_decode(_MODEL_CTX)}


def _prepare_decode(lib, case, seed):
    ctx = _decode_lengths(case)
    s = _attention_inputs(case, seed, ctx, case["batch"])
    hq, hkv, d, layers, batch = case["hq"], case["hkv"], case["d"], case["layers"], case["batch"]
    qd, kd = hq * d, hkv * d
    max_ctx = int(ctx.max())
    rope = engine.RopeCache(max_ctx, d, ROPE_BASE, lib=lib)
    positions = torch.from_numpy((ctx - 1).astype(np.int32)).cuda()
    out = torch.empty((layers, batch, qd), dtype=s["proj"].dtype, device="cuda")
    qkv = torch.empty_like(s["proj"])
    ws = lib.workspace(batch, hq, hkv, d, max_ctx)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        torch.mul(s["proj"], 1.0, out=qkv)  # the projections' output
        for li in range(layers):
            b = s["bias"][li]
            engine.decode_step(qkv[li], b[:qd], b[qd:qd + kd], b[qd + kd:], rope, s["k"], s["v"],
                               s["tables"], positions, max_ctx, li, layers, hq, hkv, d, out[li],
                               workspace=ws, lib=lib)
    s.update(case=case, lib=lib, rope=rope, positions=positions, out=out, qkv=qkv, ws=ws,
             graph=graph)
    return s


def _prepare_rows(lib, case, seed):
    x, weights = _rows_inputs(case, seed)
    H, Q, I = case["hidden"], case["qkv"], case["inter"]
    bf = dict(dtype=torch.bfloat16, device="cuda")
    outs = [{"qkv": torch.empty(Q, **bf), "h1": torch.empty(H, **bf), "act": torch.empty(I, **bf),
             "h2": torch.empty(H, **bf)} for _ in weights]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        h = x
        for w, o in zip(weights, outs):
            lib.rmsnorm_gemv(o["qkv"], h, w["n1"], EPS, w["qkv"])
            lib.gemv(o["h1"], o["qkv"][:H], w["o"], residual=h)
            lib.gate_up_silu(o["act"], o["h1"], w["n2"], EPS, w["gu"])
            lib.gemv(o["h2"], o["act"], w["down"], residual=o["h1"])
            h = o["h2"]
    return {"case": case, "x": x, "weights": weights, "outs": outs, "graph": graph}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        state["graph"].replay()
        return {"out": state["out"], "qkv": state["qkv"], "k": state["k"], "v": state["v"]}
    if kind == "prefill":
        hq, hkv, d, layers = case["hq"], case["hkv"], case["d"], case["layers"]
        qd, kd = hq * d, hkv * d
        state["qkv"].copy_(state["proj"])  # the projections' output
        scale, rope, lib = engine.sm_scale(d), state["rope"], state["lib"]
        for li in range(layers):
            b = state["bias"][li]
            lib.paged_prefill(state["qkv"][li], b[:qd], b[qd:qd + kd], b[qd + kd:], rope.cos,
                              rope.sin, state["k"], state["v"], state["tables"], state["cu"],
                              state["start"], state["rows"], state["max_ctx"], li, layers, hq, hkv,
                              d, scale, state["out"][li])
        return {"out": state["out"], "qkv": state["qkv"], "k": state["k"], "v": state["v"]}
    if kind == "rows":
        state["graph"].replay()
        return state["outs"]
    if kind == "sample":
        state["lib"].sort_and_sample(state["logits"], case["top_p"], case["top_k"], state["rand"],
                                     state["buffer"], state["idx"])
        return {"token": state["idx"], "candidates": state["buffer"][:2 * case["top_k"]]}
    m = state["model"]
    if kind == "model_prompt":
        m.forward(state["ids"], 0)
    else:
        m.idx.fill_(state["token"])
        m.pos.fill_(case["pos"])
        state["graph"].replay()
    return {"logits": m.logits(), "hidden": m.hidden, "k": m.kv.k_pool, "v": m.kv.v_pool}


# ---- what a pass cannot do without --------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "decode":
        tokens = float(_decode_lengths(case).sum())
        hq, hkv, d, B = case["hq"], case["hkv"], case["d"], case["batch"]
        bytes_ = tokens * hkv * d * 4 + tokens / 4 + B * (3 * hq + 6 * hkv) * d * 2
        return {"bytes": case["layers"] * bytes_, "flops": case["layers"] * 4.0 * tokens * hq * d}
    if kind == "prefill":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        n, s = (x.astype(np.float64) for x in _prefill_lengths(case))
        keys = float((n * s + n * (n + 1) / 2).sum())
        # qkv read, roped q and k and the output written, new K and V cached, the prefix read
        bytes_ = float(n.sum() * (3 * hq + 5 * hkv) * d * 2 + s.sum() * hkv * d * 4)
        return {"bytes": case["layers"] * bytes_, "flops": case["layers"] * 4.0 * d * hq * keys}
    if kind == "rows":
        H, Q, I, L = case["hidden"], case["qkv"], case["inter"], case["layers"]
        params = L * (Q * H + H * H + 3 * I * H)
        return {"bytes": 2.0 * params, "flops": 2.0 * params}
    if kind == "sample":
        return {"bytes": case["vocab"] * 2.0 + case["top_k"] * 8, "flops": 0}
    c = _MODEL
    layer = c.hidden_size * (c.qkv_dim + c.hidden_size + 3 * c.intermediate_size)
    layers = c.num_hidden_layers * layer
    head = c.vocab_size * c.hidden_size
    kv = c.num_hidden_layers * c.num_key_value_heads * c.head_dim * 4
    if kind == "model_prompt":
        n = case["rows"]
        att = c.num_hidden_layers * 4.0 * c.hidden_size * n * (n + 1) / 2
        return {"bytes": 2.0 * (layers + head) + n * kv, "flops": 2.0 * (layers * n + head) + att}
    # the step's own lm_head (for its token), and that of the logits handed out
    return {"bytes": 2.0 * (layers + 2 * head) + case["pos"] * kv,
            "flops": 2.0 * (layers + 2 * head)}


# 2-norm errors measured on an MI355X.  Attention is 5e-4 (fp16) and 5e-3 (bf16) from the
# 64-bit result, the roundings of q, k, the weights and the output; two orders of its sums
# differ by that at most.  Chains of one-row products with their sums in another order are up
# to 1.2e-2 apart after four layers of bf16 rounding, the whole model 1.5e-2 after 24.
def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind in ("decode", "prefill"):
        return {"rel": 2e-3} if case["dtype"] == "f16" else {"rel": 1e-2}
    return {"rel": 3e-2}


# ---- the same in 64 bits ------------------------------------------------------------------

def _rope64(n, d):
    """cos and sin of the engine's table: its angles are 32-bit (rope.rs)."""
    i = np.arange(d // 2, dtype=np.float32) * np.float32(2) / np.float32(d)
    freq = np.power(np.float32(ROPE_BASE), i, dtype=np.float32)
    theta = (np.arange(n, dtype=np.float32)[:, None] / freq[None]).astype(np.float64)
    return torch.from_numpy(np.cos(theta)).cuda(), torch.from_numpy(np.sin(theta)).cuda()


def _rotate64(x, cos, sin):
    """x [rows, heads, d] at the rows' cos and sin [rows, d / 2]."""
    a, b = x.chunk(2, dim=-1)
    c, s = cos[:, None], sin[:, None]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attend64(q, k, v, start):
    """Causal attention of rows q [n, hq, d] at positions start.. over k, v [ctx, hkv, d]."""
    n, hq, d = q.shape
    ctx, hkv = k.shape[0], k.shape[1]
    q = q.view(n, hkv, hq // hkv, d).permute(1, 2, 0, 3).reshape(hkv, -1, d).contiguous()
    out = torch.empty_like(q)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    pos = start + torch.arange(n, device="cuda")
    pos = pos.repeat(hq // hkv)
    step = max(1, (1 << 26) // ctx)
    for i in range(0, q.shape[1], step):
        sc = torch.matmul(q[:, i:i + step], kt) / math.sqrt(d)
        sc.masked_fill_(torch.arange(ctx, device="cuda")[None, None] > pos[None, i:i + step, None],
                        -math.inf)
        out[:, i:i + step] = torch.matmul(torch.softmax(sc, -1), vt)
    return out.view(hkv, hq // hkv, n, d).permute(2, 0, 1, 3).reshape(n, hq * d)


def _exact_attention(case, seed):
    if case["kind"] == "decode":
        ctx = _decode_lengths(case)
        rows, starts = np.ones_like(ctx), ctx - 1
    else:
        rows, starts = _prefill_lengths(case)
    s = _attention_inputs(case, seed, rows + starts, int(rows.sum()))
    hq, hkv, d, layers = case["hq"], case["hkv"], case["d"], case["layers"]
    qd, kd = hq * d, hkv * d
    cos, sin = _rope64(int((rows + starts).max()), d)
    qkv = s["proj"].double()
    k_all, v_all = s["k"].double(), s["v"].double()
    out = torch.empty((layers, int(rows.sum()), qd), dtype=torch.float64, device="cuda")
    r0 = 0
    for b, (n, sp) in enumerate(zip(rows.tolist(), starts.tolist())):
        ctx = n + sp
        at = torch.arange(ctx, device="cuda")
        page, slot = s["tables"][b].long()[at // PAGE], at % PAGE
        for li in range(layers):
            x = qkv[li, r0:r0 + n]
            y = x + s["bias"][li].double()
            q = _rotate64(y[:, :qd].view(n, hq, d), cos[sp:ctx], sin[sp:ctx])
            k = _rotate64(y[:, qd:qd + kd].view(n, hkv, d), cos[sp:ctx], sin[sp:ctx])
            x[:, :qd] = q.reshape(n, qd)
            x[:, qd:qd + kd] = k.reshape(n, kd)
            k_all[page[sp:], li, :, slot[sp:]] = k
            v_all[page[sp:], li, :, slot[sp:]] = y[:, qd + kd:].reshape(n, hkv, d)
            out[li, r0:r0 + n] = _attend64(q, k_all[page, li, :, slot], v_all[page, li, :, slot], sp)
        r0 += n
    return {"out": out, "qkv": qkv, "k": k_all, "v": v_all}


def _norm64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _exact_rows(case, seed):
    x, weights = _rows_inputs(case, seed)
    h, outs, H, I = x.double(), [], case["hidden"], case["inter"]
    for w in weights:
        w = {k: t.double() for k, t in w.items()}
        qkv = _norm64(h, w["n1"]) @ w["qkv"].t()
        h1 = qkv[:H] @ w["o"].t() + h
        gu = _norm64(h1, w["n2"]) @ w["gu"].t()
        act = torch.nn.functional.silu(gu[:I]) * gu[I:]
        h = act @ w["down"].t() + h1
        outs.append({"qkv": qkv, "h1": h1, "act": act, "h2": h})
    return outs


def _exact_model(case, seed):
    c, w = _MODEL, _model_weights(seed)
    hq, hkv, d, H, I = (c.num_attention_heads, c.num_key_value_heads, c.head_dim, c.hidden_size,
                        c.intermediate_size)
    if case["kind"] == "model_prompt":
        ids, start = _model_ids(seed, case["rows"]), 0
        shape = (_MODEL_CTX // PAGE, c.num_hidden_layers, hkv, PAGE, d)
        k_pool = torch.zeros(shape, dtype=torch.float64, device="cuda")
        v_pool = torch.zeros_like(k_pool)
    else:
        ids, start = _model_ids(seed, 1), case["pos"]
        k_pool, v_pool = (t.double() for t in _model_cache(seed))
    n = len(ids)
    ctx = start + n
    cos, sin = _rope64(ctx, d)
    cos, sin = cos[start:], sin[start:]
    at = torch.arange(ctx, device="cuda")
    page, slot = at // PAGE, at % PAGE  # the cache hands out pages 0, 1, 2, ...
    h = w["embed_tokens"][torch.tensor(ids, device="cuda")].double()
    for li, lw in enumerate(w["layers"]):
        lw = {k: t.double() for k, t in lw.items()}
        y = _norm64(h, lw["input_layernorm"]) @ lw["qkv_proj"].t() + lw["qkv_bias"]
        q = _rotate64(y[:, :H].reshape(n, hq, d), cos, sin)
        k_pool[page[start:], li, :, slot[start:]] = _rotate64(
            y[:, H:H + hkv * d].reshape(n, hkv, d), cos, sin)
        v_pool[page[start:], li, :, slot[start:]] = y[:, H + hkv * d:].reshape(n, hkv, d)
        att = _attend64(q, k_pool[page, li, :, slot], v_pool[page, li, :, slot], start)
        h = att @ lw["o_proj"].t() + h
        gu = _norm64(h, lw["post_attention_layernorm"]) @ lw["gate_up_proj"].t()
        h = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]) @ lw["down_proj"].t() + h
    last = h[-1:]
    logits = _norm64(last, w["final_norm"].double()) @ w["embed_tokens"].double().t()
    return {"logits": logits, "hidden": last, "k": k_pool, "v": v_pool}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_attention(case, seed)
    if kind == "rows":
        return _exact_rows(case, seed)
    if kind == "sample":
        return None  # a token and the sorted candidates: whole values
    return _exact_model(case, seed)
