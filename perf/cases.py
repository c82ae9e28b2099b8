"""Timed cases of the framework: what a program that serves a quantized model
has it do, each through the entry points such a program calls.

Four kinds:

* ``linear``: one quantized linear layer (``CiderLinear``, ``W4A8Linear``,
  ``W4A8GroupLinear``, or the raw int8 product) on M tokens, called eagerly.
  M = 1 is decode of one sequence, up to a few dozen a decode batch, a few
  hundred a mixed batch or a prefill chunk, thousands a long prompt.
* ``attention``: causal attention of a prefill chunk over the KV cache.
* ``layer``: one transformer layer of a prefill chunk, from the residual
  stream to the residual stream: called eagerly (a whole prompt at once), or
  replayed from a HIP graph whose length is on the device (chunked prefill).
* ``decode``: one token through the whole model to its logits, replayed from
  a HIP graph, as generation runs it.

Sizes are those of Qwen3-8B and of the Qwen3-VL-2B text model, the shapes
bench.py sweeps, and odd sizes around them.  Activations are N(0, 1) with 1 %
outlier columns x20, weights int8 or int4 uniform, as in bench.py.
"""

import dataclasses
import math

import torch

from cider_amd import CiderLinear, W4A8GroupLinear, W4A8Linear, int8_matmul_int32
from cider_amd import fused as FK
from cider_amd.qwen3 import QWEN3_8B, Qwen3, Qwen3Layer, rope_tables
from cider_amd.qwen3vl import QWEN3_VL_2B

DEV = "cuda"
CONFIGS = {"8b": QWEN3_8B, "vl2b": QWEN3_VL_2B}
HEAD_DIM = 128

# (N, K) of the linears that bench.py and the two configurations hold
SHAPES = [(10240, 2560), (2560, 10240), (12288, 4096), (4096, 12288), (6144, 4096), (4096, 4096),
          (24576, 4096), (4096, 2048), (2048, 2048), (12288, 2048), (2048, 6144)]
# int8 per channel, int8 per group, int4 per channel, int4 per group, raw int8 product
FORMATS = ["pc", "pg64", "pg128", "pg256", "w4", "w4g64", "w4g128", "int32"]
MOST_MACS = 4096 * 12288 * 4096


def _linear(name, fmt, M, N, K, dtype="float16", bias=False):
    return {"name": name, "kind": "linear", "fmt": fmt, "M": M, "N": N, "K": K, "dtype": dtype,
            "bias": bias}


def listed():
    return [
        # decode of one sequence, a linear called on its own: the smallest call, launch bound
        _linear("decode linear", "pc", 1, 10240, 2560),
        # the same with per-group scales, on the down projection's long rows
        _linear("decode linear per-group", "pg64", 1, 2560, 10240),
        # a decode batch of 16 sequences on int4 weights: the weights are read once for all
        _linear("decode batch int4", "w4g128", 16, 12288, 4096),
        # a ragged mixed batch of a bf16 model, with a bias
        _linear("mixed batch bf16", "pc", 137, 2560, 10240, "bfloat16", True),
        # the raw integer product, a tuning shape of the MLP
        _linear("raw int8 product", "int32", 256, 18944, 3584),
        # a long prompt: the shape the headline figure is quoted on
        _linear("prompt linear", "pc", 4096, 10240, 2560),
        # a ragged multimodal prompt (3455 tokens) on per-group weights
        _linear("prompt linear per-group", "pg128", 3455, 10240, 2560),
        # a prompt of 1334 tokens on int4 weights in the reference's packing
        _linear("prompt linear int4", "w4", 1334, 12288, 4096),
        # attention of a whole 2048-token prompt, 32 query and 8 KV heads
        {"name": "prompt attention", "kind": "attention", "c": 2048, "n": 2048, "H": 32, "KV": 8},
        # a layer of chunked prefill: 512 tokens after 1536, replayed from a graph
        {"name": "chunk layer", "kind": "layer", "model": "vl2b", "c": 512, "n": 2048,
         "graph": True},
        # a layer of a 2048-token prefill, called eagerly
        {"name": "prompt layer", "kind": "layer", "model": "8b", "c": 2048, "n": 2048,
         "graph": False},
        # one generated token after a 2048-token prompt, 36 layers and the lm_head
        {"name": "decode step", "kind": "decode", "model": "8b", "pos": 2111},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["linear", "attention", "layer", "decode"], [8, 2, 2, 1])[0]
    if kind == "linear":
        fmt = rng.choice(FORMATS)
        gs = _group(fmt) or 64
        if rng.random() < 0.7:
            N, K = rng.choice(SHAPES)
        else:  # widths between the configured ones: any N, K of whole groups
            N, K = _log(rng, 500, 12288), gs * max(1, _log(rng, 512, 12288) // gs)
        M = _log(rng, 1, min(4096, MOST_MACS // (N * K)))
        return {"kind": "linear", "fmt": fmt, "M": M, "N": N, "K": K,
                "dtype": "float16" if fmt == "int32" else rng.choice(["float16", "bfloat16"]),
                "bias": fmt not in ("w4", "int32") and rng.random() < 0.5}
    if kind == "attention":
        c = _log(rng, 33, 2048)
        n = c + (rng.randrange(0, 2048) if rng.random() < 0.5 else 0)
        H, KV = rng.choice([(32, 8), (16, 8)])
        return {"kind": "attention", "c": c, "n": min(n, 2048 + c // 4), "H": H, "KV": KV}
    if kind == "layer":
        if rng.random() < 0.5:
            c = rng.randrange(100, 513)
            return {"kind": "layer", "model": "vl2b", "c": c, "n": c + rng.randrange(0, 3000),
                    "graph": True}
        c = _log(rng, 65, 2047)
        return {"kind": "layer", "model": "8b", "c": c, "n": c, "graph": False}
    model = rng.choice(["8b", "vl2b"])
    return {"kind": "decode", "model": model,
            "pos": _log(rng, 64, 2110 if model == "8b" else 3800)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _group(fmt):
    return int(fmt[2:]) if fmt[:2] == "pg" else int(fmt[3:]) if fmt[:3] == "w4g" else 0


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _activations(M, K, g):
    """fp16 N(0, 1) with K // 100 outlier columns x20."""
    x = torch.randn(M, K, device=DEV, generator=g)
    cols = torch.randperm(K, device=DEV, generator=g)[: K // 100]
    x[:, cols] *= 20.0
    return x.half()


def _linear_inputs(case, seed):
    """The plain tensors of a linear: x, integer weights [N, K], scales, bias."""
    M, N, K, fmt = case["M"], case["N"], case["K"], case["fmt"]
    g = _gen(seed)
    if fmt == "int32":
        a = torch.randint(-128, 128, (M, K), dtype=torch.int8, device=DEV, generator=g)
        b = torch.randint(-128, 128, (N, K), dtype=torch.int8, device=DEV, generator=g)
        return a, b, None, None
    x = _activations(M, K, g).to(getattr(torch, case["dtype"]))
    lo, hi = (-7, 8) if fmt[:2] == "w4" else (-127, 128)
    w = torch.randint(lo, hi, (N, K), dtype=torch.int8, device=DEV, generator=g)
    gs = _group(fmt)
    shape = (K // gs, N) if gs else (N,)
    s = torch.rand(shape, device=DEV, generator=g) * 9e-3 + 1e-3
    if fmt[:2] == "w4":
        s = s * 16.0
    if fmt[:3] == "w4g":
        s = s.half()
    b = torch.randn(N, device=DEV, generator=g).half() if case["bias"] else None
    return x, w, s, b


def _nibbles_low_first(w):
    """[N, K] -> uint8 [N, K / 2], even k in the low nibble, two's complement."""
    u = w.to(torch.uint8) & 15
    return (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()


def _nibbles_reference(w):
    """[N, K] -> uint8 [K / 2, N], even k in the high nibble, zero point 8."""
    u = (w + 8).to(torch.uint8).t()
    return ((u[0::2] << 4) | u[1::2]).contiguous()


def _prepare_linear(case, seed):
    x, w, s, b = _linear_inputs(case, seed)
    fmt, N, K = case["fmt"], case["N"], case["K"]
    if fmt == "int32":
        return {"a": x, "b": w}
    if fmt == "w4":
        layer = W4A8Linear(_nibbles_reference(w), s, K)
    elif fmt[:3] == "w4g":
        layer = W4A8GroupLinear(_nibbles_low_first(w), s, _group(fmt), b)
    else:
        layer = CiderLinear(w, s, _group(fmt), K, N, b)
    return {"x": x, "layer": layer}


def _attention_inputs(case, seed):
    """Queries and caches as the q/k norms leave them: rows of unit variance."""
    g = _gen(seed)
    c, n, H, KV = case["c"], case["n"], case["H"], case["KV"]
    T = (n + 7) // 8 * 8
    q = torch.randn(c, H, HEAD_DIM, device=DEV, generator=g).half()
    k = torch.randn(KV, T, HEAD_DIM, device=DEV, generator=g).half()
    v = torch.randn(KV, T, HEAD_DIM, device=DEV, generator=g).half()
    return q, k, v


def _prepare_attention(case, seed):
    q, k, v = _attention_inputs(case, seed)
    return {"q": q, "k": k, "v": v, "n": case["n"],
            "ws": FK.attn_prefill_workspace(case["c"], case["n"], case["H"], DEV)}


def _layer_inputs(case, seed):
    cfg = CONFIGS[case["model"]]
    c, n = case["c"], case["n"]
    g = _gen(seed)
    layer = Qwen3Layer(cfg, g, torch.device(DEV))
    T = (n + 511) // 512 * 512
    x = _activations(c, cfg.hidden_size, g)
    pending = torch.randn(c, cfg.hidden_size, device=DEV, generator=g).half()
    kv = [torch.randn(cfg.num_kv_heads, T, HEAD_DIM, device=DEV, generator=g).half()
          for _ in range(2)]
    for t in kv:
        t[:, n - c:] = 0
    tables = rope_tables(HEAD_DIM, T, cfg.rope_theta, DEV)
    return cfg, layer, x, pending, kv[0], kv[1], tables


def _prepare_layer(case, seed):
    cfg, layer, x, pending, kc, vc, tables = _layer_inputs(case, seed)
    c, n = case["c"], case["n"]
    pos = torch.arange(n - c, n, device=DEV)
    state = {"layer": layer, "x": x, "pending": pending, "k": kc, "v": vc, "tables": tables,
             "pos": pos, "n": n, "ws": None, "graph": None}
    if not case["graph"]:
        state["ws"] = FK.attn_prefill_quantize_workspace(c, n, cfg.num_heads, DEV)
        return state
    # as chunked prefill keeps it: static input buffers, the length on the
    # device, and a workspace for any length up to the cache's capacity
    cap = kc.shape[1]
    ws = FK.attn_prefill_quantize_workspace(c, cap, cfg.num_heads, DEV)
    n_dev = torch.tensor([n], dtype=torch.int64, device=DEV)
    bx, bp = x.clone(), pending.clone()

    def chunk():
        return layer.prefill_fused(bx, bp, tables, pos, pos, kc, vc, cap, ws, n_dev)

    g, out = _captured(chunk)
    state.update(graph=g, out=out, bx=bx, bp=bp, ws=ws, n_dev=n_dev)
    return state


def _captured(fn):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.no_grad():
        fn()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(g):
        out = fn()
    torch.cuda.synchronize()
    return g, out


def _decode_model(case, seed):
    cfg = CONFIGS[case["model"]]
    model = Qwen3(dataclasses.replace(cfg), max_len=case["pos"] + 65, seed=seed, device=DEV)
    g = _gen(seed + 1)
    for cache in (model.k_cache, model.v_cache):
        for i in range(cfg.num_layers):
            cache[i].normal_(generator=g)
            cache[i, :, case["pos"]:] = 0
    tok = torch.randint(0, cfg.vocab_size, (1,), device=DEV, generator=g)
    pos = torch.tensor([case["pos"]], dtype=torch.int64, device=DEV)
    return cfg, model, tok, pos


def _prepare_decode(case, seed):
    _, model, tok, pos = _decode_model(case, seed)
    g, logits = _captured(lambda: model.decode_step(tok, pos))
    return {"model": model, "tok": tok, "pos": pos, "graph": g, "logits": logits}


def prepare(case, seed):
    return {"linear": _prepare_linear, "attention": _prepare_attention,
            "layer": _prepare_layer, "decode": _prepare_decode}[case["kind"]](case, seed)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

@torch.no_grad()
def run(state):
    if "a" in state:
        return int8_matmul_int32(state["a"], state["b"])
    if "model" in state:
        state["graph"].replay()
        return {"logits": state["logits"], "k": state["model"].k_cache,
                "v": state["model"].v_cache}
    if "q" in state:
        return FK.attn_prefill(state["q"], state["k"], state["v"], state["n"],
                               1.0 / math.sqrt(HEAD_DIM), ws=state["ws"])
    if "pending" not in state:
        return state["layer"](state["x"])
    if state["graph"] is not None:
        state["bx"].copy_(state["x"])  # the layer adds into its input
        state["bp"].copy_(state["pending"])
        state["graph"].replay()
        x, pending = state["out"]
    else:
        x, pending = state["layer"].prefill_fused(
            state["x"].clone(), state["pending"], state["tables"], state["pos"], state["pos"],
            state["k"], state["v"], state["n"], state["ws"])
    return {"x": x, "pending": pending, "k": state["k"], "v": state["v"]}


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------

def _linear_work(fmt, M, N, K):
    if fmt == "int32":
        return M * K + N * K + 4 * M * N, 2 * M * N * K
    gs = _group(fmt)
    weights = N * K // 2 if fmt[:2] == "w4" else N * K
    scales = (N * K // gs if gs else N) * (2 if fmt[:3] == "w4g" else 4)
    return 2 * M * K + weights + scales + 2 * M * N, 2 * M * N * K


def _attention_work(c, n, H, KV):
    pairs = c * (n - c) + c * (c + 1) // 2
    return 2 * HEAD_DIM * (2 * c * H + 2 * n * KV), 4 * H * HEAD_DIM * pairs


def work(case):
    if case["kind"] == "linear":
        b, f = _linear_work(case["fmt"], case["M"], case["N"], case["K"])
    elif case["kind"] == "attention":
        b, f = _attention_work(case["c"], case["n"], case["H"], case["KV"])
    else:
        cfg = CONFIGS[case["model"]]
        c, n = (1, case["pos"] + 1) if case["kind"] == "decode" else (case["c"], case["n"])
        kv = cfg.num_kv_heads
        # weights and scales, the cache's earlier rows read and the chunk's written
        b = sum(N * K + 4 * N for _, N, K in cfg.linear_shapes())
        b += 2 * 2 * HEAD_DIM * kv * n
        f = sum(2 * c * N * K for _, N, K in cfg.linear_shapes())
        f += _attention_work(c, n, cfg.num_heads, kv)[1]
        if case["kind"] == "decode":
            b = b * cfg.num_layers + 2 * cfg.vocab_size * (cfg.hidden_size + 1)
            f = f * cfg.num_layers + 2 * cfg.vocab_size * cfg.hidden_size
        else:
            b += 4 * 2 * c * cfg.hidden_size
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------
# results in 64 bits
# ---------------------------------------------------------------------------

def _quantized(x):
    """x quantized per token to int8 and back: absmax / 127, half away from zero."""
    s = x.abs().amax(1, keepdim=True) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    r = x / s
    q = torch.sign(r) * torch.floor(r.abs() + 0.5)
    return q.clamp(-128, 127) * s


def _linear64(x, w, s, b, quantize):
    """x (64 bits) [M, K] on integer weights [N, K], scales [N] or [G, N]."""
    if quantize:
        x = _quantized(x)
    wd = w.double()
    if s.dim() == 2:
        wd = (wd.view(w.shape[0], s.shape[0], -1) * s.double().t()[:, :, None]).view_as(wd)
        y = x @ wd.t().contiguous()
    else:
        y = (x @ wd.t().contiguous()) * s.double()
    return y if b is None else y + b.double()


def _rms64(x, w, eps):
    return w.double() * x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _rope64(x, cos, sin):
    h = x.shape[-1] // 2
    rot = torch.cat([-x[..., h:], x[..., :h]], dim=-1)
    return x * cos.double()[:, None, :] + rot * sin.double()[:, None, :]


def _attention64(q, k, v):
    """q [c, H, D] at the last c of the n rows of k, v [KV, n, D]."""
    c, H, D = q.shape
    KV, n, _ = k.shape
    mask = torch.arange(n, device=q.device)[None, :] > torch.arange(n - c, n,
                                                                     device=q.device)[:, None]
    out = torch.empty(c, H, D, dtype=torch.float64, device=q.device)
    for h in range(H):
        j = h // (H // KV)
        p = (q[:, h] @ k[j].t().contiguous()) / math.sqrt(D)
        out[:, h] = torch.softmax(p.masked_fill(mask, float("-inf")), dim=-1) @ v[j]
    return out.reshape(c, H * D)


def _layer64(cfg, layer, x, kc, vc, cos, sin, n, quantize):
    """One layer on the residual stream x [c, hidden] at rows n - c .. n - 1 of
    the caches (64 bits, written here).  Returns the stream after attention
    and the MLP's output."""
    c = x.shape[0]
    H, KV = cfg.num_heads, cfg.num_kv_heads

    def lin(m, v):
        return _linear64(v, m.w_int8, m.scale_w, m.bias, quantize)

    qkv = lin(layer.qkv, _rms64(x, layer.input_norm, cfg.rms_eps))
    q, k, v = qkv.view(c, H + 2 * KV, HEAD_DIM).split([H, KV, KV], dim=1)
    q = _rope64(_rms64(q, layer.q_norm, cfg.rms_eps), cos, sin)
    kc[:, n - c:n] = _rope64(_rms64(k, layer.k_norm, cfg.rms_eps), cos, sin).transpose(0, 1)
    vc[:, n - c:n] = v.transpose(0, 1)
    x = x + lin(layer.o, _attention64(q, kc[:, :n], vc[:, :n]))
    gu = lin(layer.gate_up, _rms64(x, layer.post_norm, cfg.rms_eps))
    i = cfg.intermediate_size
    return x, lin(layer.down, torch.nn.functional.silu(gu[:, :i]) * gu[:, i:])


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "linear":
        if case["fmt"] == "int32":
            return None
        x, w, s, b = _linear_inputs(case, seed)
        # one token on int8 weights is not quantized; x is taken in fp16
        quantize = case["M"] > 1 or case["fmt"][:2] == "w4"
        return _linear64(x.half().double(), w, s, b, quantize)
    if case["kind"] == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        return _attention64(q, k[:, :case["n"]], v[:, :case["n"]])
    if case["kind"] == "layer":
        cfg, layer, x, pending, kc, vc, (cos, sin) = _layer_inputs(case, seed)
        c, n = case["c"], case["n"]
        kc, vc = kc.double(), vc.double()
        x, pending = _layer64(cfg, layer, x.double() + pending.double(), kc, vc,
                              cos[n - c:n], sin[n - c:n], n, c > 1)
        return {"x": x, "pending": pending, "k": kc, "v": vc}
    cfg, model, tok, pos = _decode_model(case, seed)
    p = case["pos"]
    x = model.embed[tok].double()
    for i, layer in enumerate(model.layers):
        kc, vc = model.k_cache[i].double(), model.v_cache[i].double()
        x, down = _layer64(cfg, layer, x, kc, vc, model.cos[p:p + 1], model.sin[p:p + 1],
                           p + 1, False)
        x = x + down
    logits = _rms64(x, model.final_norm, cfg.rms_eps) @ model.lm_head.double().t().contiguous()
    return {"logits": logits, "k": None, "v": None}


def tolerance(case):
    if case["kind"] == "linear":
        if case["fmt"] == "int32":
            return "exact"
        # one rounding to the output type: 2^-12 relative on average in fp16, 2^-9 in bf16
        return {"rel": 1e-3 if case["dtype"] == "float16" else 7e-3}
    if case["kind"] == "attention":
        return {"rel": 2e-3}
    if case["kind"] == "layer":
        # a changed rounding before an int8 quantization moves values by a whole step of
        # it (0.8 % of a row's maximum) where they lay near a half
        # (measured against 64 bits: 0.022 and 0.028 on the MLP's output)
        return {"rel": 0.03, "max": 0.5}
    # measured against 64 bits: 0.0063 after 36 layers of fp16 activations
    return {"rel": 0.025, "max": 0.25}
