"""The work a user of this framework has it do, as cases that can be timed.

Two layer shapes run through every kind of case: the 200M model's layer
(hidden 896, shared 3072, 4 experts x 64, top-2, vocabulary 32000), which is
what decodes, prefills and trains in bf16 (and fp32), and the scaled layer
(hidden 2048, shared 5632, 16 experts x 256), which serves e4m3 weights and
trains its experts grouped.  Kinds:

* ``decode``: a stack of layers' MLP halves captured once in a HIP graph and
  replayed per token, as a serving loop does;
* ``layer``: one inference call on a prompt or a batch of prompts;
* ``train``: one training step of the block's MLP half (forward, backward,
  weight update, so that the next step sees other weights);
* ``model``: the 16-layer decoder: a prompt alone, or a prompt and the decode
  steps of a reply.

Token ids follow a truncated Zipf(1.1) law, activations are N(0, 1), weights
N(0, 0.02); everything is drawn on the GPU from the case's seed.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "complexity-framework_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from complexity_amd import ops  # noqa: E402
from complexity_amd.decoder import TRGQAConfig, TRGQADecoder  # noqa: E402
from complexity_amd.tr_hash import TRHashEngine, TRHashEngineConfig  # noqa: E402

VOCAB = 32000
TOP_K = 2
ROUTED_SCALE = 2.0          # the released 200M model's routed output scale
EPS = 1e-6
STD = 0.02
E4M3_MAX = 448.0
SHAPES = {
    "200m": dict(hidden=896, shared=3072, experts=4, width=64),
    "scaled": dict(hidden=2048, shared=5632, experts=16, width=256),
}
_SHARED = ("shared_gate", "shared_up", "shared_down")
_EXPERT = ("expert_gate", "expert_up", "expert_down")


def listed():
    return [
        # one step of 8 sequences through the 16 layers of the 200M model: the smallest serving batch
        {"name": "decode_8", "kind": "decode", "shape": "200m", "dtype": "bf16", "layers": 16, "tokens": 8},
        # 64 concurrent sequences
        {"name": "decode_64", "kind": "decode", "shape": "200m", "dtype": "bf16", "layers": 16, "tokens": 64},
        # the scaled layer's e4m3 weights at 32 sequences (two layers: more weights over the rotated
        # states than the last-level cache holds)
        {"name": "decode_fp8_32", "kind": "decode", "shape": "scaled", "dtype": "fp8", "layers": 2, "tokens": 32},
        # one user's prompt of a ragged length through a block's MLP half (RMSNorm and residual fused)
        {"name": "prompt_777", "kind": "layer", "shape": "200m", "dtype": "bf16", "tokens": 777, "norm": True,
         "w8a8": False},
        # the benchmark prefill: 8 prompts of 2048 tokens
        {"name": "prefill_16384", "kind": "layer", "shape": "200m", "dtype": "bf16", "tokens": 16384,
         "norm": False, "w8a8": False},
        # the fp32 layer, for checks against other implementations and small fp32 models
        {"name": "fp32_2048", "kind": "layer", "shape": "200m", "dtype": "fp32", "tokens": 2048, "norm": False,
         "w8a8": False},
        # the scaled layer with e4m3 weights on 16 prompts of 2048 tokens: the largest prefill
        {"name": "fp8_32768", "kind": "layer", "shape": "scaled", "dtype": "fp8", "tokens": 32768, "norm": False,
         "w8a8": False},
        # the same weights with e4m3 activations, on a ragged batch of prompts
        {"name": "w8a8_12001", "kind": "layer", "shape": "scaled", "dtype": "fp8", "tokens": 12001, "norm": False,
         "w8a8": True},
        # one training step of the 200M block's MLP half on 8 x 2048 tokens
        {"name": "train_16384", "kind": "train", "shape": "200m", "dtype": "bf16", "tokens": 16384},
        # the scaled layer's training step: experts run grouped, a ragged packed batch
        {"name": "train_scaled_3001", "kind": "train", "shape": "scaled", "dtype": "bf16", "tokens": 3001},
        # a chat turn of one user: a ragged prompt, then the reply's decode steps
        {"name": "reply_1x197", "kind": "model", "batch": 1, "prompt": 197, "steps": 16},
        # the prompts of 8 users at the model's full context
        {"name": "prompts_8x2048", "kind": "model", "batch": 8, "prompt": 2048, "steps": 0},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "layer", "layer", "layer", "train", "train", "model"))
    if kind == "decode":
        if rng.random() < 0.6:
            return {"kind": kind, "shape": "200m", "dtype": "bf16", "layers": 16, "tokens": _log_int(rng, 1, 128)}
        return {"kind": kind, "shape": "scaled", "dtype": "fp8", "layers": 2, "tokens": _log_int(rng, 1, 128)}
    if kind == "layer":
        what = rng.choice(("bf16", "bf16", "fp32", "fp8", "w8a8"))
        if what == "bf16":
            return {"kind": kind, "shape": "200m", "dtype": "bf16", "tokens": _log_int(rng, 129, 16384),
                    "norm": rng.random() < 0.5, "w8a8": False}
        if what == "fp32":
            return {"kind": kind, "shape": "200m", "dtype": "fp32", "tokens": _log_int(rng, 129, 4096),
                    "norm": rng.random() < 0.5, "w8a8": False}
        return {"kind": kind, "shape": "scaled", "dtype": "fp8", "tokens": _log_int(rng, 129, 32768),
                "norm": what == "fp8" and rng.random() < 0.5, "w8a8": what == "w8a8"}
    if kind == "train":
        if rng.random() < 0.6:
            return {"kind": kind, "shape": "200m", "dtype": "bf16", "tokens": _log_int(rng, 256, 16384)}
        return {"kind": kind, "shape": "scaled", "dtype": "bf16", "tokens": _log_int(rng, 256, 4096)}
    batch = _log_int(rng, 1, 8)
    if rng.random() < 0.5:
        return {"kind": kind, "batch": batch, "prompt": _log_int(rng, 32, 512), "steps": rng.randint(4, 16)}
    return {"kind": kind, "batch": batch, "prompt": _log_int(rng, 128, 2048), "steps": 0}


# --------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _zipf_ids(g, *shape):
    p = torch.arange(1, VOCAB + 1, dtype=torch.float64, device="cuda").pow(-1.1)
    n = math.prod(shape)
    return torch.multinomial((p / p.sum()).float(), n, replacement=True, generator=g).view(*shape)


def _route_table(g, experts):
    """[2, VOCAB]: two different experts for each token id, as a persisted table holds them."""
    first = torch.randint(0, experts, (VOCAB,), generator=g, device="cuda")
    step = torch.randint(1, experts, (VOCAB,), generator=g, device="cuda")
    return torch.stack((first, (first + step) % experts))


def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _layer_weights(g, shape, dtype):
    H, S, E, W = shape["hidden"], shape["shared"], shape["experts"], shape["width"]
    sizes = {"shared_gate": (S, H), "shared_up": (S, H), "shared_down": (H, S),
             "expert_gate": (E, H, W), "expert_up": (E, H, W), "expert_down": (E, W, H)}
    return {n: _normal(g, *sizes[n], std=STD, dtype=dtype) for n in _SHARED + _EXPERT}


def _inputs(case, seed):
    """Everything a layer-level case is computed from: plain tensors made from the seed."""
    shape, dt = SHAPES[case["shape"]], _dtype(case)
    g = _generator(seed)
    n = case["tokens"]
    layers = case.get("layers", 1)
    t = {
        "ids": _zipf_ids(g, 1, n) if case["kind"] != "decode" else _zipf_ids(g, n, 1),
        "tables": [_route_table(g, shape["experts"]) for _ in range(layers)],
        "weights": [_layer_weights(g, shape, dt) for _ in range(layers)],
        "norms": [(torch.rand(shape["hidden"], generator=g, device="cuda") + 0.5).to(dt) for _ in range(layers)],
    }
    t["x"] = _normal(g, *t["ids"].shape, shape["hidden"], dtype=dt)
    if case["kind"] == "train":
        t["dout"] = _normal(g, *t["x"].shape, std=0.1, dtype=dt)
    return t


def _engine(case, table, weights, layer=0):
    shape = SHAPES[case["shape"]]
    train = case["kind"] == "train"
    engine = TRHashEngine(TRHashEngineConfig(
        hidden_size=shape["hidden"], vocab_size=VOCAB, num_experts=shape["experts"], top_k=TOP_K,
        shared_width=shape["shared"], expert_width=shape["width"], routing_strategy="token_id_multi_hash",
        layer_index=layer, routed_output_scale=ROUTED_SCALE, phase="training" if train else "inference",
        precision=case["dtype"]))
    engine = engine.to(device="cuda", dtype=_dtype(case))
    with torch.no_grad():
        for name in _SHARED:
            getattr(engine, name).weight.copy_(weights[name])
        for name in _EXPERT:
            getattr(engine, name).copy_(weights[name])
    engine.load_route_table(table)
    if case["dtype"] == "fp8":
        engine.quantize_fp8_()
        engine.fp8_activations = bool(case.get("w8a8", False))
    return engine.train() if train else engine.eval()


def prepare(case, seed):
    if case["kind"] == "model":
        return _prepare_model(case, seed)
    t = _inputs(case, seed)
    engines = [_engine(case, t["tables"][i], t["weights"][i], i) for i in range(len(t["weights"]))]
    state = {"case": case, "engines": engines, "ids": t["ids"], "norms": t["norms"]}
    if case["kind"] == "train":
        state["x"] = t["x"].requires_grad_(True)
        state["dout"] = t["dout"]
        state["norm"] = torch.nn.Parameter(t["norms"][0])
        # a fine-tuning step size: every step changes the weights (and what is derived from them) a little
        state["opt"] = torch.optim.SGD([*engines[0].parameters(), state["norm"]], lr=1e-6)
        return state
    state["x"] = t["x"]
    if case["kind"] == "decode":
        _capture(state)
    return state


def _stack(state):
    h = state["x"]
    for engine, norm in zip(state["engines"], state["norms"]):
        h = engine.forward_norm_residual(h, state["ids"], norm, EPS)
    return h


def _capture(state):
    """The serving loop's graph of one step: warmed up and recorded on a stream of its own."""
    scratch = ops.workspace_scope()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), scratch, torch.cuda.stream(side):
        _stack(state)
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), scratch, torch.cuda.graph(graph):
        state["out"] = _stack(state)
    state["graph"], state["scratch"] = graph, scratch


def _model_inputs(case, seed):
    """Decoder parameters by name (the decoder's own state-dict names), route tables and token ids."""
    cfg = TRGQAConfig()
    g = _generator(seed)
    H, D, S, W, E = cfg.hidden_size, cfg.head_dim, cfg.shared_width, cfg.expert_width, cfg.num_experts
    q, kv = cfg.num_heads * D, cfg.num_kv_heads * D
    resid = STD / math.sqrt(2 * cfg.num_layers)
    bf = torch.bfloat16

    def ones(n):
        return (torch.rand(n, generator=g, device="cuda") * 0.5 + 0.75).to(bf)

    p = {"embed_tokens.weight": _normal(g, cfg.vocab_size, H, std=STD, dtype=bf), "norm.weight": ones(H)}
    tables = []
    for i in range(cfg.num_layers):
        b = f"layers.{i}."
        p[b + "input_layernorm.weight"] = ones(H)
        p[b + "post_attention_layernorm.weight"] = ones(H)
        p[b + "self_attn.q_proj.weight"] = _normal(g, q, H, std=STD, dtype=bf)
        p[b + "self_attn.k_proj.weight"] = _normal(g, kv, H, std=STD, dtype=bf)
        p[b + "self_attn.v_proj.weight"] = _normal(g, kv, H, std=STD, dtype=bf)
        p[b + "self_attn.o_proj.weight"] = _normal(g, H, q, std=resid, dtype=bf)
        p[b + "self_attn.q_norm.weight"] = ones(D)
        p[b + "self_attn.k_norm.weight"] = ones(D)
        p[b + "mlp.shared_gate.weight"] = _normal(g, S, H, std=STD, dtype=bf)
        p[b + "mlp.shared_up.weight"] = _normal(g, S, H, std=STD, dtype=bf)
        p[b + "mlp.shared_down.weight"] = _normal(g, H, S, std=resid, dtype=bf)
        p[b + "mlp.expert_gate"] = _normal(g, E, H, W, std=STD, dtype=bf)
        p[b + "mlp.expert_up"] = _normal(g, E, H, W, std=STD, dtype=bf)
        p[b + "mlp.expert_down"] = _normal(g, E, W, H, std=resid, dtype=bf)
        tables.append(_route_table(g, E))
    ids = _zipf_ids(g, case["batch"], case["prompt"] + case["steps"])
    return cfg, p, tables, ids


def _prepare_model(case, seed):
    cfg, params, tables, ids = _model_inputs(case, seed)
    decoder = TRGQADecoder(cfg).to(device="cuda", dtype=torch.bfloat16).eval()
    with torch.no_grad():
        for name, p in decoder.named_parameters():
            p.copy_(params[name])
    for block, table in zip(decoder.layers, tables):
        block.mlp.load_route_table(table)
    T = case["prompt"]
    return {"case": case, "decoder": decoder, "prompt": ids[:, :T].contiguous(),
            "reply": [ids[:, T + s].contiguous() for s in range(case["steps"])]}


# --------------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    if case["kind"] == "decode":
        state["graph"].replay()
        return state["out"]
    if case["kind"] == "model":
        return _run_model(state)
    engine = state["engines"][0]
    if case["kind"] == "layer":
        with torch.no_grad():
            if case["norm"]:
                return engine.forward_norm_residual(state["x"], state["ids"], state["norms"][0], EPS)
            return engine(state["x"], state["ids"])
    state["opt"].zero_grad(set_to_none=True)
    x = state["x"]
    x.grad = None
    out = engine.forward_norm_residual(x, state["ids"], state["norm"], EPS)
    out.backward(state["dout"])
    grads = {"x": x.grad, "norm": state["norm"].grad}
    for name in _SHARED:
        grads[name] = getattr(engine, name).weight.grad
    for name in _EXPERT:
        grads[name] = getattr(engine, name).grad
    state["opt"].step()
    return {"out": out.detach(), "grads": grads}


def _run_model(state):
    """Prompt, then one decode step for each token the caller's sampler chose."""
    d, steps = state["decoder"], state["case"]["steps"]
    with torch.no_grad():
        h = d.prefill(state["prompt"], max_new_tokens=steps, return_logits=False)
        logits = [d.logits(h[:, -1])]
        for token in state["reply"]:
            logits.append(d.decode_step(token))
        return {"logits": torch.stack(logits, 1), "hidden": h}


# --------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    if case["kind"] == "model":
        return _model_work(case)
    s = SHAPES[case["shape"]]
    H, S, E, W = s["hidden"], s["shared"], s["experts"], s["width"]
    n, layers = case["tokens"], case.get("layers", 1)
    act = 4 if case["dtype"] == "fp32" else 2
    wbytes = {"fp32": 4, "bf16": 2, "fp8": 1}[case["dtype"]]
    experts = min(E, TOP_K * n)
    weights = layers * wbytes * (3 * H * S + 3 * experts * H * W)
    rows = n * H * act
    flops = 6 * n * H * (S + TOP_K * W) * layers
    ids = 8 * n + 8 * TOP_K * min(n, VOCAB) * layers
    if case["kind"] == "train":
        # x, dout in; out, dx out; every weight read, its gradient written, and read, written by the update
        return {"bytes": 4 * rows + 3 * weights + ids, "flops": 3 * flops}
    return {"bytes": 2 * rows + weights + ids, "flops": flops}


def _model_work(case):
    c = TRGQAConfig()
    H, D, L = c.hidden_size, c.head_dim, c.num_layers
    q, kv = c.num_heads * D, c.num_kv_heads * D
    B, T, steps = case["batch"], case["prompt"], case["steps"]
    proj = H * (q + 2 * kv) + q * H
    mlp_w = 3 * H * c.shared_width + 3 * c.num_experts * H * c.expert_width
    layer_w = 2 * (proj + mlp_w)
    mlp_f = 6 * H * (c.shared_width + c.top_k * c.expert_width)
    pairs = B * (T * (T + 1) // 2)
    flops = L * (B * T * (2 * proj + mlp_f) + 4 * q * pairs) + 2 * B * H * c.vocab_size
    cache = 2 * 2 * kv * B * T * L
    head = 2 * H * c.vocab_size
    nbytes = L * layer_w + cache + head + 2 * B * T * H * 2 + 2 * B * c.vocab_size
    for i in range(steps):
        flops += L * (B * (2 * proj + mlp_f) + 4 * q * B * (T + i + 1)) + 2 * B * H * c.vocab_size
        nbytes += L * layer_w + head + 2 * 2 * kv * B * (T + i + 1) * L + 2 * B * c.vocab_size
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the measured distance from the 64-bit result (in brackets)
    if case["kind"] == "model":
        return {"rel": 0.03, "max": 0.4}        # 16 layers in bf16 (0.015)
    if case["kind"] == "decode":
        return {"rel": 0.03, "max": 0.3}        # a stack of layers, rounded to bf16 after each (0.006 to 0.0085)
    if case["dtype"] == "fp32":
        return {"rel": 6e-6, "max": 1e-4}       # fp32 sums (1.3e-6)
    if case["kind"] == "train":
        return {"rel": 0.02, "max": 0.2}        # bf16 pre-activation gradients (0.005)
    if case["dtype"] == "fp8":
        # bf16 routed rows at twice their weight (0.0053), e4m3 h besides (0.0087)
        return {"rel": 0.03 if case["w8a8"] else 0.02, "max": 0.3 if case["w8a8"] else 0.2}
    return {"rel": 0.01, "max": 0.1}            # one bf16 layer (0.0023)


# --------------------------------------------------------------------------- the same in 64 bits
def _quantized(w, dim):
    """w as e4m3 codes times one scale per output channel (amax / 448 over `dim`)."""
    w = w.float()
    amax = w.abs().amax(dim=dim, keepdim=True)
    scale = torch.where(amax > 0, amax / E4M3_MAX, torch.ones_like(amax))
    q = (w / scale).clamp(-E4M3_MAX, E4M3_MAX).to(torch.float8_e4m3fn)
    return q.double() * scale.double()


def _mx_blocks(h):
    """h as e4m3 codes with the smallest power of two per 32 features that keeps the block's maximum in range."""
    b = h.view(h.shape[0], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    scale = torch.exp2(torch.ceil(torch.log2(amax.clamp_min(1e-300) / E4M3_MAX)))
    scale = torch.where(amax > 0, scale, torch.ones_like(scale))
    return ((b / scale).float().to(torch.float8_e4m3fn).double() * scale).view_as(h)


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def _rms(x, weight):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * weight


def _mlp(x, ids, table, w, w8a8=False):
    """x [n, H] in 64 bits -> shared(x) + ROUTED_SCALE * sum of the token's two experts, half each."""
    xs = _quantized(x, 1) if w8a8 else x
    h = _silu_mul(xs @ w["shared_gate"].t(), xs @ w["shared_up"].t())
    out = (_mx_blocks(h) if w8a8 else h) @ w["shared_down"].t()
    routes = table[:, ids]
    for e in range(w["expert_gate"].shape[0]):
        rows = (routes == e).any(0).nonzero().squeeze(1)
        if rows.numel():
            xe = x.index_select(0, rows)
            y = _silu_mul(xe @ w["expert_gate"][e], xe @ w["expert_up"][e]) @ w["expert_down"][e]
            out = out.index_add(0, rows, y * (ROUTED_SCALE / TOP_K))
    return out


def exact(case, seed):
    if case["kind"] == "model":
        return _exact_model(case, seed)
    t = _inputs(case, seed)
    shape = t["x"].shape
    ids = t["ids"].reshape(-1)
    x = t["x"].reshape(-1, shape[-1]).double()
    norms = [v.double() for v in t["norms"]]
    if case["dtype"] == "fp8":
        weights = [{n: _quantized(v, 1) for n, v in w.items()} for w in t["weights"]]
    else:
        weights = [{n: v.double() for n, v in w.items()} for w in t["weights"]]
    if case["kind"] == "train":
        leaves = {"x": x, "norm": norms[0], **weights[0]}
        for v in leaves.values():
            v.requires_grad_(True)
        out = x + _mlp(_rms(x, norms[0]), ids, t["tables"][0], weights[0])
        grads = torch.autograd.grad(out, list(leaves.values()), t["dout"].reshape(out.shape).double())
        grads = dict(zip(leaves, grads))
        grads["x"] = grads["x"].view(shape)
        return {"out": out.detach().view(shape), "grads": grads}
    with torch.no_grad():
        if case["kind"] == "decode" or case["norm"]:
            for table, w, norm in zip(t["tables"], weights, norms):
                x = x + _mlp(_rms(x, norm), ids, table, w)
            return x.view(shape)
        return _mlp(x, ids, t["tables"][0], weights[0], case["w8a8"]).view(shape)


def _exact_model(case, seed):
    cfg, params, tables, ids = _model_inputs(case, seed)
    B, N = ids.shape
    D, kvh, heads = cfg.head_dim, cfg.num_kv_heads, cfg.num_heads
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D))
    ang = torch.outer(torch.arange(N, dtype=torch.float64, device="cuda"), inv)
    cos, sin = torch.cat((ang, ang), -1).cos(), torch.cat((ang, ang), -1).sin()

    def rope(v):
        return v * cos + torch.cat((-v[..., D // 2:], v[..., :D // 2]), -1) * sin

    ahead = torch.ones(N, N, dtype=torch.bool, device="cuda").triu(1)
    with torch.no_grad():
        h = params["embed_tokens.weight"].double()[ids]
        for i in range(cfg.num_layers):
            p = {n[len(f"layers.{i}."):]: v.double() for n, v in params.items() if n.startswith(f"layers.{i}.")}
            x = _rms(h, p["input_layernorm.weight"])
            q = (x @ p["self_attn.q_proj.weight"].t()).view(B, N, heads, D).transpose(1, 2)
            k = (x @ p["self_attn.k_proj.weight"].t()).view(B, N, kvh, D).transpose(1, 2)
            v = (x @ p["self_attn.v_proj.weight"].t()).view(B, N, kvh, D).transpose(1, 2).contiguous()
            q, k = rope(_rms(q, p["self_attn.q_norm.weight"])), rope(_rms(k, p["self_attn.k_norm.weight"]))
            a = torch.empty(B, N, heads * D, dtype=torch.float64, device="cuda")
            for b in range(B):
                for j in range(heads):
                    c = j // (heads // kvh)
                    s = (q[b, j] @ k[b, c].t()) / math.sqrt(D)
                    a[b, :, j * D:(j + 1) * D] = s.masked_fill(ahead, -math.inf).softmax(-1) @ v[b, c]
            h = h + a @ p["self_attn.o_proj.weight"].t()
            w = {n: p["mlp." + n + (".weight" if n in _SHARED else "")] for n in _SHARED + _EXPERT}
            m = _rms(h, p["post_attention_layernorm.weight"]).reshape(B * N, -1)
            h = h + _mlp(m, ids.reshape(-1), tables[i], w).view(B, N, -1)
        T = case["prompt"]
        last = _rms(h[:, T - 1:], params["norm.weight"].double())
        return {"logits": last @ params["embed_tokens.weight"].double().t(), "hidden": h[:, :T].contiguous()}
