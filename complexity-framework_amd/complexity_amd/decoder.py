"""TR-GQA decoder around the TR-MoE layer: the harness of the 200M model.

The decoder is the reference's TR-GQA stack (ComplexityModel with
``attention_type="gqa"``, ``mlp_type="tr_hash_engine"``) at the released 200M
shape: 16 blocks of

    h = h + o_proj(SDPA(RoPE(qk_norm(q)), RoPE(qk_norm(k)), v))    block.py:205-268
    h = h + mlp(post_attention_layernorm(h), token_ids)             block.py:270-278

with RMSNorm (norms.py:46-55), fused KQV projection and GQA of 14 query over
2 key/value heads of width 64 (gqa.py:88-165, 169-218, SDPA at :229-266),
rotary embeddings over the absolute position (rotary.py:17-80, 239-295), a
final RMSNorm and the LM head tied to the embedding (builder.py:377-519).
The MLP half of every block is ``TRHashEngine.forward_norm_residual`` with
the route table of its layer index, i.e. the HIP kernels with the block's
RMSNorm and residual add fused in.

The reference's ``generate`` raises (builder.py:525-550), so the greedy loop
here is this build's own: ``prefill`` runs the prompt and fills a static KV
cache, ``decode_step`` appends one token per sequence, and ``generate``
replays a HIP-graph capture of the decode step (the position is a device
counter, so one capture serves every step).

On a GPU in bf16 the attention half runs on the HIP kernels too
(``ops.qk_norm_rope``, ``ops.prefill_attention``, ``ops.decode_attention``): a
prompt's q/k norm, rotation and cache writes are one pass over the projection,
its attention reads the caches, and a decode step of up to
16 sequences is three launches per block (norm + projection; q/k norm,
rotation, cache write and attention; output projection + residual).

Elsewhere, decode attention over the static cache: for one new token, GQA is the 14
query heads viewed as 2 groups of 7 rows, one group per key/value head
(head h uses key/value head h // 7, as ``repeat_interleave`` pairs them), so
SDPA runs on [B, 2, 7, 64] queries against the cache without copying it;
positions past the current one are masked.  The mask rules out the flash
kernel; SDPA's memory-efficient kernel takes it, and the math kernel is
never allowed (it would route bf16 batched products through a transposed
operand).
"""

from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Callable, Dict, List, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import ops
from .tr_hash import TRHashBackend, TRHashEngine, TRHashEngineConfig

try:   # torch >= 2.3
    from torch.nn.attention import SDPBackend, sdpa_kernel
except ImportError:  # pragma: no cover - the image ships torch 2.10
    SDPBackend = None
    sdpa_kernel = None


@dataclass(frozen=True)
class TRGQAConfig:
    """The released TR-HASH MoE 200M shape (docs/tr-hash-200m-release.md)."""

    vocab_size: int = 32000
    hidden_size: int = 896
    num_layers: int = 16
    num_heads: int = 14
    num_kv_heads: int = 2
    head_dim: int = 64
    shared_width: int = 3072
    num_experts: int = 4
    expert_width: int = 64
    top_k: int = 2
    route_hash_count: int = 2
    route_weights: tuple = (0.5, 0.5)
    shared_output_scale: float = 1.0
    routed_output_scale: float = 2.0
    norm_eps: float = 1e-6
    rope_theta: float = 10000.0
    max_position_embeddings: int = 2048
    initializer_range: float = 0.02

    @property
    def kv_groups(self) -> int:
        return self.num_heads // self.num_kv_heads


class RMSNorm(nn.Module):
    """x * rsqrt(mean(x^2) + eps) * weight in the input dtype (norms.py:47-56)."""

    def __init__(self, size: int, eps: float):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(size))
        self.eps = eps

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        variance = x.pow(2).mean(-1, keepdim=True)
        return self.weight * (x * torch.rsqrt(variance + self.eps))


def _rotate_half(x: torch.Tensor) -> torch.Tensor:
    h = x.shape[-1] // 2
    return torch.cat((-x[..., h:], x[..., :h]), dim=-1)


def rope_tables(head_dim: int, positions: int, theta: float):
    """cos/sin [positions, head_dim] in fp32 (rotary.py:41-56: emb = [freqs, freqs])."""
    inv_freq = 1.0 / (theta ** (torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim))
    t = torch.arange(positions, dtype=torch.float32)
    freqs = torch.outer(t, inv_freq)
    emb = torch.cat((freqs, freqs), dim=-1)
    return emb.cos(), emb.sin()


class GQAttention(nn.Module):
    """Grouped-query attention with QK RMSNorm and RoPE (gqa.py:43-165)."""

    def __init__(self, cfg: TRGQAConfig):
        super().__init__()
        self.cfg = cfg
        H, D = cfg.hidden_size, cfg.head_dim
        self.k_proj = nn.Linear(H, cfg.num_kv_heads * D, bias=False)
        self.q_proj = nn.Linear(H, cfg.num_heads * D, bias=False)
        self.v_proj = nn.Linear(H, cfg.num_kv_heads * D, bias=False)
        self.o_proj = nn.Linear(cfg.num_heads * D, H, bias=False)
        self.q_norm = RMSNorm(D, 1e-6)
        self.k_norm = RMSNorm(D, 1e-6)
        self.scale = 1.0 / math.sqrt(D)
        self._kqv: Optional[torch.Tensor] = None
        self._kqv_key = None

    def kqv_weight(self) -> torch.Tensor:
        """[k; q; v] rows of one fused projection (gqa.py:211-218), cached on
        the three weights' storage and version."""
        ws = (self.k_proj.weight, self.q_proj.weight, self.v_proj.weight)
        key = tuple((w.data_ptr(), w._version) for w in ws)
        if self._kqv is None or self._kqv_key != key:
            with torch.no_grad():
                self._kqv = torch.cat(ws, dim=0)
            self._kqv_key = key
        return self._kqv

    def project(self, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor):
        """q [B, 14, T, D], k/v [B, 2, T, D] after QK norm and RoPE; cos/sin
        [T, D] (or [B, T, D]) in x's dtype."""
        B, T, _ = x.shape
        cfg = self.cfg
        kqv = F.linear(x, self.kqv_weight())
        kd, qd = cfg.num_kv_heads * cfg.head_dim, cfg.num_heads * cfg.head_dim
        k, q, v = kqv.split([kd, qd, kd], dim=-1)
        q = q.view(B, T, cfg.num_heads, cfg.head_dim).transpose(1, 2)
        k = k.view(B, T, cfg.num_kv_heads, cfg.head_dim).transpose(1, 2)
        v = v.view(B, T, cfg.num_kv_heads, cfg.head_dim).transpose(1, 2)
        q, k = self.q_norm(q), self.k_norm(k)
        if cos.dim() == 2:
            cos, sin = cos[None, None], sin[None, None]
        else:
            cos, sin = cos[:, None], sin[:, None]
        q = q * cos + _rotate_half(q) * sin
        k = k * cos + _rotate_half(k) * sin
        return q, k, v

    def prefill_attention(self, q, k, v) -> torch.Tensor:
        """Causal SDPA over the prompt; each key/value head serves kv_groups
        query heads (gqa.py:150-152, 229-266).  The reduced-precision kernels
        take the grouped heads as they are, without a repeated copy."""
        g = self.cfg.kv_groups
        if q.device.type == "cuda" and q.dtype != torch.float32 and sdpa_kernel is not None:
            return _sdpa(q, k, v, None, causal=True, scale=self.scale, grouped=g > 1)
        k = k.repeat_interleave(g, dim=1)
        v = v.repeat_interleave(g, dim=1)
        return _sdpa(q, k, v, None, causal=True, scale=self.scale)

    def decode_attention(self, q, k_cache, v_cache, mask) -> torch.Tensor:
        """One new token per sequence: q [B, 14, 1, D] as [B, 2, 7, D] against
        the static cache [B, 2, L, D] with the position mask [1, 1, 1, L]."""
        B = q.shape[0]
        cfg = self.cfg
        qg = q.reshape(B, cfg.num_kv_heads, cfg.kv_groups, cfg.head_dim)
        out = _sdpa(qg, k_cache, v_cache, mask, causal=False, scale=self.scale)
        return out.reshape(B, cfg.num_heads, 1, cfg.head_dim)

    def output(self, attn: torch.Tensor) -> torch.Tensor:
        B, _, T, _ = attn.shape
        return self.o_proj(attn.transpose(1, 2).reshape(B, T, -1))


def _sdpa(q, k, v, mask, *, causal: bool, scale: float, grouped: bool = False) -> torch.Tensor:
    """SDPA on the flash / memory-efficient kernels for reduced precision (the
    math kernel raises instead of running); any kernel for fp32."""
    if q.dtype == torch.float32 or sdpa_kernel is None:
        return F.scaled_dot_product_attention(q, k, v, attn_mask=mask, is_causal=causal, scale=scale)
    with sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]):
        if grouped:
            return F.scaled_dot_product_attention(q, k, v, attn_mask=mask, is_causal=causal, scale=scale,
                                                  enable_gqa=True)
        return F.scaled_dot_product_attention(q, k, v, attn_mask=mask, is_causal=causal, scale=scale)


class TRGQABlock(nn.Module):
    def __init__(self, cfg: TRGQAConfig, layer_index: int, backend: str):
        super().__init__()
        self.input_layernorm = RMSNorm(cfg.hidden_size, cfg.norm_eps)
        self.self_attn = GQAttention(cfg)
        self.post_attention_layernorm = RMSNorm(cfg.hidden_size, cfg.norm_eps)
        self.mlp = TRHashEngine(TRHashEngineConfig(
            hidden_size=cfg.hidden_size, vocab_size=cfg.vocab_size, num_experts=cfg.num_experts,
            top_k=cfg.top_k, shared_width=cfg.shared_width, expert_width=cfg.expert_width,
            initializer_range=cfg.initializer_range, routing_strategy="token_id_multi_hash",
            layer_index=layer_index, route_hash_count=cfg.route_hash_count, route_weights=cfg.route_weights,
            shared_output_scale=cfg.shared_output_scale, routed_output_scale=cfg.routed_output_scale,
            attention_backbone="gqa", phase="inference", precision="bf16", backend=backend))
        self.layer_index = layer_index


def _plain(mod: nn.Module, cls: type, *shape: int) -> bool:
    """A module of exactly `cls` (so not parametrized or replaced) without
    hooks or bias, its weight in bf16, of `shape` and laid out as the kernels
    read it (contiguous, 16-byte aligned): what a kernel may stand in for."""
    if type(mod) is not cls or mod._forward_hooks or mod._forward_pre_hooks:
        return False
    w = mod._parameters.get("weight")
    return (w is not None and w.dtype is torch.bfloat16 and w.shape == shape and w.is_contiguous()
            and w.data_ptr() % 16 == 0 and mod._parameters.get("bias") is None)


def _values(t: torch.Tensor) -> bool:
    """A tensor whose memory a kernel may read in place of the torch
    operations: no function transform, forward-mode derivative or trace has to
    see them."""
    return (type(t) in (torch.Tensor, nn.Parameter) and torch.autograd.forward_ad._current_level < 0
            and torch._C._functorch.peek_interpreter_stack() is None and torch._C._len_torch_dispatch_stack() == 0
            and not torch.jit.is_tracing() and not torch.compiler.is_compiling())


def _pinned(block: nn.Module) -> bool:
    """A block whose engine is pinned to PYTORCH (a replaced MLP half is not)."""
    config = getattr(block._modules.get("mlp"), "config", None)
    return getattr(config, "backend", None) is TRHashBackend.PYTORCH


def _other_autocast() -> bool:
    """Autocast to another type than the kernels': the projections come out in it."""
    return torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") is not torch.bfloat16


class _StepPlan:
    """The layers of a decode step as one native call takes them
    (``trmoe_decoder_step``): the pointers of every block's weights, packs and
    caches, with what they were read from.  ``current`` looks at all of it
    again before each step: module, parameter and cache objects, in-place
    versions, storage, norm and attention constants, packs, routing, and what
    ``_hip_attention`` asks of a decoder.  Without the plan a step spends about
    100 us per layer in Python, against 30 us of kernels."""

    def __init__(self, cfg: "TRGQAConfig", device: torch.device):
        # nothing here refers back to the decoder: one that is let go gives its
        # memory back at once
        self.cfg, self.device = cfg, device
        self.dims = ops.N.DecoderDims()
        self.layers = None
        self.engines = []   # (engine, config, strategy, E, W, pack entry, route table)
        self.members = []   # (owner's dict, name, object)
        self.tensors = []   # (owner's dict, name, tensor, version, pointer)
        self.values = []    # (object's dict, name, value)
        self.caches = []    # (k or v, layer, tensor, pointer, shape)
        self.stands = []    # (module that a kernel stands in for, its class, weight, shape)
        self.attns = []
        self.keep = []      # what the pointers point into

    def _watch(self, owner: nn.Module, name: str) -> nn.Module:
        mod = owner._modules[name]
        self.members.append((owner._modules, name, mod))
        return mod

    def _weight(self, owner: nn.Module, name: str) -> torch.Tensor:
        t = owner._parameters[name]
        self.tensors.append((owner._parameters, name, t, t._version, t.data_ptr()))
        return t

    def _value(self, owner: nn.Module, name: str) -> float:
        v = getattr(owner, name)
        self.values.append((owner.__dict__, name, v))
        return v

    def _cache(self, dec: "TRGQADecoder", name: str, layer: int) -> torch.Tensor:
        t = getattr(dec, name)[layer]
        self.caches.append((name == "k_cache", layer, t, t.data_ptr(), t.shape))
        return t

    def _stand_in(self, mod: nn.Module) -> torch.Tensor:
        t = self._weight(mod, "weight")
        self.stands.append((mod, type(mod), t, t.shape))
        return t

    @classmethod
    def build(cls, dec: "TRGQADecoder", device: torch.device) -> Optional["_StepPlan"]:
        """None when a block needs the general path: a replaced MLP half,
        adapted or e4m3 weights, grouped experts, layers that differ in shape.
        For decoders that ``_hip_attention`` takes."""
        with ops.decode_copies_together():
            return cls._build(dec, device)

    @classmethod
    def _build(cls, dec: "TRGQADecoder", device: torch.device) -> Optional["_StepPlan"]:
        if dec.mlp_fn is not None or len(dec.k_cache) != len(dec.layers) or len(dec.v_cache) != len(dec.layers):
            return None
        cfg, rows, shapes = dec.cfg, [], set()
        plan = cls(cfg, device)
        plan._watch(dec, "layers")
        first = dec.k_cache[0] if dec.k_cache else None
        if first is not None and (first.ndim != 4 or first.shape[1::2] != (cfg.num_kv_heads, cfg.head_dim)):
            return None
        for i, (name, block) in enumerate(dec.layers._modules.items()):
            plan.members.append((dec.layers._modules, name, block))
            attn, mlp = plan._watch(block, "self_attn"), plan._watch(block, "mlp")
            plan.attns.append(attn)
            norm_in, norm_post = plan._watch(block, "input_layernorm"), plan._watch(block, "post_attention_layernorm")
            if not _plain(norm_post, RMSNorm, cfg.hidden_size) or type(mlp) is not TRHashEngine or mlp._fp8:
                return None
            for n in ("shared_gate", "shared_up", "shared_down"):
                mod = mlp._modules.get(n)
                plan.members.append((mlp._modules, n, mod))
                if mod is not None:
                    if type(mod) is not nn.Linear:
                        return None
                    plan._weight(mod, "weight")
            if any(n not in mlp._parameters for n in ("expert_gate", "expert_up", "expert_down")):
                return None   # parametrized
            for n in ("expert_gate", "expert_up", "expert_down"):
                plan._weight(mlp, n)
            decision = mlp._decide(plan._weight(norm_post, "weight"))
            if decision.selected is not TRHashBackend.HIP:
                return None
            packed = mlp._hip_packed(norm_post.weight)
            if packed.strategy != ops.STRATEGY_DENSE or packed.act_dtype is not torch.bfloat16:
                return None
            c, table = mlp.config, mlp._active_route_table
            if table.dtype is not torch.int64 or not table.is_contiguous():
                return None
            shapes.add((packed.shared_width, packed.num_experts, packed.expert_width, tuple(table.shape),
                        tuple(c.route_weights), c.shared_output_scale, c.routed_output_scale,
                        plan._value(norm_in, "eps"), plan._value(norm_post, "eps"), plan._value(attn.q_norm, "eps"),
                        plan._value(attn.k_norm, "eps"), plan._value(attn, "scale")))
            caches = plan._cache(dec, "k_cache", i), plan._cache(dec, "v_cache", i)
            for t in caches:
                if (t.dtype is not torch.bfloat16 or t.device != first.device or t.shape != first.shape
                        or not t.is_contiguous()):
                    return None
            for n in ("k_proj", "q_proj", "v_proj"):
                if "weight" not in plan._watch(attn, n)._parameters:
                    return None   # parametrized: kqv_weight() materialises it per call
                plan._weight(attn._modules[n], "weight")
            kqv = attn.kqv_weight()
            frags = packed.fragments("dense_gate_up", cfg.hidden_size), packed.fragments("dense_down",
                                                                                         packed.dense_features)
            if None in frags:
                return None   # a graph records, and nothing has built them before
            gu, dn = frags[0][0], frags[1][0]
            ptrs = (plan._stand_in(norm_in), kqv, *(plan._stand_in(plan._watch(attn, n))
                                                   for n in ("q_norm", "k_norm", "o_proj")), *caches, gu, dn, table)
            if any(t.data_ptr() % 16 for t in ptrs) or kqv.dtype is not torch.bfloat16:
                return None
            plan.keep.append(ptrs)
            rows.append(ops.N.DecoderLayer(*(t.data_ptr() for t in ptrs)))
            plan.engines.append((mlp, c, mlp.routed_strategy, mlp._active_num_experts, mlp._active_expert_width,
                                 mlp._packed_norm, table))
            mlp.last_backend, mlp.last_norm = decision, "fused"
        if len(shapes) != 1:
            return None
        S, E, W, (top_k, vocab), rw, ss, rs, e_in, e_post, e_q, e_k, scale = shapes.pop()
        if e_in != e_post or e_q != e_k or e_in <= 0.0:
            return None
        d = plan.dims
        d.layers, d.hidden, d.cache_length, d.vocab_size = len(rows), cfg.hidden_size, dec.k_cache[0].shape[2], vocab
        d.shared_width, d.expert_width, d.num_experts, d.top_k = S, W, E, top_k
        d.num_heads, d.num_kv_heads = cfg.num_heads, cfg.num_kv_heads
        d.norm_eps, d.qk_eps, d.attn_scale, d.shared_scale, d.routed_scale = e_in, e_q, scale, ss, rs
        d.route_weights[:] = (list(rw) + [0.0] * 4)[:4]
        d.cache_batch = dec.k_cache[0].shape[0]
        plan.layers = (ops.N.DecoderLayer * len(rows))(*rows)
        return plan

    def current(self, dec: "TRGQADecoder", device: torch.device) -> bool:
        if (dec.mlp_fn is not None or len(dec.layers) != len(self.engines) or device != self.device
                or dec.cfg is not self.cfg or dec.embed_tokens.weight.dtype is not torch.bfloat16 or _other_autocast()):
            return False
        for eng, cfg, strategy, E, W, entry, table in self.engines:
            if (eng._packed_norm is not entry or eng.config is not cfg or eng.routed_strategy != strategy
                    or eng._active_num_experts != E or eng._active_expert_width != W
                    or eng._active_route_table is not table or eng._fp8):
                return False
        k, v, n = dec.k_cache, dec.v_cache, len(self.engines)
        if len(k) != n or len(v) != n:
            return False
        for is_k, i, t, p, shape in self.caches:
            if (k if is_k else v)[i] is not t or t.data_ptr() != p or t.shape != shape:
                return False
        bf16 = torch.bfloat16
        for mod, cls, t, shape in self.stands:
            if (type(mod) is not cls or mod._forward_hooks or mod._forward_pre_hooks or t.dtype is not bf16
                    or t.shape != shape or not t.is_contiguous() or mod._parameters.get("bias") is not None):
                return False
        for attn in self.attns:
            if type(attn) is not GQAttention:
                return False
        for d, n, m in self.members:
            if d.get(n) is not m:
                return False
        for d, n, t, v, p in self.tensors:
            if d.get(n) is not t or t._version != v or t.data_ptr() != p:
                return False
        return all(d.get(n) == x for d, n, x in self.values)


# Replaces a block's MLP half (tests compare against a decoder whose MLPs run
# another definition): (layer index, h [B, T, H], token ids [B, T], block)
# -> h + mlp(post_attention_layernorm(h)).
MLPFn = Callable[[int, torch.Tensor, torch.Tensor, TRGQABlock], torch.Tensor]


class TRGQADecoder(nn.Module):
    """16-layer TR-GQA decoder with a static KV cache and a greedy loop."""

    def __init__(self, cfg: TRGQAConfig = TRGQAConfig(), backend: str = "auto", mlp_fn: Optional[MLPFn] = None):
        super().__init__()
        self.cfg = cfg
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size)
        self.layers = nn.ModuleList(TRGQABlock(cfg, i, backend) for i in range(cfg.num_layers))
        self.norm = RMSNorm(cfg.hidden_size, cfg.norm_eps)
        self.mlp_fn = mlp_fn
        self.k_cache: List[torch.Tensor] = []
        self.v_cache: List[torch.Tensor] = []
        self.cache_len = 0
        self._pos: Optional[torch.Tensor] = None   # device int64 [1]: next decode position
        self._rope = None
        self._rope32 = None
        self._step_plan: Optional[_StepPlan] = None
        self._graph = None

    def __getstate__(self):
        # a copy builds a plan of its own: this one points at this module's
        # weights and caches
        return {**self.__dict__, "_step_plan": None}

    # ------------------------------------------------------------------ weights
    @torch.no_grad()
    def init_weights(self, seed: int = 0) -> "TRGQADecoder":
        """Seeded GPT-style init (builder.py:177-232): N(0, 0.02) for linears,
        expert tensors and the embedding; o_proj and the MLP down projections
        N(0, 0.02 / sqrt(2 * layers)); norm weights one.  Drawn on the CPU in
        parameter order, so every device and dtype sees the same values."""
        g = torch.Generator().manual_seed(seed)
        std = self.cfg.initializer_range
        residual_std = std / math.sqrt(2 * self.cfg.num_layers)
        for name, p in self.named_parameters():
            if name.endswith("layernorm.weight") or name.endswith("norm.weight"):
                p.fill_(1.0)
                continue
            s = residual_std if (name.endswith("o_proj.weight") or name.endswith("expert_down")
                                 or name.endswith("shared_down.weight")) else std
            p.copy_((torch.randn(p.shape, generator=g, dtype=torch.float32) * s).to(p.dtype))
        return self

    # ------------------------------------------------------------------ pieces
    def _mlp(self, block: TRGQABlock, h: torch.Tensor, ids: torch.Tensor) -> torch.Tensor:
        if self.mlp_fn is not None:
            return self.mlp_fn(block.layer_index, h, ids, block)
        norm = block.post_attention_layernorm
        return block.mlp.forward_norm_residual(h, ids, norm.weight, norm.eps)

    def _rope_tables(self, positions: int, device, dtype):
        if self._rope is None or self._rope[0].shape[0] < positions or self._rope[0].device != device \
                or self._rope[0].dtype != dtype:
            n = max(positions, self.cfg.max_position_embeddings)
            cos, sin = rope_tables(self.cfg.head_dim, n, self.cfg.rope_theta)
            self._rope = (cos.to(device=device, dtype=dtype), sin.to(device=device, dtype=dtype))
        return self._rope

    def _rope_tables32(self, positions: int, device):
        """fp32 cos / sin for the HIP attention kernels."""
        if self._rope32 is None or self._rope32[0].shape[0] < positions or self._rope32[0].device != device:
            cos, sin = rope_tables(self.cfg.head_dim, max(positions, self.cfg.max_position_embeddings),
                                   self.cfg.rope_theta)
            self._rope32 = (cos.to(device), sin.to(device))
        return self._rope32

    def _hip_attention(self, device: torch.device) -> bool:
        """Whether the attention half runs on the HIP kernels: bf16 on a GPU,
        dimensions they take, a decoder that is not pinned to PYTORCH, and
        modules as built here (a replaced, adapted or hooked one is called)."""
        cfg = self.cfg
        if (device.type != "cuda" or self.embed_tokens.weight.dtype is not torch.bfloat16
                or ops.attention_unsupported(cfg.hidden_size, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim)):
            return False
        if _other_autocast():
            return False
        for block in self.layers:
            m = block._modules
            attn = m["self_attn"]
            if type(attn) is not GQAttention or _pinned(block):
                return False
            a = attn._modules
            H, D = cfg.hidden_size, cfg.head_dim
            if not (_plain(m["input_layernorm"], RMSNorm, H) and _plain(a["q_norm"], RMSNorm, D)
                    and _plain(a["k_norm"], RMSNorm, D) and _plain(a["o_proj"], nn.Linear, H, cfg.num_heads * D)):
                return False
            # the kernels norm q and k with one eps, and take a positive scale
            if a["q_norm"].eps != a["k_norm"].eps or not attn.scale > 0:
                return False
        return True

    def _norm(self, norm: RMSNorm, h: torch.Tensor, hip: bool) -> torch.Tensor:
        if not hip:
            return norm(h)
        return ops.rmsnorm_forward(h.reshape(-1, h.shape[-1]), norm.weight, norm.eps)[0].view(h.shape)

    def _hip_norm(self, norm: RMSNorm, h: torch.Tensor) -> bool:
        """Whether a GPU's h goes through `norm` on the RMSNorm kernel."""
        return (_values(h) and not torch.is_grad_enabled() and h.dtype is torch.bfloat16 and _plain(norm, RMSNorm, h.shape[-1])
                and ops.rmsnorm_unsupported(h, norm.weight) is None
                and not any(_pinned(b) for b in list(self.layers._modules.values())[:1]))

    def logits(self, h: torch.Tensor) -> torch.Tensor:
        hip = h.device.type == "cuda" and self._hip_norm(self.norm, h)
        return F.linear(self._norm(self.norm, h, hip), self.embed_tokens.weight)

    # ------------------------------------------------------------------ prompt
    @torch.no_grad()
    def prefill(self, input_ids: torch.Tensor, max_new_tokens: int = 0, return_logits: bool = True,
                timings: Optional[Dict[str, list]] = None):
        """Runs the prompt [B, T], allocates the static KV cache for
        T + max_new_tokens positions and fills its first T; returns the logits
        [B, T, V] (or the last hidden state when return_logits is False).
        timings: lists of (start, end) CUDA events per layer under "attention"
        and "mlp"."""
        B, T = input_ids.shape
        cfg = self.cfg
        dev = input_ids.device
        dt = self.embed_tokens.weight.dtype
        # static cache rounded to 64 positions (the masked decode kernel wants
        # an aligned mask row; positions past the current one are masked)
        L = (T + max_new_tokens + 63) // 64 * 64
        self.k_cache = [torch.empty(B, cfg.num_kv_heads, L, cfg.head_dim, device=dev, dtype=dt)
                        for _ in self.layers]
        self.v_cache = [torch.empty_like(c) for c in self.k_cache]
        if L > T:   # the prompt fills the rest
            for c in self.k_cache + self.v_cache:
                c[:, :, T:].zero_()
        self.cache_len = T
        self._graph = None
        self._step_plan = None
        hip = self._hip_attention(dev)
        if hip:
            cos, sin = self._rope_tables32(L, dev)
        else:
            cos, sin = self._rope_tables(L, dev, dt)
            cos, sin = cos[:T], sin[:T]
        h = self.embed_tokens(input_ids)
        for i, block in enumerate(self.layers):
            ev = _events(timings, "attention")
            attn = block.self_attn
            x = self._norm(block.input_layernorm, h, hip)
            if hip:
                q = ops.qk_norm_rope(F.linear(x, attn.kqv_weight()).view(B * T, -1), B, cfg.num_heads,
                                     attn.q_norm.weight, attn.k_norm.weight, attn.q_norm.eps, cos, sin,
                                     self.k_cache[i], self.v_cache[i])
                h = h + attn.o_proj(ops.prefill_attention(q, self.k_cache[i], self.v_cache[i], attn.scale))
            else:
                q, k, v = attn.project(x, cos, sin)
                self.k_cache[i][:, :, :T].copy_(k)
                self.v_cache[i][:, :, :T].copy_(v)
                h = h + attn.output(attn.prefill_attention(q, k, v))
            _end(ev)
            ev = _events(timings, "mlp")
            h = self._mlp(block, h, input_ids)
            _end(ev)
        self._pos = torch.full((1,), T, dtype=torch.int64, device=dev)
        return self.logits(h) if return_logits else h

    # ------------------------------------------------------------------ decode
    def _decode_body(self, ids: torch.Tensor) -> torch.Tensor:
        """One token per sequence at device position self._pos (ids [B]);
        returns logits [B, V].  Graph-capturable: no host reads."""
        cfg = self.cfg
        B = ids.shape[0]
        if B != self.k_cache[0].shape[0]:   # the caches' rows are the batch's sequences
            raise RuntimeError(f"decode of {B} sequences over a KV cache of {self.k_cache[0].shape[0]}")
        L = self.k_cache[0].shape[2]
        dt = self.embed_tokens.weight.dtype
        pos = self._pos
        if self._step_plan is not None and not self._step_plan.current(self, ids.device):
            self._step_plan = None
        if B <= ops.DECODE_ATTN_MAX_BATCH and (self._step_plan is not None or self._hip_attention(ids.device)):
            return self._decode_body_hip(ids, pos, L)
        cos_t, sin_t = self._rope_tables(L, ids.device, dt)
        cos = cos_t.index_select(0, pos)           # [1, D]
        sin = sin_t.index_select(0, pos)
        span = torch.arange(L, device=ids.device)
        mask = torch.where(span <= pos, 0.0, -1e9).to(dt).view(1, 1, 1, L)
        tok = ids.view(B, 1)
        h = self.embed_tokens(tok)
        for i, block in enumerate(self.layers):
            x = block.input_layernorm(h)
            q, k, v = block.self_attn.project(x, cos, sin)
            self.k_cache[i].index_copy_(2, pos, k)
            self.v_cache[i].index_copy_(2, pos, v)
            attn = block.self_attn.decode_attention(q, self.k_cache[i], self.v_cache[i], mask)
            h = h + block.self_attn.output(attn)
            h = self._mlp(block, h, tok)
        return self.logits(h).view(B, -1)

    def _decode_body_hip(self, ids: torch.Tensor, pos: torch.Tensor, L: int) -> torch.Tensor:
        cfg = self.cfg
        B = ids.shape[0]
        cos, sin = self._rope_tables32(L, ids.device)
        tok = ids.view(B, 1)
        h = self.embed_tokens(tok).view(B, -1)
        if self._step_plan is None:
            self._step_plan = _StepPlan.build(self, ids.device)
        if self._step_plan is not None and h.is_contiguous():
            ids = tok.view(B).to(torch.int64).contiguous()
            ops.decoder_step(h, self._step_plan.dims, self._step_plan.layers, ids, pos, cos, sin)
            return self.logits(h)
        for i, block in enumerate(self.layers):
            attn, norm = block.self_attn, block.input_layernorm
            a = ops.decode_attention(h, norm.weight, norm.eps, attn.kqv_weight(), cfg.num_heads, attn.q_norm.weight,
                                     attn.k_norm.weight, attn.q_norm.eps, cos, sin, pos, self.k_cache[i],
                                     self.v_cache[i], attn.scale)
            h = ops.decode_linear(a, attn.o_proj.weight, h)
            h = self._mlp(block, h.view(B, 1, -1), tok).view(B, -1)
        return self.logits(h)

    @torch.no_grad()
    def decode_step(self, ids: torch.Tensor) -> torch.Tensor:
        """Eager decode of one token per sequence; advances the position."""
        if self.cache_len >= self.k_cache[0].shape[2]:
            raise RuntimeError("KV cache full: prefill with a larger max_new_tokens")
        out = self._decode_body(ids)
        self._pos.add_(1)
        self.cache_len += 1
        return out

    @torch.no_grad()
    def capture_decode(self, batch: int):
        """Captures one greedy decode step in a HIP graph: static ids in,
        argmax ids out (written back as the next step's input), position
        advanced on the device.  Warm-up runs happen on a copy of the cache
        state and are undone."""
        dev = self.embed_tokens.weight.device
        self._g_ids = torch.zeros(batch, dtype=torch.int64, device=dev)
        self._g_logits = None
        saved_pos = self._pos.clone()
        saved = [(k.clone(), v.clone()) for k, v in zip(self.k_cache, self.v_cache)]
        # the graph owns the scratch its launches were recorded with
        self._g_scratch = ops.workspace_scope()
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with self._g_scratch, torch.cuda.stream(stream):
            for _ in range(2):   # builds every lazy pack before capture
                self._graph_step()
                self._pos.copy_(saved_pos)
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with self._g_scratch, torch.cuda.graph(graph):
            self._graph_step()
        self._pos.copy_(saved_pos)
        for (k, v), (k0, v0) in zip(zip(self.k_cache, self.v_cache), saved):
            k.copy_(k0)
            v.copy_(v0)
        self._graph = graph
        return graph

    def _graph_step(self):
        logits = self._decode_body(self._g_ids)
        self._g_logits = logits
        self._g_ids.copy_(logits.argmax(dim=-1))
        self._pos.add_(1)

    @torch.no_grad()
    def generate(self, input_ids: torch.Tensor, steps: int, use_graph: bool = True) -> torch.Tensor:
        """Greedy continuation of the prompt [B, T]: the prompt's next token
        then `steps` decode steps of one token per sequence -> [B, steps + 1]."""
        h = self.prefill(input_ids, steps + 1, return_logits=False)
        first = self.logits(h[:, -1:]).argmax(dim=-1).view(-1)
        return self.continue_greedy(first, steps, use_graph)

    @torch.no_grad()
    def continue_greedy(self, first: torch.Tensor, steps: int, use_graph: bool = True) -> torch.Tensor:
        """`steps` greedy decode steps after prefill, starting from the token
        `first` [B]; returns [B, steps + 1] (first included)."""
        B = first.shape[0]
        out = torch.empty(B, steps + 1, dtype=torch.int64, device=first.device)
        out[:, 0] = first
        if self.cache_len + steps > self.k_cache[0].shape[2]:
            raise RuntimeError("KV cache too small: prefill with a larger max_new_tokens")
        if use_graph:
            if self._graph is None:
                self.capture_decode(B)
            self._g_ids.copy_(first)
            for s in range(1, steps + 1):
                self._graph.replay()
                out[:, s] = self._g_ids
            self.cache_len += steps
            return out
        ids = first
        for s in range(1, steps + 1):
            ids = self.decode_step(ids).argmax(dim=-1)
            out[:, s] = ids
        return out


def _events(timings, key):
    if timings is None:
        return None
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    timings.setdefault(key, []).append((s, e))
    return e


def _end(ev):
    if ev is not None:
        ev.record()
