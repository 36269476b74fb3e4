"""The host side of the decode step's native call on the CPU: the kernels'
entry points are replaced by recorders, so that what a step hands to them, and
what it refuses, can be looked at without a device."""

import copy
import ctypes
import dataclasses
import gc
import io
import pickle
import weakref
from types import SimpleNamespace

import pytest
import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.functional as F
from torch.fx.experimental.proxy_tensor import make_fx

from complexity_amd import _native, ops
from complexity_amd import decoder as dec
from complexity_amd.decoder import TRGQAConfig, TRGQADecoder
from complexity_amd.tr_hash import TRHashBackend, TRHashEngine

CFG = TRGQAConfig(vocab_size=64, hidden_size=64, num_layers=2, num_heads=2, num_kv_heads=1, shared_width=64,
                  num_experts=4, expert_width=8, max_position_embeddings=64)
IDS = torch.arange(2 * 6).view(2, 6)


class _Pack(SimpleNamespace):
    def fragments(self, name, cols):
        return self.frag, cols


def _fake_pack(self, norm_weight=None, current=None):
    if self._packed_norm is None:
        self._packed_norm = ("key", _Pack(
            strategy=ops.STRATEGY_DENSE, act_dtype=torch.bfloat16, shared_width=64, num_experts=4, expert_width=8,
            dense_features=128, frag=torch.zeros(64, dtype=torch.uint8)))
    return self._packed_norm[1]


@pytest.fixture()
def model(monkeypatch):
    """A decoder after a prompt of two sequences whose steps go to recorders
    (`model.calls`: one (name, arguments) per kernel call)."""
    torch.manual_seed(0)
    m = TRGQADecoder(CFG, backend="pytorch").to(torch.bfloat16).init_weights(1).eval()
    m.prefill(IDS, max_new_tokens=8)
    m.calls = []
    monkeypatch.setattr(TRGQADecoder, "_hip_attention", lambda self, device: True)
    monkeypatch.setattr(TRHashEngine, "_decide", lambda self, h: SimpleNamespace(selected=TRHashBackend.HIP))
    monkeypatch.setattr(TRHashEngine, "_hip_packed", _fake_pack)
    monkeypatch.setattr(TRGQADecoder, "_mlp", lambda self, block, h, ids: h)
    monkeypatch.setattr(ops, "decoder_step", lambda *a: m.calls.append(("step", a)))

    def attention(x, *a):
        m.calls.append(("attention", (x, *a)))
        return torch.zeros(x.shape[0], CFG.num_heads * 64, dtype=x.dtype)

    monkeypatch.setattr(ops, "decode_attention", attention)
    monkeypatch.setattr(ops, "decode_linear", lambda a, w, h: h)
    return m


def _names(m):
    return [n for n, _ in m.calls]


def test_step_goes_to_one_call(model):
    model.decode_step(IDS[:, 0])
    assert _names(model) == ["step"]
    h, dims, layers = model.calls[0][1][:3]
    assert h.shape == (2, 64) and dims.cache_batch == 2 and len(layers) == 2
    assert [l.k_cache for l in layers] == [c.data_ptr() for c in model.k_cache]


@pytest.mark.parametrize("blocks", [False, True])
@pytest.mark.parametrize("ids", [IDS[:, :1], IDS[:, 0].int(), IDS[:, :1].int(), IDS.t()[0]],
                         ids=["column", "int32", "int32_column", "strided"])
def test_forms_of_the_token_ids(model, ids, blocks):
    if blocks:
        model.mlp_fn = lambda i, h, tok, block: h
    out = model.decode_step(ids)
    assert out.shape == (2, CFG.vocab_size)
    want = F.embedding(IDS[:, 0], model.embed_tokens.weight)
    for name, a in model.calls:
        assert torch.equal(a[0], want)
        if name == "step":
            assert a[3].dtype == torch.int64 and a[3].is_contiguous() and torch.equal(a[3], IDS[:, 0])


@pytest.mark.parametrize("batch", [1, 3, 5, 16])
def test_other_batch_than_the_caches_is_refused(model, batch):
    with pytest.raises(RuntimeError):
        model.decode_step(torch.zeros(batch, dtype=torch.int64))
    assert model.calls == [] and model.cache_len == 6


def _caches(m):
    m.k_cache = [c.clone() for c in m.k_cache]


def _longer_caches(m):
    m.k_cache = [torch.cat((c, c), 2) for c in m.k_cache]
    m.v_cache = [torch.cat((c, c), 2) for c in m.v_cache]


def _one_cache(m):
    m.v_cache[1] = m.v_cache[1].clone()


def _cache_storage(m):
    m.v_cache[0].set_(m.v_cache[0].clone())


def _scale(m):
    for b in m.layers:
        b.self_attn.scale = 0.25


def _eps(m):
    for b in m.layers:
        b.input_layernorm.eps = b.post_attention_layernorm.eps = 1e-3


def _qk_eps(m):
    for b in m.layers:
        b.self_attn.q_norm.eps = b.self_attn.k_norm.eps = 1e-4


@pytest.mark.parametrize("change", [_caches, _longer_caches, _one_cache, _cache_storage, _scale, _eps, _qk_eps])
def test_changes_between_steps_are_seen(model, change):
    model.decode_step(IDS[:, 0])
    plan = model._step_plan
    model.decode_step(IDS[:, 0])
    assert model._step_plan is plan   # nothing changed: the same plan again
    change(model)
    model.decode_step(IDS[:, 1])
    assert _names(model) == ["step"] * 3
    dims, layers = model.calls[2][1][1:3]
    assert [l.k_cache for l in layers] == [c.data_ptr() for c in model.k_cache]
    assert [l.v_cache for l in layers] == [c.data_ptr() for c in model.v_cache]
    b = model.layers[0]
    got = (dims.cache_length, dims.norm_eps, dims.qk_eps, dims.attn_scale)
    assert got == pytest.approx((model.k_cache[0].shape[2], b.input_layernorm.eps, b.self_attn.q_norm.eps,
                                 b.self_attn.scale))


class _OtherLinear(torch.nn.Linear):
    pass


class _OtherAttention(dec.GQAttention):
    pass


def _attn(m):
    return m.layers[1].self_attn


def test_a_decoder_let_go_after_a_step_is_gone(model):
    m = copy.copy(model)
    m.__dict__ = dict(model.__dict__)
    m.decode_step(IDS[:, 0])
    assert m._step_plan is not None and model._step_plan is None
    gone = weakref.ref(m._step_plan)   # lives as long as the decoder's attributes
    gc.collect()
    gc.disable()
    try:
        del m
        assert gone() is None   # no cycle that only the collector would find
    finally:
        gc.enable()


def test_another_configuration_is_seen(model, monkeypatch):
    model.decode_step(IDS[:, 0])
    monkeypatch.setattr(TRGQADecoder, "_hip_attention", _ask)
    model.cfg = dataclasses.replace(CFG, vocab_size=32)
    with pytest.raises(_Asked):
        model.decode_step(IDS[:, 1])


class _Asked(Exception):
    pass


def _ask(self, device):
    raise _Asked


@pytest.mark.parametrize("change", [
    lambda m: _attn(m).q_norm.register_forward_hook(lambda *a: None),
    lambda m: m.layers[0].input_layernorm.register_forward_pre_hook(lambda *a: None),
    lambda m: setattr(_attn(m).o_proj, "bias", torch.nn.Parameter(torch.zeros(64, dtype=torch.bfloat16))),
    lambda m: setattr(_attn(m).o_proj, "__class__", _OtherLinear),
    lambda m: setattr(_attn(m), "__class__", _OtherAttention),
    lambda m: setattr(_attn(m).o_proj.weight, "data", _attn(m).o_proj.weight.data.view(128, 64).t()),
    lambda m: setattr(_attn(m).k_norm.weight, "data", _attn(m).k_norm.weight.data[:32]),
    lambda m: m.embed_tokens.float(),
    lambda m: setattr(m._step_plan, "device", torch.device("meta")),
], ids=["hook", "pre_hook", "bias", "class", "attention_class", "strided", "narrowed", "embedding", "device"])
def test_a_plan_stands_for_what_the_kernels_take(model, monkeypatch, change):
    """A current plan is taken without asking ``_hip_attention`` again, which
    is asked as soon as anything that it looks at has changed."""
    model.decode_step(IDS[:, 0])
    monkeypatch.setattr(TRGQADecoder, "_hip_attention", _ask)
    model.decode_step(IDS[:, 1])
    assert _names(model) == ["step"] * 2
    change(model)
    with pytest.raises(_Asked):
        model.decode_step(IDS[:, 2])
    assert _names(model) == ["step"] * 2 and model._step_plan is None


def test_autocast_drops_the_plan(model, monkeypatch):
    model.decode_step(IDS[:, 0])
    monkeypatch.setattr(TRGQADecoder, "_hip_attention", _ask)
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda device: True)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda device: torch.float16)
    with pytest.raises(_Asked):
        model.decode_step(IDS[:, 1])


def test_unequal_caches_take_the_blocks(model):
    model.decode_step(IDS[:, 0])
    model.k_cache[1] = torch.cat((model.k_cache[1], model.k_cache[1]), 2)
    model.decode_step(IDS[:, 1])
    assert _names(model) == ["step"] + ["attention"] * 2


class _Twice(torch.nn.Module):
    def forward(self, w):
        return w * 2


@pytest.mark.parametrize("name", ["q_proj", "k_proj", "v_proj"])
def test_parametrized_projection_takes_the_blocks(model, name):
    attn = model.layers[1].self_attn
    torch.nn.utils.parametrize.register_parametrization(getattr(attn, name), "weight", _Twice())
    model.decode_step(IDS[:, 0])
    assert _names(model) == ["attention"] * 2
    kqv = model.calls[1][1][3]
    assert torch.equal(kqv, torch.cat([getattr(attn, n).weight for n in ("k_proj", "q_proj", "v_proj")]))


def test_parametrization_between_steps_is_seen(model):
    model.decode_step(IDS[:, 0])
    attn = model.layers[0].self_attn
    torch.nn.utils.parametrize.register_parametrization(attn.q_proj, "weight", _Twice())
    model.decode_step(IDS[:, 1])
    torch.nn.utils.parametrize.remove_parametrizations(attn.q_proj, "weight", leave_parametrized=True)
    model.decode_step(IDS[:, 2])
    assert _names(model) == ["step"] + ["attention"] * 2 + ["step"]


@pytest.mark.parametrize("how", ["deepcopy", "pickle", "save"])
def test_copies_do_not_take_the_plan_along(model, how):
    model.decode_step(IDS[:, 0])
    assert model._step_plan is not None
    calls, model.calls = model.calls, []
    if how == "deepcopy":
        other = copy.deepcopy(model)
    else:
        f = io.BytesIO()
        if how == "pickle":
            pickle.dump(model, f)
            f.seek(0)
            other = pickle.load(f)   # written just above
        else:
            torch.save(model, f)
            f.seek(0)
            other = torch.load(f, weights_only=False)
    assert model._step_plan is not None and other._step_plan is None
    model.calls = calls
    for m in (other, model):
        m.decode_step(IDS[:, 1])
        layers = calls[-1][1][2]
        assert [l.k_cache for l in layers] == [c.data_ptr() for c in m.k_cache]
    assert _names(model) == ["step"] * 3


def test_native_step_refuses_another_batch():
    lib = _native.load()
    d = _native.DecoderDims()
    d.layers, d.hidden, d.cache_length, d.vocab_size, d.shared_width, d.expert_width = 1, 64, 64, 64, 64, 8
    d.num_heads, d.num_kv_heads, d.num_experts, d.top_k, d.cache_batch = 2, 1, 4, 2, 2
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.c_void_p((ctypes.addressof(buf) + 255) // 256 * 256)
    layer = (_native.DecoderLayer * 1)()
    nbytes = lib.trmoe_decoder_step_workspace_bytes(ctypes.byref(d), 5)
    assert nbytes > 0
    st = lib.trmoe_decoder_step(ctypes.byref(d), ctypes.cast(layer, ctypes.c_void_p), p, 5, p, p, p, p, 64, p, nbytes, None)
    assert st == _native.ERR_INVALID and b"batch" in lib.trmoe_last_error()


# ---------------------------------------------------------------------------
# which decoders the HIP attention half takes (looks at modules only)
# ---------------------------------------------------------------------------
CUDA = torch.device("cuda:0")


def _decoder(cfg=CFG, **kw):
    return TRGQADecoder(cfg, **kw).to(torch.bfloat16).eval()


def test_attention_takes_the_decoder_as_built():
    assert _decoder()._hip_attention(CUDA)


def test_unequal_q_and_k_eps_take_the_general_path():
    """The kernels norm q and k with one eps."""
    m = _decoder()
    m.layers[1].self_attn.k_norm.eps = 1e-2
    assert not m._hip_attention(CUDA)
    m.layers[1].self_attn.q_norm.eps = 1e-2
    assert m._hip_attention(CUDA)


def test_replaced_mlps_need_no_engine():
    """A replaced MLP half is only called: it has no engine's configuration."""
    m = _decoder()
    for b in m.layers:
        b.mlp = torch.nn.Identity()
    assert m._hip_attention(CUDA)
    assert not _decoder(backend="pytorch")._hip_attention(CUDA)


@pytest.mark.parametrize("what", ["identity", "no_layers"])
def test_logits_without_engines(what):
    m = _decoder(TRGQAConfig(vocab_size=64, hidden_size=64, num_layers=0) if what == "no_layers" else CFG)
    for b in m.layers:
        b.mlp = torch.nn.Identity()
    with torch.no_grad():
        assert m._hip_norm(m.norm, torch.zeros(2, 64, dtype=torch.bfloat16))
        pinned = _decoder(backend="pytorch")
        assert not pinned._hip_norm(pinned.norm, torch.zeros(2, 64, dtype=torch.bfloat16))


def _misaligned(p):
    flat = torch.zeros(p.numel() + 8, dtype=p.dtype)
    return torch.nn.Parameter(flat[1:1 + p.numel()].view_as(p))


def _misaligned_o(m):
    m.layers[1].self_attn.o_proj.weight = _misaligned(m.layers[1].self_attn.o_proj.weight)


def _one_q(m):
    m.layers[0].self_attn.q_norm.weight = torch.nn.Parameter(torch.ones(1, dtype=torch.bfloat16))


def _one_in(m):
    m.layers[0].input_layernorm.weight = torch.nn.Parameter(torch.ones(1, dtype=torch.bfloat16))


@pytest.mark.parametrize("change", [_misaligned_o, _one_q, _one_in])
def test_weights_the_kernels_cannot_read_take_the_general_path(change):
    """Kernels read 16 bytes at a time, and whole rows of norm weights."""
    m = _decoder()
    change(m)
    assert not m._hip_attention(CUDA)


def test_logits_norm_weight_of_one_value():
    m = _decoder()
    h = torch.zeros(2, 64, dtype=torch.bfloat16)
    with torch.no_grad():
        assert m._hip_norm(m.norm, h)
        m.norm.weight = torch.nn.Parameter(torch.ones(1, dtype=torch.bfloat16))
        assert not m._hip_norm(m.norm, h)


@pytest.mark.parametrize("dtype,takes", [(torch.float16, False), (torch.bfloat16, True)])
def test_autocast_to_another_type_takes_the_general_path(monkeypatch, dtype, takes):
    """Under autocast to fp16 the projections come out in fp16."""
    m = _decoder()
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda device_type="cuda": True)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda device_type: dtype)
    assert m._hip_attention(CUDA) is takes


def test_logits_under_function_transforms():
    """vmap, forward-mode derivatives and traces see the torch operations."""
    m = _decoder()
    h = torch.randn(3, 2, 64, generator=torch.Generator().manual_seed(0)).bfloat16()
    seen = []

    def look(x):
        seen.append(m._hip_norm(m.norm, x))
        return x

    with torch.no_grad():
        look(h)
        torch.func.vmap(look)(h)
        with fwAD.dual_level():
            look(fwAD.make_dual(h, h))
        with torch._subclasses.FakeTensorMode() as mode:
            look(mode.from_tensor(h))
        make_fx(look)(h)
    assert seen == [True, False, False, False, False]


@pytest.mark.parametrize("name", ["qk_norm_rope", "prefill_attention", "decode_attention", "decode_linear",
                                  "decoder_step", "rmsnorm_forward", "layer_forward"])
def test_calls_of_the_decoder_run_on_their_tensors_device(name):
    """The library launches on the current device: what the decoder calls by
    itself makes the tensors' GPU current."""
    assert hasattr(getattr(ops, name), "__wrapped__")


@pytest.mark.parametrize("scale,takes", [(0.0, False), (-0.125, False), (0.25, True)])
def test_attention_scale_that_is_not_positive_takes_the_general_path(scale, takes):
    m = _decoder()
    m.layers[1].self_attn.scale = scale
    assert m._hip_attention(CUDA) is takes
