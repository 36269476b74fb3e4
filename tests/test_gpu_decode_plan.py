"""The native decode step against the per-block path (the same kernels, block
by block): bit-identical logits, and every change a user can make between two
steps is picked up: in-place and replaced weights, a replaced or hooked module,
active capacity, routing, the MLP override, a new prompt."""

import pytest
import torch
import torch.nn.functional as F

from complexity_amd import decoder as dec
from complexity_amd.decoder import TRGQAConfig, TRGQADecoder

pytestmark = pytest.mark.gpu

CFG = TRGQAConfig(vocab_size=512, hidden_size=256, num_layers=3, num_heads=4, num_kv_heads=2, shared_width=1024,
                  num_experts=4, expert_width=32, max_position_embeddings=64)


@pytest.fixture()
def model(gpu):
    torch.manual_seed(0)
    return TRGQADecoder(CFG).to(gpu, torch.bfloat16).init_weights(3).eval()


def _steps(m, batch, n, plan, change=None):
    """n decode steps after a prompt; `change(m, s)` runs before step s."""
    g = torch.Generator().manual_seed(1)
    ids = torch.randint(0, 512, (batch, 7 + n), generator=g).to(m.norm.weight.device)
    m.prefill(ids[:, :7], max_new_tokens=n)
    out, used = [], []
    build = dec._StepPlan.build
    if not plan:
        dec._StepPlan.build = classmethod(lambda cls, *a: None)
    try:
        for s in range(n):
            if change is not None:
                change(m, s)
            out.append(m.decode_step(ids[:, 7 + s]))
            used.append(m._step_plan is not None)
    finally:
        dec._StepPlan.build = build
    return torch.stack(out), used


@pytest.mark.parametrize("batch", [1, 3, 9, 16])
def test_step_equals_blocks(model, batch):
    got, used = _steps(model, batch, 4, True)
    want, unused = _steps(model, batch, 4, False)
    assert all(used) and not any(unused)
    assert torch.equal(got, want)


def _scale_weight(m, s):
    if s in (1, 2):
        with torch.no_grad():
            m.layers[1].mlp.shared_up.weight.mul_(2.0 if s == 1 else 0.5)


def _replace_weight(m, s):
    if s == 1:
        lin = m.layers[0].self_attn.o_proj
        m.keep = lin.weight
        lin.weight = torch.nn.Parameter(lin.weight.detach() * 2)
    elif s == 2:
        m.layers[0].self_attn.o_proj.weight = m.keep


def _swap_data(m, s):
    if s == 1:
        w = m.layers[2].self_attn.q_proj.weight
        m.keep = w.data
        w.data = w.data.roll(1, 0).contiguous()
    elif s == 2:
        m.layers[2].self_attn.q_proj.weight.data = m.keep


def _capacity(m, s):
    if s in (1, 2):
        for b in m.layers:
            b.mlp.set_active_capacity(num_experts=2 if s == 1 else 4)


def _strategy(m, s):
    m.layers[1].mlp.routed_strategy = "grouped" if s == 1 else "auto"


def _override(m, s):
    m.mlp_fn = (lambda i, h, ids, block: h) if s == 1 else None


@pytest.mark.parametrize("change", [_scale_weight, _replace_weight, _swap_data, _capacity, _strategy, _override])
def test_changes_between_steps(model, change):
    got, _ = _steps(model, 2, 4, True, change)
    want, _ = _steps(model, 2, 4, False, change)
    plain, _ = _steps(model, 2, 4, True)
    assert torch.equal(got, want)
    assert torch.equal(got[0], plain[0]) and not torch.equal(got[1], plain[1])


def _reorder(m, s):
    """A beam's caches follow another sequence."""
    if s == 1:
        order = torch.tensor([1, 0], device=m.norm.weight.device)
        m.k_cache = [c.index_select(0, order) for c in m.k_cache]
        m.v_cache = [c.index_select(0, order) for c in m.v_cache]


def _eps(m, s):
    for b in m.layers:
        b.self_attn.q_norm.eps = b.self_attn.k_norm.eps = 1e-2 if s == 1 else 1e-6


def _scale(m, s):
    for b in m.layers:
        b.self_attn.scale = 0.5 if s == 1 else 0.125


@pytest.mark.parametrize("change", [_reorder, _eps, _scale])
def test_caches_and_constants_between_steps(model, change):
    got, used = _steps(model, 2, 4, True, change)
    want, _ = _steps(model, 2, 4, False, change)
    plain, _ = _steps(model, 2, 4, True)
    assert all(used) and torch.equal(got, want)
    assert torch.equal(got[0], plain[0]) and not torch.equal(got[1], plain[1])


def test_hooked_norm_is_called(model):
    seen = []
    handle = model.layers[1].input_layernorm.register_forward_hook(lambda mod, args, out: seen.append(1))
    _, used = _steps(model, 2, 2, True)
    assert len(seen) == 3 and not any(used)   # the prompt and two steps
    handle.remove()
    assert all(_steps(model, 2, 2, True)[1])


def test_k_norm_eps_of_its_own(model):
    """k is normed with k_norm's own eps: the prompt and the steps of the
    general path, whose rounding to bf16 after each operation is the bound."""
    for b in model.layers:
        b.self_attn.k_norm.eps = 0.5
    got, _ = _steps(model, 2, 3, True)
    ref = TRGQADecoder(CFG, backend="pytorch").to(got.device).eval()
    ref.load_state_dict({k: v.float() if v.is_floating_point() else v for k, v in model.state_dict().items()})
    for b in ref.layers:
        b.self_attn.k_norm.eps = 0.5
    want, _ = _steps(ref, 2, 3, True)
    assert float((got.float() - want).abs().max() / want.abs().max()) <= 2e-2


class _Wrapped(torch.nn.Module):
    """A replaced MLP half that offers what the decoder calls, and no more."""

    def __init__(self, engine):
        super().__init__()
        self.engine = [engine]

    def forward_norm_residual(self, *a):
        return self.engine[0].forward_norm_residual(*a)


def test_replaced_mlp_module(model):
    want, _ = _steps(model, 2, 3, False)
    model.layers[1].mlp = _Wrapped(model.layers[1].mlp)
    got, used = _steps(model, 2, 3, True)
    assert not any(used) and torch.equal(got, want)


def test_prompt_under_fp16_autocast(model):
    ids = torch.arange(20, device=model.norm.weight.device).view(2, 10)
    want = model.prefill(ids)
    with torch.autocast("cuda", dtype=torch.float16):
        got = model.prefill(ids)
    # fp16 projections of a bf16 residual stream: the decoder's bf16 bar
    assert float((got.float() - want.float()).abs().max() / want.float().abs().max()) <= 2e-2


def test_logits_under_vmap_and_forward_mode(model):
    h = torch.randn(3, 2, 256, generator=torch.Generator().manual_seed(0)).to(model.norm.weight.device).bfloat16()
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        want = F.linear(model.norm(h), model.embed_tokens.weight)   # the torch operations
        mapped = torch.func.vmap(model.logits)(h)
        out, tangent = torch.autograd.forward_ad.unpack_dual(model.logits(torch.autograd.forward_ad.make_dual(h, h * 0.5)))
    # bf16 outputs of one product in another order: a step (2^-8) of the largest
    assert float((mapped.float() - want.float()).abs().max() / want.float().abs().max()) <= 2.0 ** -8
    assert torch.equal(out, want) and tangent is not None and bool(tangent.float().abs().sum() > 0)
