"""A decoded token of 5..32 sequences on the hybrid stack: modules with anything around them are called, operands that the hand-written
products do not take go the general way."""
import pytest
import torch

from timeviper_amd.model.llm.nano import HybridMambaAttentionDynamicCache, NemotronHConfig, NemotronHForCausalLM

pytestmark = pytest.mark.gpu
DEV = "cuda"
B = 8


def model():
    cfg = NemotronHConfig(vocab_size=256, hidden_size=256, intermediate_size=384, num_hidden_layers=3, hybrid_override_pattern="M-*",
                          num_attention_heads=4, head_dim=128, num_key_value_heads=2, ssm_state_size=16, mamba_num_heads=8,
                          mamba_n_groups=2, mamba_head_dim=16, mamba_chunk_size=16)
    torch.manual_seed(0)
    return NemotronHForCausalLM(cfg).bfloat16().to(DEV).eval()


def decode(m):
    """logits of two tokens behind a prompt, and the conv state"""
    g = torch.Generator(device=DEV).manual_seed(9)
    ids = torch.randint(0, 256, (B, 42), device=DEV, generator=g)
    with torch.no_grad():
        cache = HybridMambaAttentionDynamicCache(m.config, B, dtype=torch.bfloat16, device=DEV)
        m(input_ids=ids[:, :40], past_key_values=cache, use_cache=True, cache_position=torch.zeros(1, dtype=torch.long))
        got = [m(input_ids=ids[:, t:t + 1], past_key_values=cache, use_cache=True, cache_position=torch.full((1,), t)).logits[:, -1] for t in (40, 41)]
    return torch.stack(got), cache.conv_states[0].float()


class Doubled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


def wrap(m, where, how):
    """-> calls seen while decoding"""
    seen, parent = [], m.backbone.layers
    owner, name = {"in_proj": (parent[0].mixer, "in_proj"), "out_proj": (parent[0].mixer, "out_proj"), "up_proj": (parent[1].mixer, "up_proj"),
                   "down_proj": (parent[1].mixer, "down_proj"), "v_proj": (parent[2].mixer, "v_proj"), "o_proj": (parent[2].mixer, "o_proj"),
                   "mixer": (parent[1], "mixer"), "lm_head": (m, "lm_head")}[where]
    mod = getattr(owner, name)
    note = lambda x: seen.append(1) if x.shape[1] == 1 else None
    if how == "subclass":
        new = Doubled(mod.in_features, mod.out_features, bias=mod.bias is not None)
        new.weight, new.bias = mod.weight, mod.bias
        setattr(owner, name, new)
        new.register_forward_pre_hook(lambda _, a: note(a[0]))      # (of no effect: the type alone decides)
    elif how == "hook":
        mod.register_forward_hook(lambda _, a, y: (note(a[0]), 2 * y)[1])
    else:
        mod.register_forward_pre_hook(lambda _, a: (note(a[0]), (2 * a[0],))[1])
    return seen


@pytest.mark.parametrize("where,how", [("in_proj", "hook"), ("out_proj", "pre-hook"), ("up_proj", "subclass"), ("down_proj", "hook"), ("v_proj", "hook"),
                                       ("o_proj", "subclass"), ("mixer", "hook"), ("lm_head", "hook")])
def test_modules_are_called(where, how, monkeypatch):
    m = model()
    plain = decode(m)[0]
    seen = wrap(m, where, how)
    got, conv = decode(m)
    assert len(seen) == (3 if where == "lm_head" else 2), "each token calls the module"      # (the prompt reads its last position alone)
    monkeypatch.setenv("TV_DECODE_FUSED", "0")
    want, conv0 = decode(m)
    rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())
    assert rel(got, want) < 2e-2 and rel(conv, conv0) < 2e-2
    assert rel(plain, want) > 5e-2                                  # (what stands around the module matters)


def test_autocast_reaches_the_modules(monkeypatch):
    from timeviper_amd import kernels as K
    m = model()
    calls = []
    real = K.rows_linear
    monkeypatch.setattr(K, "rows_linear", lambda *a, **k: (calls.append(a[0].shape), real(*a, **k))[1])
    decode(m)
    assert calls
    calls.clear()
    with torch.autocast("cuda", torch.bfloat16):
        decode(m)
    assert not calls


def test_operands_the_products_do_not_take(monkeypatch):
    """A convolution kept in fp32, and weights off 16-byte alignment: the general operators, as with one sequence's worth of them"""
    m = model()
    m.backbone.layers[0].mixer.conv1d.float()
    for mod in (m.backbone.layers[0].mixer.out_proj, m.backbone.layers[1].mixer.up_proj, m.backbone.layers[2].mixer.o_proj, m.lm_head):
        w = torch.empty(mod.weight.numel() + 4, dtype=torch.bfloat16, device=DEV)[4:].view(mod.weight.shape)
        assert w.data_ptr() % 16 == 8
        w.copy_(mod.weight.detach())
        mod.weight = torch.nn.Parameter(w, requires_grad=False)
    got, conv = decode(m)
    monkeypatch.setenv("TV_DECODE_FUSED", "0")
    want, conv0 = decode(m)
    rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())
    assert rel(got, want) < 2e-2 and rel(conv, conv0) < 2e-2
