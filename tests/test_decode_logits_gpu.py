"""The logits of a decoded token as fp32 out of the product itself, the last norm in front of it, and the counters behind the greedy choice: the values of
the separate launches, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mk(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed + sum(shape)), device=DEV).bfloat16()


# rows of one work-group or less, a remainder of the waves, K that the matrix cores do not take (8, 4 488) or the split kernel does (8 192, 10 240)
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k,bias", [(1, 64, False), (1001, 4488, True), (9001, 4480, False), (513, 8, True), (20000, 8192, False), (7000, 10240, True)])
def test_logits(rows, n, k, bias):
    from timeviper_amd import kernels as K
    x, w, b = _mk(rows, 1, k), _mk(n, k, seed=1) * k ** -0.5, _mk(n, seed=2) if bias else None
    got = K.gemv_fused(x, w, b, out_dtype=torch.float32)
    want = K.gemv_fused(x, w, b).float()
    assert got.dtype == torch.float32 and got.shape == want.shape and torch.equal(got, want)


@pytest.mark.parametrize("n,k", [(9001, 4480), (100, 8), (4000, 8192), (513, 1032)])
@pytest.mark.parametrize("add", [True, False])
@pytest.mark.parametrize("nw", [torch.float32, torch.bfloat16])
def test_norm_in_front(n, k, add, nw):
    from timeviper_amd import kernels as K
    x, d, w, g = _mk(1, 1, k), _mk(1, 1, k, seed=3) if add else None, _mk(n, k, seed=1) * k ** -0.5, _mk(k, seed=4).to(nw)
    got = K.gemv_fused(x, w, None, K.GEMV_RMSNORM, delta=d, norm_weight=g, eps=1e-5, out_dtype=torch.float32)
    want = K.gemv_fused(x, w, None, K.GEMV_RMSNORM, delta=d, norm_weight=g, eps=1e-5).float()
    assert torch.equal(got, want)


@pytest.mark.parametrize("rows,n,k", [(2, 100, 64), (5, 9001, 4480), (17, 4099, 4480), (32, 515, 1024)])
def test_rows_rounded(rows, n, k):
    from timeviper_amd import kernels as K
    x, w, b = _mk(rows, k), _mk(n, k, seed=1) * k ** -0.5, _mk(n, seed=2)
    assert torch.equal(K.rows_linear(x, w, b, out_dtype=torch.float32, rounded=True), K.rows_linear(x, w, b).float())


@pytest.mark.parametrize("rows,n", [(1, 8192), (5, 131072), (3, 100), (2, 8195)])
@pytest.mark.parametrize("lens", [1, 64, 70])
def test_counters(rows, n, lens):
    from timeviper_amd import kernels as K
    x = torch.randn(rows, n, generator=torch.Generator(device=DEV).manual_seed(n), device=DEV)
    p, c = torch.tensor([41], device=DEV), torch.arange(lens, dtype=torch.int32, device=DEV)
    want = c + 1
    assert torch.equal(K.argmax_rows(x, (p, c)), x.argmax(-1)) and torch.equal(c, want) and p.item() == 42


def test_a_cache_that_counts_otherwise_is_asked():
    from timeviper_amd.model.llm.nano import HybridMambaAttentionDynamicCache as Cache

    class Other(Cache):
        def advance_static_device(self):
            raise AssertionError("not called here")
    pair = (torch.zeros(1, dtype=torch.int64), torch.zeros(2, dtype=torch.int32))
    for cls, want in ((Cache, pair), (Other, None)):
        c = cls.__new__(cls)
        c._static = {3: pair}
        assert c.static_counters() is want
        c._static = {3: pair, 4: pair}
        assert c.static_counters() is None


def _last_norm(llm, how):
    """what a caller may have put in the way of the norm in front of the logits; returns a list of the norm's calls that a hook saw"""
    seen, norm, head = [], llm.backbone.norm_f, llm.lm_head
    if how == "hook":
        norm.register_forward_hook(lambda *a: seen.append(1))
    elif how == "half":
        norm.weight = torch.nn.Parameter(norm.weight.detach().half(), requires_grad=False)
    elif how == "strided":
        norm.weight = torch.nn.Parameter(norm.weight.detach().repeat_interleave(2)[::2], requires_grad=False)
    elif how == "fp32":
        norm.weight = torch.nn.Parameter(norm.weight.detach().float(), requires_grad=False)
    elif how == "subclass":
        head.__class__ = type("Mine", (torch.nn.Linear,), {})
    elif how == "bias":
        head.bias = torch.nn.Parameter(torch.zeros(head.out_features, device=DEV, dtype=torch.bfloat16), requires_grad=False)
    return seen


# the norm goes with the product, or is called, with the same logits either way
@pytest.mark.parametrize("how,inside", [("plain", True), ("fp32", True), ("bias", True), ("hook", False), ("half", False), ("strided", False), ("subclass", False), ("hidden", False),
                                        ("two", False)])
def test_a_model_of_which_one_token_is_decoded(how, inside, monkeypatch):
    from timeviper_amd import kernels as K
    from timeviper_amd.model.llm.nano import HybridMambaAttentionDynamicCache, NemotronHConfig, NemotronHForCausalLM
    cfg = NemotronHConfig(vocab_size=1000, hidden_size=256, intermediate_size=512, num_hidden_layers=3, hybrid_override_pattern="M*-", num_attention_heads=4, head_dim=128,
                          num_key_value_heads=2, ssm_state_size=128, mamba_num_heads=8, mamba_n_groups=2, mamba_head_dim=80)
    torch.manual_seed(3)
    llm = NemotronHForCausalLM(cfg).to(DEV).bfloat16().eval().requires_grad_(False)
    llm.backbone.norm_f.weight.copy_(1 + 0.1 * _mk(256))
    B, ids = 2 if how == "two" else 1, torch.arange(40, device=DEV).view(1, 40)
    calls, real = [], K.gemv_fused
    monkeypatch.setattr(K, "gemv_fused", lambda *a, **k: (calls.append(k.get("norm_weight") is not None and k.get("out_dtype") is torch.float32), real(*a, **k))[1])

    def decode():
        cache = HybridMambaAttentionDynamicCache(cfg, B, dtype=torch.bfloat16, device=DEV)
        llm(input_ids=ids[:, :-1].expand(B, -1), past_key_values=cache, use_cache=True, cache_position=torch.arange(39))
        calls.clear()
        return llm(input_ids=ids[:, -1:].expand(B, -1).contiguous(), past_key_values=cache, use_cache=True, cache_position=torch.tensor([39]), output_hidden_states=how == "hidden")
    with torch.inference_mode():
        seen = _last_norm(llm, how)
        out = decode()
        assert any(calls) is inside and len(seen) == (2 if how == "hook" else 0)
        monkeypatch.setattr("timeviper_amd.model.llm.nano._norm_and_head", lambda bb, head: False)
        want = decode()
        assert not any(calls)
    if how == "hidden":
        assert out.hidden_states[-1].shape == (1, 1, 256)
    assert out.logits.dtype == torch.float32 and torch.equal(out.logits, want.logits)
