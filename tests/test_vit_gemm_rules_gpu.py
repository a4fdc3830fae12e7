"""The hand-written ViT products below a few tiles per compute unit, where the dispatch now takes the persistent kernels, against float64;
and the blocks' choice between them and the library."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


# fewer tiles than work-groups (and than XCDs), one ragged row or column of tiles, one and two rounds of either tile shape
@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (257, 264, 1152), (729, 1152, 1152), (2916, 3456, 1152), (7290, 1152, 1152), (10935, 1152, 1152),
                                   (13122, 1152, 1152), (700, 1152, 4352)])
@pytest.mark.parametrize("epilogue", ["bias", "gelu", "relu2", "accumulate"])
def test_few_tiles(M, N, K, epilogue):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, b = r(M, K).to(BF), (r(N, K) * K ** -0.5).to(BF), r(N).to(BF)
    s = x.double() @ w.double().T
    mag = x.double().abs() @ w.double().abs().T * (K * 2.0 ** -24)             # fp32 sums of K products
    if epilogue == "accumulate":
        c = r(M, N).to(BF)
        want = s + c.double()
        got = ops.linear_fused(x, w, None, epilogue=ops.GEMM_ACCUM, out=c.clone())
        bound = mag + want.abs() * 2.0 ** -8                                   # one rounding to bf16
    else:
        z = s + b.double()
        got = ops.linear_fused(x, w, b, epilogue={"bias": ops.GEMM_BIAS, "gelu": ops.GEMM_BIAS_GELU, "relu2": ops.GEMM_BIAS_RELU2}[epilogue])
        if epilogue == "gelu":                                                 # of the rounded sum (slope below 1.13), rounded again
            want, bound = F.gelu(z), 1.13 * (mag + z.abs() * 2.0 ** -8) + F.gelu(z).abs() * 2.0 ** -8 + 2.0 ** -20
        elif epilogue == "relu2":                                              # of the rounded sum, rounded again
            e = mag + z.abs() * 2.0 ** -8
            want = F.relu(z) ** 2
            bound = 2 * F.relu(z) * e + e * e + (want + e) * 2.0 ** -8
        else:
            want, bound = z, mag + z.abs() * 2.0 ** -8
    assert ((got.double() - want).abs() <= bound * 1.01 + 1e-30).all()


@pytest.mark.parametrize("frames,own", [(1, ()), (4, ("gelu",)), (10, ("qkv", "gelu", "accumulate")), (18, ("qkv", "gelu"))])
def test_blocks_choose(frames, own, monkeypatch):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.vit.siglip import Block
    torch.manual_seed(frames)
    blk = Block(1152, 16, 4304).to(DEV, BF).eval().requires_grad_(False)
    x = torch.randn(frames, 729, 1152, device=DEV).to(BF)
    names = {ops.GEMM_BIAS: "qkv", ops.GEMM_BIAS_GELU: "gelu", ops.GEMM_ACCUM: "accumulate"}
    calls, real = [], ops.linear_fused
    monkeypatch.setattr(ops, "linear_fused", lambda *a, **k: (calls.append(names[k["epilogue"]]), real(*a, **k))[1])
    with torch.no_grad():
        y, pend = blk.forward_stream(x.clone(), None)
        got = y.float() + pend
        blk.float()
        z = x.float()
        n, t, c = z.shape
        q, k, v = blk.attn.qkv(blk.norm1(z)).view(n, t, 3, 16, c // 16).permute(2, 0, 3, 1, 4)
        z = z + blk.attn.proj(((q @ k.transpose(-1, -2)) * blk.attn.scale).softmax(-1).matmul(v).transpose(1, 2).reshape(n, t, c))
        ref = z + blk.mlp.fc2(F.gelu(blk.mlp.fc1(blk.norm2(z))))
    assert sorted(set(calls)) == sorted(own)
    assert ((got - ref).norm() / ref.norm()) < 1e-2


@pytest.mark.parametrize("rows,N,K,relu2,own", [(1500, 22656, 4480, False, True), (300, 22656, 4480, False, False), (6011, 4480, 10240, False, True),
                                                (8000, 4480, 10240, False, False), (2048, 15680, 4480, True, True), (2048, 15680, 4480, False, False)])
def test_long_prompts(rows, N, K, relu2, own, monkeypatch):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    torch.manual_seed(rows)
    with torch.device("meta"):
        lin = torch.nn.Linear(K, N, bias=False, dtype=BF)
    lin = lin.to_empty(device=DEV).requires_grad_(False)
    lin.weight.normal_(0, K ** -0.5)
    x = torch.randn(1, rows, K, device=DEV).to(BF)
    calls, real = [], ops.linear_fused
    monkeypatch.setattr(ops, "linear_fused", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    with torch.no_grad():
        got = nano._prompt_linear(lin, x, relu2)
        sel = slice(rows - 300, rows)                          # (the last, ragged tile among them)
        ref = x[0, sel].double() @ lin.weight.double().T
    if relu2:
        ref = F.relu(ref) ** 2
    assert bool(calls) == own
    # 2^-8 a rounding of bf16: one, or a squared one (twice) and another; 5 % for the fp32 sums
    assert (got[0, sel].double() - ref).abs().max() <= 1.05 * (3 if relu2 else 1) * 2.0 ** -8 * ref.abs().max()


def test_weights_off_their_alignment_are_the_librarys(monkeypatch):
    """qkv, proj and fc2 weights at an address that is no multiple of 16 bytes: the block runs, and none of them on the hand-written kernels"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.vit.siglip import Block
    torch.manual_seed(0)
    blk = Block(1152, 16, 4352).to(DEV, BF).eval().requires_grad_(False)
    x = torch.randn(10, 729, 1152, device=DEV).to(BF)
    with torch.no_grad():
        want = blk.forward_stream(x.clone(), None)[0]
    for mod in (blk.attn.qkv, blk.attn.proj, blk.mlp.fc1, blk.mlp.fc2):
        w = torch.empty(mod.weight.numel() + 4, dtype=BF, device=DEV)[4:].view(mod.weight.shape)
        w.copy_(mod.weight)
        mod.weight = torch.nn.Parameter(w, requires_grad=False)
        assert w.data_ptr() % 16 == 8
    calls, real = [], ops.linear_fused
    monkeypatch.setattr(ops, "linear_fused", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    with torch.no_grad():
        got = blk.forward_stream(x.clone(), None)[0]
    assert not calls
    assert ((got.float() - want.float()).norm() / want.float().norm()) < 1e-2


# (width, tokens a frame, frames) -> the qkv projection is faster on the persistent kernel: padded widths alone, two to six rounds of tiles, ragged rows
@pytest.mark.parametrize("width,heads,tokens,frames,own", [(1152, 16, 729, 15, True), (1152, 16, 729, 33, True), (1152, 16, 729, 9, True),
                                                           (1152, 16, 729, 5, False), (1152, 16, 729, 41, False), (1152, 16, 256, 32, False),
                                                           (768, 12, 576, 16, False), (1024, 16, 261, 24, False)])
def test_qkv_rule(width, heads, tokens, frames, own):
    from timeviper_amd.model.vit.siglip import Attention
    attn = Attention(width, heads).to(DEV, BF).requires_grad_(False)
    with torch.no_grad():
        assert attn._own_qkv(torch.empty(frames, tokens, width, device=DEV, dtype=BF)) is own


@pytest.mark.parametrize("rows,n,own", [(7290, 1152, True), (34992, 1152, True), (13122, 1152, False), (10368, 768, False), (73728, 768, False)])
def test_accumulate_rule(rows, n, own):
    from timeviper_amd.model.vit.siglip import _own_accumulate
    assert _own_accumulate(rows, n) is own


def test_hook_on_fc1_of_a_short_clip(monkeypatch):
    """3 654 rows of the 1 024 wide tower: fused as it stands, called with a hook on it"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.vit.siglip import Mlp
    torch.manual_seed(0)
    mlp = Mlp(1024, 4096).to(DEV, BF).requires_grad_(False)
    x = torch.randn(14, 261, 1024, device=DEV).to(BF)
    calls, real = [], ops.linear_fused
    monkeypatch.setattr(ops, "linear_fused", lambda *a, **k: (calls.append(1), real(*a, **k))[1])
    with torch.no_grad():
        plain = mlp(x)
        assert calls == [1]
        handle = mlp.fc1.register_forward_hook(lambda m, a, y: 2 * y)
        got = mlp(x)
        handle.remove()
        want = F.linear(F.gelu(2 * F.linear(x, mlp.fc1.weight, mlp.fc1.bias)), mlp.fc2.weight, mlp.fc2.bias)
    assert calls == [1]
    rel = lambda a, b: float((a.float() - b.float()).norm() / b.float().norm())
    assert rel(got, want) < 1e-2 < rel(plain, want)


def test_qkv_switch(monkeypatch):
    """TV_VIT_OWN_QKV: 0 never, unset by the rule, 1 by the rule and from 65 536 rows on"""
    from timeviper_amd.model.vit.siglip import Attention
    attn = Attention(1152, 16).to(DEV, BF).requires_grad_(False)
    got = {}
    for switch in ("0", None, "1"):
        monkeypatch.setenv("TV_VIT_OWN_QKV", switch) if switch else monkeypatch.delenv("TV_VIT_OWN_QKV")
        with torch.no_grad():
            got[switch] = [attn._own_qkv(torch.empty(n, 729, 1152, device=DEV, dtype=BF)) for n in (2, 20, 60, 90)]
    assert got == {"0": [False] * 4, None: [False, True, False, False], "1": [False, True, False, True]}
