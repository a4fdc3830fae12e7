"""Products of a short prompt's rows (csrc/gemm_mid.hip) against float64, at the edges of its tiles and splits, and the layers that take them."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


# rows: edges of the 32-row tiles and of the three layouts of waves; N: below a tile, ragged, with and without a split of K;
# K: fewer stages than the rings have, odd counts of them
@pytest.mark.parametrize("M", [2, 31, 33, 64, 65, 97, 128, 129, 203, 256])
@pytest.mark.parametrize("N,K", [(4, 64), (100, 192), (1000, 1152), (4480, 4544), (8196, 320), (24580, 128)])
@pytest.mark.parametrize("relu2,bias", [(False, False), (True, True)])
def test_products(M, N, K, relu2, bias):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M * 31 + N + K)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x = r(M, K + 24).to(BF)[:, 8:8 + K]                        # a slice: rows of another stride
    w = (r(N, K + 8) * K ** -0.5).to(BF)[:, :K]
    b = r(N).to(BF) if bias else None
    got = ops.mid_linear(x, w, b, relu2).double()
    s = x.double() @ w.double().T + (0 if b is None else b.double())
    # fp32 sums of K products (relative 2^-24 each, of the sum of magnitudes), one rounding to bf16 (8 significant bits: 2^-8; squared: twice that and one more)
    acc = (x.double().abs() @ w.double().abs().T + (0 if b is None else b.double().abs())) * K * 2.0 ** -24
    e = acc * (1 + 2.0 ** -8) + s.abs() * 2.0 ** -8
    if relu2:
        want = F.relu(s) ** 2
        bound = 2 * F.relu(s) * e + e * e + (want + e) * 2.0 ** -8 + 1e-30
    else:
        want, bound = s, e + 1e-30
    assert ((got - want).abs() <= bound).all()
    assert torch.equal(got, ops.mid_linear(x, w, b, relu2).double())      # the splits add in one order


# W with and without the caches (splits of K, or the rows of W from end to end), on both sides of 64 and 128 rows, splits that start 4 KiB apart and not
@pytest.mark.parametrize("M", [64, 65, 128, 129, 256])
@pytest.mark.parametrize("N,K", [(16388, 512), (2048, 4096), (1152, 5120), (1152, 4992)])
def test_split_and_whole_rows(M, N, K):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device=DEV).to(BF), (torch.randn(N, K, generator=g, device=DEV) * K ** -0.5).to(BF)
    got, want = ops.mid_linear(x, w).double(), x.double() @ w.double().T
    # fp32 sums (relative 2^-24 a product of the sum of magnitudes), one rounding to bf16
    acc = (x.double().abs() @ w.double().abs().T) * K * 2.0 ** -24
    assert ((got - want).abs() <= acc * (1 + 2.0 ** -8) + want.abs() * 2.0 ** -8 + 1e-30).all()


# both sides of the lines between the loads of W: 96 rows, rows of W that start 16 KiB apart, 72 000 000 entries
@pytest.mark.parametrize("M", [95, 96, 203])
@pytest.mark.parametrize("N,K", [(1152, 8192), (1152, 8128), (8192, 8768), (8256, 8768)])
def test_loads_of_split_rows(M, N, K):
    """whole numbers: exact, whatever the order of the sums"""
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = (torch.randint(-3, 4, s, generator=g, device=DEV).to(BF) for s in ((M, K), (N, K)))
    assert torch.equal(ops.mid_linear(x, w), (x.double() @ w.double().T).to(BF))


@pytest.mark.parametrize("tokens", [2, 17, 48, 200, 256, 257])
def test_layers_take_them(tokens, monkeypatch):
    """The hybrid stack's projections: the short-prompt products within a rounding of torch.nn.Linear; hooks and gradients keep the module."""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    torch.manual_seed(tokens)
    # (a size that the rule takes up to 256 rows; 4 096 -> 2 048 is faster in the library from 65 on)
    lin = torch.nn.Linear(8192, 4096, bias=True, device=DEV, dtype=BF).requires_grad_(False)
    x = torch.randn(1, tokens, 8192, device=DEV, dtype=BF)
    calls = []
    for name in ("mid_linear", "rows_linear"):
        real = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, _r=real, _n=name, **k: (calls.append(_n), _r(*a, **k))[1])
    want = F.linear(x.double(), lin.weight.double(), lin.bias.double())
    for relu2 in (False, True):
        calls.clear()
        with torch.no_grad():
            got = nano._prompt_linear(lin, x, relu2)
        assert calls == (["rows_linear"] if tokens <= 32 else ["mid_linear"] if tokens <= 256 else [])
        ref = F.relu(want) ** 2 if relu2 else want
        # 2^-8 a rounding of bf16: one, or a squared one (twice) and another; 5 % for the fp32 sums
        assert (got.double() - ref).abs().max() <= 1.05 * (3 if relu2 else 1) * 2.0 ** -8 * ref.abs().max()
    calls.clear()
    nano._prompt_linear(lin, x)                                # gradients enabled
    seen = []
    handle = lin.register_forward_hook(lambda *a: seen.append(1))
    with torch.no_grad():
        nano._prompt_linear(lin, x)
    handle.remove()
    assert not calls and seen


# two and three matrices: edges of the tiles of each, with and without a split of K, rows of W of another stride
@pytest.mark.parametrize("M", [2, 33, 64, 65, 128, 129, 256])
@pytest.mark.parametrize("Ns,K", [((4096, 4), 4096), ((4000, 132, 100), 4160), ((5120, 1024, 1024), 4480), ((24580, 300, 64), 4096)])
def test_several_matrices(M, Ns, K):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + sum(Ns))
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x = r(1, M, K).to(BF)
    ws = [(r(n, K + 8) * K ** -0.5).to(BF)[:, :K] for n in Ns]
    assert ops.mid_linears_take(x, ws)
    got = ops.mid_linears(x, ws)
    for y, w in zip(got, ws):
        assert y.shape == (1, M, w.shape[0]) and y.is_contiguous()
        want = x[0].double() @ w.double().T
        # fp32 sums (relative 2^-24 a product of the sum of magnitudes), one rounding to bf16
        acc = (x[0].double().abs() @ w.double().abs().T) * K * 2.0 ** -24
        assert ((y[0].double() - want).abs() <= acc * (1 + 2.0 ** -8) + want.abs() * 2.0 ** -8 + 1e-30).all()
    assert all(torch.equal(a, b) for a, b in zip(got, ops.mid_linears(x, ws)))
    x2 = r(M, 2 * K).to(BF)[:, :K]                             # rows that are not dense: without the native host side
    assert all(torch.equal(a, b) for a, b in zip(ops.mid_linears(x2, ws), ops.mid_linears(x2.contiguous(), ws)))


@pytest.mark.parametrize("tokens", [2, 40, 256, 257])
def test_attention_takes_them(tokens, monkeypatch):
    """q, k and v of a prompt in one launch, within a rounding of the modules; hooks, biases and gradients keep the modules"""
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    cfg = nano.NemotronHConfig.nemotron_nano_9b_v2(vocab_size=256, num_hidden_layers=1, hybrid_override_pattern="*")
    torch.manual_seed(tokens)
    att = nano.NemotronHAttention(cfg, 0).to(DEV, BF).requires_grad_(False)
    x = torch.randn(1, tokens, cfg.hidden_size, device=DEV, dtype=BF)
    calls, real = [], ops.mid_linears
    monkeypatch.setattr(ops, "mid_linears", lambda *a: (calls.append(1), real(*a))[1])
    with torch.no_grad():
        got = att._qkv(x)
    assert bool(calls) == (tokens <= 256)
    for y, m in zip(got, (att.q_proj, att.k_proj, att.v_proj)):
        want = F.linear(x.double(), m.weight.double())
        assert (y.double() - want).abs().max() <= 1.05 * 2.0 ** -8 * want.abs().max()
    calls.clear()
    att._qkv(x)                                                # gradients enabled
    seen = []
    handle = att.k_proj.register_forward_hook(lambda *a: seen.append(1))
    with torch.no_grad():
        att._qkv(x)
    handle.remove()
    assert not calls and seen


@pytest.mark.parametrize("tokens,n,k,name", [(19, 15680, 4480, "rows_linear"), (20, 15680, 4480, "mid_linear"), (32, 4480, 10240, "mid_linear"), (32, 12288, 4096, "rows_linear"),
                                             (32, 4480, 5120, "rows_linear")])
def test_large_matrices_of_twenty_rows(tokens, n, k, name, monkeypatch):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    torch.manual_seed(n)
    lin = torch.nn.Linear(k, n, bias=False, device=DEV, dtype=BF).requires_grad_(False)
    x = torch.randn(1, tokens, k, device=DEV, dtype=BF)
    calls, real = [], getattr(ops, name)
    monkeypatch.setattr(ops, name, lambda *a, **kw: (calls.append(1), real(*a, **kw))[1])
    with torch.no_grad():
        got = nano._prompt_linear(lin, x)
    want = F.linear(x.double(), lin.weight.double())
    assert calls and (got.double() - want).abs().max() <= 1.05 * 2.0 ** -8 * want.abs().max()


def test_wide_outputs_rule():
    from timeviper_amd import kernels as ops
    for rows, n, want in ((79, 22656, False), (80, 22656, True), (256, 16384, True), (200, 16380, False), (257, 22656, False)):
        assert ops.mid_takes(torch.empty(1, rows, 4480, device=DEV, dtype=BF), torch.empty(n, 4480, device=DEV, dtype=BF)) is want


def test_widest_outputs_rule():
    from timeviper_amd import kernels as ops
    for rows, n, want in ((80, 32768, True), (256, 32768, True), (80, 32772, False), (256, 65536, False), (64, 65536, True)):
        assert ops.mid_takes(torch.empty(1, rows, 4480, device=DEV, dtype=BF), torch.empty(n, 4480, device=DEV, dtype=BF)) is want


@pytest.mark.parametrize("n,k,rows,mid", [(4480, 10240, 23, False), (4480, 10240, 24, True), (15680, 4480, 19, False), (15680, 4480, 20, True), (24576, 6144, 20, False), (9216, 5120, 24, True),
                                          (8192, 8192, 32, False), (8196, 8192, 32, True), (4868, 9280, 32, False), (12288, 4096, 32, False), (4480, 5120, 32, False)])
def test_rule_in_front_of_the_rows(n, k, rows, mid):
    from timeviper_amd import kernels as ops
    assert ops.mid_before_rows(torch.empty(1, rows, k, device=DEV, dtype=BF), torch.empty(n, k, device=DEV, dtype=BF)) is mid


@pytest.mark.parametrize("ns,k,rows,one", [((6144, 6144, 6144), 6144, 16, False), ((6144, 6144, 6144), 6144, 17, True), ((5120, 5120, 5120), 5120, 2, True), ((16384, 2048, 2048), 12288, 2, True)])
def test_rule_of_large_projections(ns, k, rows, one):
    from timeviper_amd import kernels as ops
    assert ops.mid_linears_take(torch.empty(1, rows, k, device=DEV, dtype=BF), [torch.empty(n, k, device=DEV, dtype=BF) for n in ns]) is one
