"""Products whose contraction is split over work-groups (tv_gemm_split_fwd), and the rule that sends a prompt's products there."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF = torch.bfloat16


# rows and outputs around a tile of 256, two to five steps of 64 columns a split, shares of unequal length
@pytest.mark.parametrize("M,N,K,splits", [(1, 4, 128, 1), (255, 260, 192, 1), (256, 256, 320, 2), (257, 516, 384, 3), (300, 252, 1088, 7), (513, 1024, 4160, 13),
                                          (40, 300, 64 * 64 * 2, 64), (700, 768, 960, 1)])
@pytest.mark.parametrize("bias", [None, BF, torch.float32])
def test_against_64_bits(M, N, K, splits, bias):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + K)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    wide = r(M, K + 8).to(BF)
    x, w = wide[:, :K], (K ** -0.5 * r(N, K)).to(BF)          # rows of x at a distance of their own
    b = None if bias is None else r(N).to(bias)
    ref = x.double() @ w.double().T + (0 if b is None else b.double())
    mag = x.double().abs() @ w.double().abs().T + (0 if b is None else b.double().abs())
    for relu2 in (False, True):
        got, want = ops.split_linear(x, w, b, relu2, splits).double(), F.relu(ref) ** 2 if relu2 else ref
        sums = mag * K * 2.0 ** -24                           # fp32 sums of K products in any order
        if relu2:                                             # one rounding in front of the square, one behind it
            e = sums + 2.0 ** -8 * ref.abs()
            bound = (2 * ref.abs() + e) * e + 1.01 * 2.0 ** -8 * (ref.abs() + e) ** 2
        else:
            bound = sums + 2.0 ** -8 * (ref.abs() + sums)
        assert ((got - want).abs() <= bound).all(), (relu2, (got - want).abs().max())


def test_refused():
    from timeviper_amd import kernels as ops
    x, w = torch.zeros(300, 192, device=DEV, dtype=BF), torch.zeros(64, 192, device=DEV, dtype=BF)
    for args in ((x, w, None, False, 2), (x, w, None, False, 0), (x, w, None, False, 65), (x[:, :96].contiguous(), w[:, :96].contiguous())):
        with pytest.raises(ops.TimeViperHipError):
            ops.split_linear(*args)
    with pytest.raises(ops.TimeViperHipError):
        ops.split_linear(x, torch.zeros(66, 192, device=DEV, dtype=BF))
    with pytest.raises(ops.TimeViperHipError):
        ops.split_linear(torch.zeros(300, 196, device=DEV, dtype=BF)[:, 4:], w)


# whole tiles in front of the split ones, none and all of them; bands of fewer than four tiles of rows
@pytest.mark.parametrize("M,N,K,splits,full", [(300, 700, 320, 2, 5), (1300, 516, 384, 3, 8), (1300, 516, 384, 2, 17), (520, 300, 448, 3, 6), (520, 300, 448, 2, 1)])
def test_whole_tiles_in_front(M, N, K, splits, full):
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(M + full)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, b = r(M, K).to(BF), (K ** -0.5 * r(N, K)).to(BF), r(N)
    want, mag = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    got = ops.split_linear(x, w, b, False, splits, full).double()
    sums = mag * K * 2.0 ** -24
    assert ((got - want).abs() <= sums + 2.0 ** -8 * (want.abs() + sums)).all()
    with pytest.raises(ops.TimeViperHipError):
        ops.split_linear(x, w, b, False, splits, 1000)


# both sides of each line of the rule, and the route
@pytest.mark.parametrize("N,K,relu2,rows,plan", [
    (4480, 10240, False, 256, None), (4480, 10240, False, 257, (7, 0)), (4480, 10240, False, 1000, (3, 0)), (4480, 10240, False, 1700, (2, 0)), (4480, 10240, False, 2000, None),
    (8192, 28672, False, 600, None), (4096, 11008, False, 3900, None), (4096, 4096, False, 12000, None), (4480, 10240, False, 3000, (1, 0)), (4480, 10240, False, 6011, None),
    (4480, 10240, False, 4096, (8, 256)), (4480, 10240, False, 5600, None), (4480, 15680, False, 5000, (2, 256)), (4480, 15680, False, 5600, (1, 0)),
    (4480, 15680, False, 8192, (4, 512)), (4480, 15680, False, 10007, (1, 0)), (15680, 4480, True, 512, None), (15680, 4480, True, 1000, (1, 0)), (15680, 4480, True, 1400, (2, 256)),
    (15680, 4480, True, 2048, None), (15680, 4480, False, 1400, None), (15680, 4480, False, 1000, None), (4480, 5120, False, 512, None), (4480, 5120, False, 3000, (1, 0)),
    (5120, 4480, False, 7000, (5, 512)), (22656, 4480, False, 768, (16, 256)), (22656, 4480, False, 1400, None), (1024, 4480, False, 3000, None),
    (8192, 8192, False, 400, (4, 0)), (8192, 8192, False, 1000, None), (12288, 4096, True, 800, None), (12288, 4096, True, 1000, (1, 0)), (4480, 15680, False, 7000, None),
    (4096, 4096, False, 5000, None), (4480, 4544, False, 4096, (8, 256)), (28672, 8192, False, 600, None), (28672, 8192, False, 700, (3, 256)), (5376, 5632, False, 8835, None),
    (5248, 5632, False, 8835, (1, 0)), (21440, 11840, False, 9244, None), (7680, 8064, False, 9993, None), (9088, 12800, False, 1335, None), (9088, 12800, False, 1500, (1, 0)),
    (13312, 18432, False, 280, None), (13312, 18432, False, 500, (2, 0))])
def test_rule(N, K, relu2, rows, plan, monkeypatch):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    with torch.device("meta"):
        lin = torch.nn.Linear(K, N, bias=False, dtype=BF)
    lin = lin.to_empty(device=DEV).requires_grad_(False)
    x = torch.empty(1, rows, K, device=DEV, dtype=BF)
    assert ops.split_takes(x, lin.weight, relu2) == plan
    assert ops.split_takes(x[:, :, 1:], lin.weight[:, 1:], relu2) is None
    calls = []
    monkeypatch.setattr(ops, "split_linear", lambda x, w, b, r, *p: calls.append((r, *p)))
    if plan or ops.large_takes(x, lin.weight, relu2):
        plan = plan or ops.tail_plan(rows, N, K)              # (linear_fused: the persistent kernel, or whole tiles in front of split ones)
        with torch.no_grad():
            nano._prompt_linear(lin, x, relu2)
        nano._prompt_linear(lin, x[:, :300])                  # gradients enabled: the module
    assert calls == ([(relu2, *plan)] if plan else [])


def test_linear_fused_takes_what_it_took():
    """shared last rounds inside linear_fused: an odd number of steps stays refused, rows with strides are copied once and keep their leading shape"""
    from timeviper_amd import kernels as ops
    g = torch.Generator(device=DEV).manual_seed(1)
    w = (0.02 * torch.randn(4480, 4224, generator=g, device=DEV)).to(BF)
    x = torch.randn(2, 2048, 2 * 4224, generator=g, device=DEV).to(BF)[:, :, ::2]
    assert ops.tail_plan(4096, 4480, 4224) and ops.tail_plan(4096, 4480, 4160)
    got = ops.linear_fused(x, w)
    assert got.shape == (2, 2048, 4480) and torch.equal(got.view(4096, 4480), ops.linear_fused(x.reshape(4096, 4224), w))
    with pytest.raises(ops.TimeViperHipError):
        ops.linear_fused(x[..., :4160].contiguous(), w[:, :4160].contiguous())
