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


# both sides of each line of the rule, and the route
@pytest.mark.parametrize("N,K,relu2,rows,splits", [(4480, 10240, False, 256, 0), (4480, 10240, False, 257, 7), (4480, 10240, False, 1000, 3), (4480, 10240, False, 1700, 2),
                                                   (4480, 10240, False, 2000, 0), (8192, 28672, False, 600, 0), (4096, 11008, False, 3900, 0), (4096, 4096, False, 12000, 0), (4480, 10240, False, 3000, 1), (4480, 10240, False, 6011, 0), (4480, 15680, False, 5000, 2),
                                                   (4480, 15680, False, 8192, 0), (4480, 15680, False, 10007, 1), (15680, 4480, True, 512, 0), (15680, 4480, True, 1000, 1),
                                                   (15680, 4480, False, 1000, 0), (4480, 5120, False, 512, 0), (4480, 5120, False, 3000, 1), (1024, 4480, False, 3000, 0)])
def test_rule(N, K, relu2, rows, splits, monkeypatch):
    from timeviper_amd import kernels as ops
    from timeviper_amd.model.llm import nano
    with torch.device("meta"):
        lin = torch.nn.Linear(K, N, bias=False, dtype=BF)
    lin = lin.to_empty(device=DEV).requires_grad_(False)
    x = torch.empty(1, rows, K, device=DEV, dtype=BF)
    assert ops.split_takes(x, lin.weight, relu2) == splits
    assert ops.split_takes(x[:, :, 1:], lin.weight[:, 1:], relu2) == 0
    calls = []
    monkeypatch.setattr(ops, "split_linear", lambda x, w, b, r, s: calls.append((r, s)))
    monkeypatch.setattr(ops, "linear_fused", lambda *a, **k: None)
    monkeypatch.setattr(ops, "mid_linear", lambda *a, **k: None)
    if splits:
        with torch.no_grad():
            nano._prompt_linear(lin, x, relu2)
        nano._prompt_linear(lin, x[:, :300])                  # gradients enabled: the module
    assert calls == ([(relu2, splits)] if splits else [])
